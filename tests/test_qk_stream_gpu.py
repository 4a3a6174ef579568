"""nv_qkv_stream (csrc/qk_stream.hip) against float64 and against the two launches it stands for: edges of its 256 x 256 tiles, heads that
end inside one, columns behind the values, tokens without a cache row, an odd number of K blocks."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("T,K,H,G,d,dv,rot,rest", [
    (1, 128, 1, 1, 64, 16, 0, 0), (257, 192, 3, 1, 64, 64, 32, 3), (511, 320, 6, 2, 64, 48, 64, 6), (256, 256, 2, 2, 128, 128, 32, 2),
    (700, 128, 5, 5, 128, 64, 64, 5), (385, 448, 8, 4, 128, 128, 128, 16), (2049, 640, 16, 8, 128, 128, 32, 16),
    (300, 256, 4, 2, 64, 64, 0, 1), (8700, 128, 8, 8, 64, 64, 32, 8)])
def test_against_float64_and_two_launches(T, K, H, G, d, dv, rot, rest):
    from byox_vllm_amd import kernels
    torch.manual_seed(T + K + rot)
    N, scale, mscale = H * d + G * (d + dv) + rest, d ** -0.5, 1.25
    x = torch.randn(T, K + 8, device=DEV).bfloat16()[:, :K]
    w = (torch.randn(N, K, device=DEV) * K ** -0.5).bfloat16()
    positions = torch.randint(0, 5000, (T,), device=DEV)
    slots = torch.randperm(T + 9, device=DEV)[:T].int()
    slots[::7] = -1
    freq = (10000.0 ** (-torch.arange(0, rot, 2, device=DEV, dtype=torch.float32) / rot)) if rot else None
    caches = [torch.full((T + 9, G * (d + dv)), 7.0, device=DEV, dtype=torch.bfloat16) for _ in range(2)]
    args = dict(inv_freq=freq, rot_dims=rot, mscale=mscale)
    q, others = kernels.qkv_project_store(x, w, positions, scale, slots, caches[0], H, G, d, dv, **args)
    y = x.double() @ w.double().t()
    proj = kernels.linear(x, w, out_dtype=torch.float32)
    q2 = kernels.qk_rotate_store(proj, (0, H * d, (H + G) * d), positions, scale, slots, caches[1], H, G, d, dv, **args)
    # fp32 sums of K exact products, angles and their functions in fp32 (positions of 13 bits), a rotation
    tol = 4 * K * 2.0 ** -24 + (5000 * 2.0 ** -23 if rot else 0.0)

    def turned(v, heads):
        v = v.reshape(T, heads, d).clone()
        if rot:
            angle = positions.double()[:, None] * freq.double()
            co, si = (angle.cos() * mscale)[:, None], (angle.sin() * mscale)[:, None]
            a, b = v[..., :rot // 2].clone(), v[..., rot // 2:rot].clone()
            v[..., :rot // 2], v[..., rot // 2:rot] = a * co - b * si, b * co + a * si
        return v.reshape(T, -1)
    assert (q.double() - turned(y[:, :H * d], H) * scale).abs().max() < tol * 4 * scale
    assert (q - q2).abs().max() < tol * 4 * scale
    assert others.shape == (T, rest) and (rest == 0 or (others.double() - y[:, N - rest:]).abs().max() < tol * 4)
    want = torch.cat([turned(y[:, H * d:(H + G) * d], G), y[:, (H + G) * d:N - rest]], -1)
    kept = slots >= 0
    got = caches[0][slots[kept].long()].double()
    assert ((got - want[kept]).abs() <= 2.0 ** -8 * want[kept].abs() + tol * 4).all()
    untouched = torch.ones(T + 9, dtype=torch.bool, device=DEV)
    untouched[slots[kept].long()] = False
    assert (caches[0][untouched] == 7.0).all()


def test_which_calls_take_it():
    """Which calls take it; a projection with hooks is called as a module."""
    from byox_vllm_amd import kernels
    from byox_vllm_amd.layers.linear import DenseLinear
    torch.manual_seed(3)
    w = (torch.randn(2576, 512, device=DEV) * 0.05).bfloat16()      # 16 + 2 + 2 heads of 128, 16 others
    x = torch.randn(16384, 512, device=DEV).bfloat16()
    assert kernels.qkv_streams(x, w, 16, 2, 128, 128, 32, False)
    assert not kernels.qkv_streams(x[:4095], w, 16, 2, 128, 128, 32, False)          # too few rows
    assert not kernels.qkv_streams(x[:8192], w, 16, 2, 128, 128, 32, False)          # a share of 0.68
    assert not kernels.qkv_streams(x, w, 16, 2, 128, 128, 32, True)                  # pairs next to each other
    shapes = [kernels.qkv_streams(torch.empty(M, K, device=DEV, dtype=torch.bfloat16), torch.empty(2576, K, device=DEV, dtype=torch.bfloat16), 16, 2,
                                  128, 128, 32, False) for M, K in ((9500, 2048), (9500, 2176), (16384, 12288), (16384, 12416))]
    assert shapes == [True, False, True, False]      # beyond K = 2048 a share of 0.78 (9500 rows: 0.73), to 12288
    assert not kernels.qkv_streams(x, w, 32, 4, 32, 64, 32, False)                   # heads of 32
    assert not kernels.qkv_streams(x, w, 15, 2, 128, 128, 32, False)                 # heads that do not divide: refused behind it
    assert not kernels.qkv_streams(x.float(), w.float(), 16, 2, 128, 128, 32, False)
    assert not kernels.qkv_streams(x, w, 16, 2, 128, 128, 16, False)                 # halves of 8
    from byox_vllm_amd.layers.linear import called_plainly
    layer = DenseLinear(8, 8)
    assert called_plainly(layer, DenseLinear)
    layer.register_forward_hook(lambda *_: None)
    assert not called_plainly(layer, DenseLinear)


@pytest.mark.parametrize("hook", [False, True])
def test_layer_against_two_launches(hook, monkeypatch):
    """SlidingAttention.forward over prompt pieces of five requests, its second run's cache: the projection with rotation and store in one pass,
    and the two launches behind a product that a hook sees."""
    from byox_vllm_amd import kernels
    from byox_vllm_amd.layers.sliding_attention import SlidingAttention
    from byox_vllm_amd.utils.context import reset_context, set_context
    torch.manual_seed(11)
    width, H, G, d, page = 512, 16, 2, 128, 16
    past, new = [0, 5, 64, 0, 300], [9000, 6000, 1, 1300, 83]
    default = torch.get_default_dtype()
    torch.set_default_dtype(torch.bfloat16)
    try:
        with torch.device(DEV):
            layer = SlidingAttention(width, H, G, d, d, d ** -0.5, 256, 4, rot_dims=32)
    finally:
        torch.set_default_dtype(default)
    for p in layer.parameters():
        p.data.normal_(0.0, p.size(1) ** -0.5)
    pages = [-(-(a + b) // page) for a, b in zip(past, new)]
    order = torch.randperm(sum(pages)).tolist()
    tables = [[order.pop() for _ in range(n)] for n in pages]
    where = [(i, a + j) for i, (a, b) in enumerate(zip(past, new)) for j in range(b)]
    ints = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    slots = ints([tables[i][t // page] * page + t % page for i, t in where])
    positions = torch.tensor([t for _, t in where], device=DEV)
    step = dict(cu_seqlens_q=ints([sum(new[:i]) for i in range(6)]), max_seqlen_q=max(new), slot_mapping=slots, past_lens=ints(past),
                block_tables=ints([t + [0] * (max(pages) - len(t)) for t in tables]), seq_of_token=ints([i for i, _ in where]))
    h = torch.randn(sum(new), width, device=DEV).bfloat16()
    start = torch.randn(sum(pages) * page, G * 2 * d, device=DEV).bfloat16()
    for _ in range(2):
        layer.runs[layer.add_run()].block_size = page
    calls, seen = [], []
    one_pass, says = kernels.qkv_project_store, kernels.qkv_streams
    monkeypatch.setattr(kernels, "qkv_project_store", lambda *a, **k: calls.append(1) or one_pass(*a, **k))
    if hook:
        layer.inp.register_forward_hook(lambda *_: seen.append(1))

    def forward():
        for own in layer.runs:
            own.cache = start.clone()
        set_context(True, **step)
        y = layer(h, positions, run=1)
        reset_context()
        assert torch.equal(layer.runs[0].cache, start)
        return y, layer.runs[1].cache
    got, cache = forward()
    assert len(calls) == (0 if hook else 1) and len(seen) == (1 if hook else 0)
    monkeypatch.setattr(kernels, "qkv_streams", lambda *_: False)
    want, cache2 = forward()
    assert len(calls) == (0 if hook else 1) and says(h, layer.inp.weight, H, G, d, d, 32, False)
    rest = torch.ones(start.size(0), dtype=torch.bool, device=DEV)
    rest[slots.long()] = False
    assert torch.equal(cache[rest], start[rest])
    # the product behind a module is on the same tiles here (kernels.linear_streams), so the sums are the same
    assert torch.equal(got, want) and torch.equal(cache, cache2)
