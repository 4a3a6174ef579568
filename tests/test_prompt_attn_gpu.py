"""Prompt attention over paged rows (csrc/prompt_attn.h) against float64: heads of 64 and 128, one to five query heads per key
head, portions that end inside tiles and continue from cached tokens, pages of a power of two and not, windows, kept first
keys, chunks, sinks, gates, values that are the keys; and the rotating page store in its four-numbers-per-access form."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
CASES = [  # window, keep, chunk, sink, gate ("", "head", "number"), values are keys
    (0, 0, 0, False, "", False), (70, 0, 0, False, "head", False), (33, 5, 0, True, "head", False),
    (0, 0, 64, False, "number", False), (0, 0, 0, True, "number", True), (200, 300, 0, False, "", False)]


def i32(v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


@pytest.mark.parametrize("options", CASES)
@pytest.mark.parametrize("D,R,G,block", [(128, 2, 2, 64), (64, 1, 3, 48), (128, 4, 1, 16), (64, 3, 2, 256), (128, 5, 1, 80)])
def test_against_float64(D, R, G, block, options):
    from byox_vllm_amd import kernels
    window, keep, chunk, with_sink, gate_form, same = options
    torch.manual_seed(D + R + G + window)
    new, past = [1, 63, 64, 65, 150, 2], [100, 0, 7, 64, 33, 0]
    H, width = R * G, G * D if same else 2 * G * D
    pages = [-(-(a + b) // block) for a, b in zip(new, past)]
    order, tables = torch.randperm(sum(pages) + 2).tolist(), []
    for n in pages:
        tables.append([order.pop() for _ in range(n)])
    cache = torch.randn((sum(pages) + 2) * block, width).to(torch.bfloat16)
    cu = [0]
    for n in new:
        cu.append(cu[-1] + n)
    T = cu[-1]
    q = torch.randn(T, H * D) * D ** -0.5 * 2.0
    sink = torch.randn(H).to(torch.bfloat16) if with_sink else None
    gate = torch.randn(T, H if gate_form == "head" else H * D) if gate_form else None
    want = torch.zeros(T, H, D, dtype=torch.float64)
    for b, t in enumerate(tables):
        n = past[b] + new[b]
        rows = torch.cat([cache[p * block:(p + 1) * block] for p in t])[:n].double()
        k = rows[:, :G * D].view(n, G, D)
        v = k if same else rows[:, G * D:].view(n, G, D)
        i, j = torch.arange(past[b], n)[:, None], torch.arange(n)[None]
        seen = j <= i
        if window:
            seen &= (i - j < window) | (j < keep)
        if chunk:
            seen &= i // chunk == j // chunk
        for h in range(H):
            s = q[cu[b]:cu[b + 1]].to(torch.bfloat16).double().view(-1, H, D)[:, h] @ k[:, h // R].t()
            s = s.masked_fill(~seen, float("-inf"))
            top = s.amax(-1, keepdim=True)
            e = torch.exp(s - top)
            below = e.sum(-1, keepdim=True) + (torch.exp(sink[h].double() - top) if with_sink else 0.0)
            want[cu[b]:cu[b + 1], h] = e / below @ v[:, h // R]
    if gate_form:
        want = want * torch.sigmoid(gate.double()).view(T, H, -1)
    out = torch.zeros(T, H * D + 8, dtype=torch.bfloat16, device=DEV)
    cols = max(pages)
    kernels.paged_softmax_attn(q.to(DEV), cache.to(DEV), i32([t + [0] * (cols - len(t)) for t in tables]), i32(cu), i32(past),
                               i32([b for b, n in enumerate(new) for _ in range(n)]), max(new), H, G, D, D, block, out,
                               window=window, keep_first=keep, chunk=chunk, sink=None if sink is None else sink.to(DEV),
                               gate=None if gate is None else gate.to(DEV), gate_per_head=gate_form == "head",
                               values_are_keys=same)
    got = out[:, :H * D].double().cpu().view(T, H, D)
    # probabilities rounded to 8 bits of mantissa (their sum is not), values exact, one rounding of the result: a row's error
    # is at most 2^-9 of sum p |v| <= max |v| twice over, here three units of the result's scale at most
    assert torch.isfinite(got).all()
    off = (got - want).abs().amax(-1)
    bound = 2.0 ** -8 * want.abs().amax(-1) + 2.0 ** -9 * 4.0
    assert (off <= bound).all(), float((off - bound).max())
    assert (got - want).norm() <= 2.0 ** -8 * want.norm()
    assert not out[:, H * D:].any()


@pytest.mark.parametrize("window,keep", [(0, 0), (50, 4)])
@pytest.mark.parametrize("D,R,G", [(128, 1, 2), (64, 2, 2), (64, 3, 1), (128, 8, 1)])
def test_steps_of_single_tokens_and_pieces(D, R, G, window, keep):
    """Decoding requests beside prompt pieces, more requests than a wavefront has lanes, one of them without tokens, pieces at
    the edges of a tile of 128 / R tokens: against float64, and the entry that is not told how many requests there are."""
    from byox_vllm_amd import kernels
    from byox_vllm_amd._C import check, dtype_code, lib, ptr, stream
    torch.manual_seed(D + R)
    TQ, H, block = 128 // R, R * G, 32
    new = [1] * 70 + [0, TQ, TQ + 1, 1, TQ - 1, 2 * TQ, 3]
    past = [(37 * i) % 90 for i in range(70)] + [5, 0, 64, 200, 7, 31, 0]
    pages = [-(-(a + b) // block) for a, b in zip(new, past)]
    order, tables = torch.randperm(sum(pages)).tolist(), []
    for n in pages:
        tables.append([order.pop() for _ in range(n)])
    cache = torch.randn(sum(pages) * block, 2 * G * D).to(torch.bfloat16)
    cu = [0]
    for n in new:
        cu.append(cu[-1] + n)
    T = cu[-1]
    q = torch.randn(T, H * D) * D ** -0.5 * 2.0
    want = torch.zeros(T, H, D, dtype=torch.float64)
    for b, t in enumerate(tables):
        n = past[b] + new[b]
        rows = torch.cat([cache[p * block:(p + 1) * block] for p in t])[:n].double()
        i, j = torch.arange(past[b], n)[:, None], torch.arange(n)[None]
        seen = (j <= i) & ((i - j < window) | (j < keep)) if window else j <= i
        for h in range(H):
            g = h // R
            s = q[cu[b]:cu[b + 1]].to(torch.bfloat16).double().view(-1, H, D)[:, h] @ rows[:, g * D:(g + 1) * D].t()
            want[cu[b]:cu[b + 1], h] = torch.softmax(s.masked_fill(~seen, float("-inf")), -1) @ rows[:, (G + g) * D:(G + g + 1) * D]
    q, cache, tables, ints = q.to(DEV), cache.to(DEV), i32([t + [0] * (max(pages) - len(t)) for t in tables]), (
        i32(cu), i32(past), i32([b for b, n in enumerate(new) for _ in range(n)]))
    out = torch.full((T, H * D), float("nan"), dtype=torch.bfloat16, device=DEV)
    kernels.paged_softmax_attn(q, cache, tables, *ints, max(new), H, G, D, D, block, out, window=window, keep_first=keep)
    untold = torch.full_like(out, float("nan"))
    check(lib().nv_paged_softmax_attn(ptr(q), ptr(cache), ptr(tables), tables.size(1), *map(ptr, ints), ptr(untold), H * D, T, max(new),
                                      H, G, D, D, block, window, 0, keep, 0.0, 1.0, 0, 0, ptr(None), ptr(None), 0, 0, ptr(None), 0,
                                      dtype_code(out.dtype), stream()), "nv_paged_softmax_attn")
    for got in (out, untold):
        got = got.double().cpu().view(T, H, D)
        assert torch.isfinite(got).all()
        # as above: probabilities rounded to 8 bits of mantissa, one rounding of the result
        assert ((got - want).abs().amax(-1) <= 2.0 ** -8 * want.abs().amax(-1) + 2.0 ** -9 * 4.0).all()
        assert (got - want).norm() <= 2.0 ** -8 * want.norm()


@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("options", CASES)
@pytest.mark.parametrize("D,R,G", [(128, 2, 2), (64, 3, 1)])
def test_a_value_that_is_not_finite_stays_out_of_rows_that_do_not_see_it(D, R, G, options, bad):
    """One number of one token's value row is an infinity or a NaN: tokens ahead of it, and those it is out of the window or the
    chunk of, keep their rows; the others have one number per head that is not finite."""
    from byox_vllm_amd import kernels
    window, keep, chunk, with_sink, gate_form, same = options
    torch.manual_seed(D + R)
    block, H, past, new = 48, R * G, [70, 0], [180, 40]
    pages = [-(-(a + b) // block) for a, b in zip(new, past)]
    order, tables = torch.randperm(sum(pages)).tolist(), []
    for n in pages:
        tables.append([order.pop() for _ in range(n)])
    cache = torch.randn(sum(pages) * block, G * D if same else 2 * G * D).to(torch.bfloat16)
    T, cols = sum(new), max(pages)
    q = torch.randn(T, H * D, device=DEV) * D ** -0.5 * 2.0
    sink = torch.randn(H, device=DEV).to(torch.bfloat16) if with_sink else None
    gate = torch.randn(T, H if gate_form == "head" else H * D, device=DEV) if gate_form else None
    ints = (i32([t + [0] * (cols - len(t)) for t in tables]), i32([0, new[0], T]), i32(past), i32([0] * new[0] + [1] * new[1]))

    def rows(c):
        out = torch.zeros(T, H * D, dtype=torch.bfloat16, device=DEV)
        kernels.paged_softmax_attn(q, c.to(DEV), *ints, max(new), H, G, D, D, block, out, window=window, keep_first=keep, chunk=chunk,
                                   sink=sink, gate=gate, gate_per_head=gate_form == "head", values_are_keys=same)
        return out.double().cpu().view(T, H, D)
    want = rows(cache)
    for at in (0, 69, 70, 133, 200, 249):               # position in the first request
        spoilt = cache.clone()
        spoilt[tables[0][at // block] * block + at % block, (0 if same else G * D) + 5] = bad       # head 0's sixth number
        got = rows(spoilt)
        i = torch.arange(past[0], past[0] + new[0])
        sees = i >= at
        if window:
            sees &= (i - at < window) | (at < keep)
        if chunk:
            sees &= i // chunk == at // chunk
        sees = torch.cat([sees, torch.zeros(new[1], dtype=torch.bool)])
        # probabilities of rows formed again are summed in another order; one rounding of the result
        near = (got - want).abs() <= 2.0 ** -7 * want.abs() + 2.0 ** -9
        assert near[~sees].all(), at
        assert near[:, R:].all(), at
        assert not torch.isfinite(got[sees][:, :R, 5]).any(), at
        if not same:                                    # (a key that is not finite spoils the row's scores)
            others = [n for n in range(D) if n != 5]
            assert near[sees][:, :R][..., others].all(), at


@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("dim,vdim,rot", [(64, 64, 32), (128, 64, 128), (20, 12, 8), (24, 24, 12), (16, 8, 0)])
def test_rotating_store(dim, vdim, rot, interleaved):
    from byox_vllm_amd import kernels
    torch.manual_seed(dim + rot)
    T, H, G = 37, 4, 2
    cols = (H + G) * dim + G * vdim
    proj = torch.randn(T, cols + 4)
    positions = torch.randint(0, 3000, (T,))
    freq = (1.0 / 10000.0 ** (torch.arange(0, max(rot, 2), 2).float() / max(rot, 2)))[:rot // 2]
    cache = torch.zeros(T + 3, G * (dim + vdim), device=DEV)
    slots = torch.randperm(T + 3)[:T].to(torch.int32)
    q = kernels.qk_rotate_store(proj.to(DEV), (0, H * dim, (H + G) * dim), positions.to(DEV), 0.3, slots.to(DEV), cache, H, G, dim,
                                vdim, inv_freq=freq.to(DEV) if rot else None, rot_dims=rot, interleaved=interleaved)

    def turn(x):          # [T, heads, dim]
        x, angle = x.double().clone(), (positions.float()[:, None] * freq[None]).double()[:, None]     # angles are fp32 products
        a, b = (slice(0, rot, 2), slice(1, rot, 2)) if interleaved else (slice(0, rot // 2), slice(rot // 2, rot))
        u, v = x[..., a].clone(), x[..., b].clone()
        x[..., a], x[..., b] = u * angle.cos() - v * angle.sin(), v * angle.cos() + u * angle.sin()
        return x
    heads = turn(proj[:, :(H + G) * dim].view(T, H + G, dim)) if rot else proj[:, :(H + G) * dim].double().view(T, H + G, dim)
    assert torch.allclose(q.double().cpu().view(T, H, dim), heads[:, :H] * 0.3, rtol=1e-6, atol=1e-6)
    rows = cache.double().cpu()[slots.long()]
    assert torch.allclose(rows[:, :G * dim].view(T, G, dim), heads[:, H:], rtol=1e-6, atol=2e-6)
    assert torch.equal(rows[:, G * dim:], proj[:, (H + G) * dim:cols].double())
