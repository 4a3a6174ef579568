"""Query rows and norms of latent attention (csrc/latent_attn.hip) against float64.  Whole query rows: one, two and four tokens to a workgroup, last
workgroups with fewer, rows shorter and longer than a workgroup's lanes, rotations that end inside the rotated part."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


# the line between the two forms: 1024 tokens below 32 rotated numbers, 4096 without one
@pytest.mark.parametrize("T", [1, 5, 1024, 1025, 2048, 2049, 2051, 4096, 4097])
@pytest.mark.parametrize("H,d,r,rot", [(1, 4, 8, 8), (3, 32, 16, 8), (4, 96, 32, 32), (5, 96, 32, 32), (9, 100, 28, 24), (2, 64, 0, 0)])
@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("dtype,out_dtype", [(torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32), (torch.float32, torch.float32)])
def test_rows(T, H, d, r, rot, interleaved, dtype, out_dtype):
    from byox_vllm_amd import kernels
    torch.manual_seed(T + H)
    q, positions = torch.randn(T, H * (d + r)).to(dtype), torch.randint(0, 100, (T,))
    freq = 10000.0 ** (-torch.arange(0, max(rot, 2), 2).float() / max(rot, 2))
    want = q.double().view(T, H, d + r).clone()
    if rot:
        part, half = want[..., d:d + rot].clone(), rot // 2
        angle = (positions.float()[:, None] * freq).double()[:, None]      # the product is the kernel's, in fp32
        a, b = (part[..., 0::2], part[..., 1::2]) if interleaved else (part[..., :half], part[..., half:])
        x, y = (a * angle.cos() - b * angle.sin()) * 1.25, (b * angle.cos() + a * angle.sin()) * 1.25
        want[..., d:d + rot] = torch.stack([x, y], -1).flatten(-2) if interleaved else torch.cat([x, y], -1)
    want = (want * 0.125).view(T, -1)
    got = kernels.latent_q_rows(q.to(DEV), positions.to(DEV), freq.to(DEV), 1.25, H, d, r, rot, 0.125, interleaved, out_dtype)
    assert got.dtype == out_dtype
    # cosines within 2 units of 2^-24, two products and their sum of numbers below 6; then one rounding of the result
    assert ((got.double().cpu() - want).abs() <= 2.0 ** -20 + (2.0 ** -8 * want.abs() if out_dtype == torch.bfloat16 else 0.0)).all()


@pytest.mark.parametrize("T", [1, 3, 9])
@pytest.mark.parametrize("q_rank,rank,r", [(4, 8, 8), (256, 260, 16), (260, 256, 0), (1024, 1020, 64), (1028, 512, 32), (768, 1028, 32)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_both_norms(T, q_rank, rank, r, dtype):
    """A wavefront to a row, and (more than 1024 numbers) a workgroup to a row; one token has no place in the cache."""
    from byox_vllm_amd import kernels
    torch.manual_seed(T + rank)
    x = torch.randn(T, q_rank + rank + r + 4) * 2.0
    qw, w, positions = torch.randn(q_rank).to(dtype), torch.randn(rank).to(dtype), torch.randint(0, 100, (T,))
    freq = 10000.0 ** (-torch.arange(0, max(r, 2), 2).float() / max(r, 2))
    slots = [T + 1 - i for i in range(T)]
    slots[T // 2] = -1
    cache = torch.full((T + 2, rank + r), 7.0, dtype=dtype, device=DEV)
    d = x.to(DEV)
    got = kernels.latent_kv_store(d[:, q_rank:q_rank + rank + r], w.to(DEV), positions.to(DEV), freq.to(DEV), 1.0,
                                  torch.tensor(slots, dtype=torch.int32, device=DEV), cache, rank, r, r, 1e-5, False, q=d[:, :q_rank],
                                  q_norm_w=qw.to(DEV))
    def norm(v, f):
        return v * torch.rsqrt(v.pow(2).mean(-1, keepdim=True) + 1e-5) * f.double()
    a, b = x[:, q_rank + rank:q_rank + rank + r].double().chunk(2, -1)
    angle = (positions.float()[:, None] * freq[:r // 2]).double()
    turned = torch.cat([a * angle.cos() - b * angle.sin(), b * angle.cos() + a * angle.sin()], -1)
    want = torch.full((T + 2, rank + r), 7.0, dtype=torch.float64)
    rows = torch.cat([norm(x[:, q_rank:q_rank + rank].double(), w), turned], -1)
    for i, s in enumerate(slots):
        if s >= 0:
            want[s] = rows[i]
    for have, should in ((got, norm(x[:, :q_rank].double(), qw)), (cache, want)):
        # a sum of squares of 1028 numbers (its error halved by the root), root, quotient and two products; then one rounding
        bound = (1028 / 64 + 8) * 2.0 ** -24 * should.abs() + 2.0 ** -20 + (2.0 ** -8 * should.abs() if dtype == torch.bfloat16 else 0.0)
        assert ((have.double().cpu() - should).abs() <= bound).all()


@pytest.mark.parametrize("rank", [512, 516, 768, 1020, 1024])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_norms_add_their_squares_in_one_order(rank, dtype):
    """A row's norm is the same number whether a wavefront takes it (beside the query's) or a workgroup (alone): to the last bit."""
    from byox_vllm_amd import kernels
    torch.manual_seed(rank)
    T, r = 301, 32
    x, w = (torch.randn(T, rank + r) * 2.0).to(DEV), torch.randn(rank).to(dtype).to(DEV)
    rest = (torch.arange(T).to(DEV), torch.rand(r // 2).to(DEV), 1.0, torch.arange(T, dtype=torch.int32).to(DEV))
    alone, beside = (torch.empty(T, rank + r, dtype=dtype, device=DEV) for _ in range(2))
    kernels.latent_kv_store(x, w, *rest, alone, rank, r, r, 1e-5)
    got = kernels.latent_kv_store(x, w, *rest, beside, rank, r, r, 1e-5, q=x[:, :rank], q_norm_w=w)
    assert torch.equal(beside, alone) and torch.equal(got, alone[:, :rank])


@pytest.mark.parametrize("B", [1, 2, 64, 65, 66, 131])
@pytest.mark.parametrize("width,dtype", [(24, torch.bfloat16), (544, torch.bfloat16), (20, torch.bfloat16), (12, torch.float32), (7, torch.float32)])
def test_rows_gathered_from_pages(B, width, dtype):
    """Requests found 64 starts at a time, some without tokens; rows in pieces of 16 bytes and in single numbers."""
    from byox_vllm_amd._C import check, dtype_code, lib, ptr, stream
    torch.manual_seed(B + width)
    block = 16
    past, new = torch.randint(0, 40, (B,)).tolist(), torch.randint(0, 30, (B,)).tolist()
    past[0], new[0] = 3, 2
    if B > 1:
        past[1] = new[1] = 0
    pages = [-(-(a + b) // block) for a, b in zip(past, new)]
    order = torch.randperm(sum(pages)).tolist()
    tables, cu_k, cu_q = torch.zeros(B, max(pages), dtype=torch.int32), [0], [0]
    cache = torch.randn(sum(pages) * block, width).to(dtype)
    want = torch.zeros(sum(pages) * block, width, dtype=dtype)
    for b in range(B):
        for i in range(pages[b]):
            tables[b, i] = p = order.pop()
            filled = min(block, past[b] + new[b] - i * block)
            want[cu_k[b] + i * block:cu_k[b] + i * block + filled] = cache[p * block:p * block + filled]
        cu_k.append(cu_k[-1] + pages[b] * block)
        cu_q.append(cu_q[-1] + new[b])
    out = torch.full_like(want, 9.0).to(DEV)
    args = [t.to(DEV) for t in (cache, tables, *(torch.tensor(v, dtype=torch.int32) for v in (cu_k, cu_q, past)))]
    check(lib().nv_latent_gather(ptr(args[0]), ptr(args[1]), tables.size(1), *map(ptr, args[2:]), B, block, width, ptr(out), cu_k[-1],
                                 dtype_code(dtype, allow_f32=True), stream()), "nv_latent_gather")
    assert torch.equal(out.cpu(), want)
