"""The copies of the expanded latent form (csrc/latent_attn.hip): whole rows of keys and values and whole rotated query rows, with
heads that split into 16-byte pieces and that do not."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,dim,rot,vdim,rank", [(16, 96, 32, 128, 512), (3, 8, 8, 16, 24), (2, 12, 4, 20, 36), (3, 7, 2, 5, 9), (2, 8, 0, 8, 8)])
def test_expand(dtype, H, dim, rot, vdim, rank):
    from byox_vllm_amd._C import check, dtype_code, lib, ptr, stream
    rows = 37
    kv, c = torch.randn(rows, H * (dim + vdim), device=DEV).to(dtype), torch.randn(rows, rank + rot, device=DEV).to(dtype)
    out = torch.empty(rows, H * (dim + rot + vdim), device=DEV, dtype=dtype)
    check(lib().nv_latent_expand(ptr(kv), ptr(c), ptr(out), rows, H, dim, rot, vdim, rank, dtype_code(dtype, allow_f32=True),
                                 stream()), "nv_latent_expand")
    k = torch.cat([kv[:, :H * dim].view(rows, H, dim), c[:, None, rank:].expand(rows, H, rot)], -1).reshape(rows, -1)
    assert torch.equal(out, torch.cat([k, kv[:, H * dim:]], -1))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("H,dim,rot,rot_dims", [(16, 96, 32, 32), (3, 8, 8, 6), (2, 7, 2, 2), (1, 20, 600, 600)])
def test_query_rows(dtype, interleaved, H, dim, rot, rot_dims):
    from byox_vllm_amd import kernels
    T, scale, mag = 11, 0.3, 1.25
    q = torch.randn(T, H * (dim + rot), device=DEV).to(dtype)
    pos = torch.randint(0, 5000, (T,), device=DEV)
    freq = (10000.0 ** (-torch.arange(rot_dims // 2, device=DEV) / max(1, rot_dims // 2))).float()
    got = kernels.latent_q_rows(q, pos, freq, mag, H, dim, rot, rot_dims, scale, interleaved).view(T, H, dim + rot).double()
    want = q.double().view(T, H, dim + rot).clone()
    a = (pos.float()[:, None] * freq).double()[:, None]          # the angle is rounded to fp32
    x = want[..., dim:dim + rot_dims].clone()
    u, v = (x[..., 0::2], x[..., 1::2]) if interleaved else x.chunk(2, -1)
    y, z = u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin()
    want[..., dim:dim + rot_dims] = mag * (torch.stack([y, z], -1).flatten(-2) if interleaved else torch.cat([y, z], -1))
    assert ((got - want * scale).abs() <= 8 * 2.0 ** -24 * (want * scale).abs().max()).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rank,rot,q_rank", [(512, 32, 1024), (24, 8, 36), (9, 2, 7), (4100, 4, 4096), (8, 0, 4104), (512, 30, 1022)])
def test_norms_of_both_latents(dtype, rank, rot, q_rank):
    """The latent's norm and store with the query latent's norm beside it, in fours and one by one; an unkept token."""
    from byox_vllm_amd import kernels
    torch.manual_seed(rank)
    T, eps = 9, 1e-5
    dn = torch.randn(T, q_rank + rank + rot + 5, device=DEV)
    w, qw = (torch.rand(rank, device=DEV) + 0.5).to(dtype), (torch.rand(q_rank, device=DEV) + 0.5).to(dtype)
    slots = torch.randperm(16, device=DEV)[:T].int()
    slots[4] = -1
    cache = torch.zeros(16, rank + rot, dtype=dtype, device=DEV)
    pos = torch.zeros(T, dtype=torch.int64, device=DEV)
    freq = torch.ones(max(1, rot // 2), device=DEV)
    kv, q = dn[:, q_rank:q_rank + rank + rot], dn[:, :q_rank]
    got = kernels.latent_kv_store(kv, w, pos, freq, 1.0, slots, cache, rank, rot, rot, eps, q=q, q_norm_w=qw)

    def rms(x, f):
        x = x.double()
        return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * f.double()
    # the sum of squares in fp32 in any order, then the reciprocal root, two products and the storage type's rounding
    tol = (rank + q_rank) ** 0.5 * 2.0 ** -24 + (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -21)
    keep = slots >= 0
    rows = cache[slots[keep].long()].double()
    for a, b in ((got.double(), rms(q, qw)), (rows[:, :rank], rms(kv[keep][:, :rank], w))):
        assert ((a - b).abs() <= tol * b.abs()).all()
    assert torch.equal(rows[:, rank:], kv[keep][:, rank:].to(dtype).double())          # position 0: nothing turns
    empty = torch.ones(16, dtype=torch.bool, device=DEV)
    empty[slots[keep].long()] = False
    assert not cache[empty].any()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rank,rot", [(512, 32), (508, 4), (514, 2), (4096, 8), (4100, 4), (9, 2)])
def test_the_latent_alone(dtype, rank, rot):
    """Without a query latent: in fours from 512 numbers on, else one by one; the same cache as beside one."""
    from byox_vllm_amd import kernels
    torch.manual_seed(rank)
    T, eps = 9, 1e-5
    kv, q = torch.randn(T, rank + rot, device=DEV), torch.randn(T, 64, device=DEV)
    w, qw = (torch.rand(rank, device=DEV) + 0.5).to(dtype), torch.ones(64, device=DEV).to(dtype)
    slots, pos = torch.randperm(16, device=DEV)[:T].int(), torch.zeros(T, dtype=torch.int64, device=DEV)
    slots[4] = -1
    freq = torch.ones(max(1, rot // 2), device=DEV)
    alone, beside = (torch.zeros(16, rank + rot, dtype=dtype, device=DEV) for _ in range(2))
    assert kernels.latent_kv_store(kv, w, pos, freq, 1.0, slots, alone, rank, rot, rot, eps) is None
    kernels.latent_kv_store(kv, w, pos, freq, 1.0, slots, beside, rank, rot, rot, eps, q=q, q_norm_w=qw)
    # the same sum of squares in another order, then the reciprocal root and the storage type's rounding
    tol = rank ** 0.5 * 2.0 ** -24 + (2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -21)
    assert ((alone.double() - beside.double()).abs() <= tol * beside.double().abs()).all()
    assert (alone.abs().sum(-1) > 0).sum() == T - 1
