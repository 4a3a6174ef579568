"""Latent attention of single tokens (csrc/latent_token.h) against float64: row widths of one to seventeen 64-byte units, one to
twenty heads, contexts around the 32 keys of a tile and the keys of a whole round of wavefronts, windows, pages of a power of
two and not, alone and shared by several workgroups."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def i32(v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


@pytest.mark.parametrize("window", [0, 33, 512])
@pytest.mark.parametrize("H,R,r,block", [(16, 512, 32, 256), (4, 128, 32, 48), (8, 256, 32, 64), (20, 384, 32, 16), (1, 16, 16, 80),
                                         (16, 96, 64, 256)])
@pytest.mark.parametrize("shared", [True, False])
def test_against_float64(H, R, r, block, window, shared):
    from byox_vllm_amd import kernels
    torch.manual_seed(H + R + window)
    contexts = [1, 31, 32, 33, 127, 129, 700, 2049] + ([] if shared else [40] * 600)
    pages = [-(-n // block) for n in contexts]
    order, tables = torch.randperm(sum(pages) + 1).tolist(), []
    for n in pages:
        tables.append([order.pop() for _ in range(n)])
    cache = torch.randn((sum(pages) + 1) * block, R + r).to(torch.bfloat16)
    B, scale = len(contexts), 0.7 * (R + r) ** -0.5
    q = torch.randn(B, H, R + r)
    cols = max(pages)
    got = kernels.latent_attn(q.view(B, -1).to(DEV), cache.to(DEV), i32([t + [0] * (cols - len(t)) for t in tables]),
                              i32(list(range(B + 1))), i32([n - 1 for n in contexts]), i32(list(range(B))), H, R, r, block, window,
                              scale, max_q=1).double().cpu().view(B, H, R)
    for b, n in enumerate(contexts[:12]):
        rows = torch.cat([cache[p * block:(p + 1) * block] for p in tables[b]])[max(0, n - window) if window else 0:n].double()
        w = torch.softmax(q[b].double() @ rows.t() * scale, -1)
        want = w @ rows[:, :R]
        # queries and probabilities carry 16 bits of mantissa; the result is rounded to 8
        bound = 2.0 ** -8 * want.abs() + 2.0 ** -13 * (w @ rows[:, :R].abs()) + 1e-6
        assert ((got[b] - want).abs() <= bound).all(), (n, float(((got[b] - want).abs() - bound).max()))
