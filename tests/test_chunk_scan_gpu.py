"""Prompts through the sixteen-token chunks of csrc/chunk_scan.h: against float64 recurrences written out here and against the
token-by-token walk of the same library, at the edges of chunks, of the 64 tokens whose gates are read at once, and of the
key and value sizes the kernel serves; decays from none to one that leaves nothing after a token."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
LENS = [1, 15, 16, 17, 31, 64, 65, 130]
# fp32 products and sums of up to 128 terms in other orders than the oracle's: 128 * 2^-24 of the result's scale, and a few
# exponentials of sums of sixteen log decays, 16 * 2^-24 relative each; four times that
TOL = 4 * (128 + 16) * 2.0 ** -24


def i32(v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


def close(got, want, what, magnified=1.0):
    """``magnified``: by how much a row's own arithmetic enlarges the errors of its operands."""
    got, want = got.double().cpu(), want.double().cpu()
    scale = want.pow(2).mean().sqrt().clamp_min(1e-6)
    off = ((got - want).abs() / torch.maximum(scale, want.abs()) / magnified).max()
    assert torch.isfinite(got).all() and off < TOL, f"{what}: off by {off:.3g}"


def walk(cu, past, start, step, width):
    """float64: start(b, fresh) -> state, step(state, t) -> (state, row)."""
    out, states = torch.zeros(cu[-1], width, dtype=torch.float64), []
    for b in range(len(past)):
        s = start(b, past[b] == 0)
        for t in range(cu[b], cu[b + 1]):
            s, out[t] = step(s, t)
        states.append(s)
    return out, states


def batch():
    cu = [0]
    for n in LENS:
        cu.append(cu[-1] + n)
    past = [0 if i % 3 else 7 for i in range(len(LENS))]
    slots = [(5 * i + 2) % (len(LENS) + 1) for i in range(len(LENS))]      # a permutation with one slot left out
    assert len(set(slots)) == len(slots)
    return cu, past, slots


def pool(cu, past, slots, shape, make):
    """fp32 slots: what earlier tokens left where there are some, NaN where a request starts."""
    state = torch.full((len(slots) + 1, *shape), float("nan"))
    for b, slot in enumerate(slots):
        if past[b]:
            state[slot] = make()
    return state


@pytest.mark.parametrize("H,d,dv", [(2, 64, 128), (1, 128, 128), (3, 32, 64), (2, 20, 24), (1, 4, 4), (2, 100, 68), (1, 36, 128)])
@pytest.mark.parametrize("decay", ["slow", "mixed", "hard"])
def test_gated_linear_attention(H, d, dv, decay):
    from byox_vllm_amd import kernels
    torch.manual_seed(H * 1000 + d + dv)
    cu, past, slots = batch()
    T, tau, eps = cu[-1], 4.0, 1e-5
    proj = torch.randn(T, 2 * H * d + 2 * H * dv + 4)
    offs = (0, H * d, 2 * H * d, 2 * H * d + H * dv)
    z = {"slow": torch.randn(T, H * d) + 6.0, "mixed": 4.0 * torch.randn(T, H * d), "hard": 40.0 * torch.randn(T, H * d) - 40.0}[decay]
    w = torch.randn(dv)
    state = pool(cu, past, slots, (H, d, dv), lambda: torch.randn(H, d, dv))
    q, k, v, g = (proj[:, o:o + n].double().view(T, H, -1) for o, n in zip(offs, (H * d, H * d, H * dv, H * dv)))
    a = torch.sigmoid(z.double()).pow(1 / tau).view(T, H, d)

    def step(S, t):
        S = S * a[t][..., None] + k[t][..., None] * v[t][:, None]
        o = (S * q[t][..., None]).sum(1) * d ** -0.5
        o = o * torch.rsqrt(o.pow(2).mean(-1, keepdim=True) + eps) * w.double() * torch.nn.functional.silu(g[t])
        return S, o.reshape(-1)
    want, ends = walk(cu, past, lambda b, fresh: torch.zeros(H, d, dv, dtype=torch.float64) if fresh else state[slots[b]].double(),
                      step, H * dv)
    dev = state.to(DEV)
    got = kernels.gla_recurrent(proj.to(DEV), offs, z.to(DEV), dev, i32(cu), i32(past), i32(slots), w.to(DEV), H, d, dv, tau,
                                d ** -0.5, eps)
    close(got, want, "rows")
    close(torch.stack([dev[s] for s in slots]), torch.stack(ends), "states")
    # the token-by-token kernel on the same arguments
    from byox_vllm_amd._C import check, lib, ptr, stream
    dev2, out2 = state.to(DEV), torch.empty_like(got)
    p, zz, ww, args = proj.to(DEV), z.to(DEV), w.to(DEV), [i32(cu), i32(past), i32(slots)]
    check(lib().nv_gla_recurrent(ptr(p), p.stride(0), *offs, ptr(zz), zz.stride(0), ptr(dev2), *map(ptr, args), ptr(ww), ptr(out2),
                                 len(LENS), H, d, dv, tau, d ** -0.5, eps, 2, stream()), "nv_gla_recurrent")
    close(got, out2, "rows against the walk")
