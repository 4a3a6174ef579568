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


def batch(lens=LENS):
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    past = [0 if i % 3 else 7 for i in range(len(lens))]
    slots = [(5 * i + 2) % (len(lens) + 1) for i in range(len(lens))]      # a permutation with one slot left out
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
@pytest.mark.parametrize("lens", [LENS, [400], [63, 64, 65, 257, 2], [1, 129, 300]])       # the last three: runs side by side
def test_gated_linear_attention(H, d, dv, decay, lens):
    from byox_vllm_amd import kernels
    torch.manual_seed(H * 1000 + d + dv)
    cu, past, slots = batch(lens)
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
                                d ** -0.5, eps, max_q=max(lens))
    close(got, want, "rows")
    close(torch.stack([dev[s] for s in slots]), torch.stack(ends), "states")
    # the token-by-token kernel on the same arguments
    from byox_vllm_amd._C import check, lib, ptr, stream
    dev2, out2 = state.to(DEV), torch.empty_like(got)
    p, zz, ww, args = proj.to(DEV), z.to(DEV), w.to(DEV), [i32(cu), i32(past), i32(slots)]
    check(lib().nv_gla_recurrent(ptr(p), p.stride(0), *offs, ptr(zz), zz.stride(0), ptr(dev2), *map(ptr, args), ptr(ww), ptr(out2),
                                 len(lens), H, d, dv, tau, d ** -0.5, eps, 2, stream()), "nv_gla_recurrent")
    close(got, out2, "rows against the walk")


@pytest.mark.parametrize("H,d,dv", [(2, 64, 128), (1, 128, 128), (3, 32, 64), (2, 20, 24), (1, 4, 4), (2, 100, 68), (1, 36, 128)])
@pytest.mark.parametrize("forget", [4.0, 0.0, -30.0])
def test_exponential_gates(H, d, dv, forget, monkeypatch):
    from byox_vllm_amd import kernels
    torch.manual_seed(H * 1000 + d + dv)
    cu, past, slots = batch()
    T, cap, copies = cu[-1], 15.0, -(-dv // 64)
    cols = 2 * H * d + H * dv
    proj, bias = torch.randn(T, cols + 2 * H + (-(cols + 2 * H)) % 4), torch.zeros(cols + 2 * H)
    proj[:, cols:] *= 3.0
    bias[cols:cols + H], bias[cols + H:] = -1.0, forget

    def start():
        n, m = torch.randn(H, d), torch.randn(H, 1)
        return torch.cat([torch.randn(H, d * dv)] + [n, m] * copies, 1)
    state = pool(cu, past, slots, (H, d * dv + copies * (d + 1)), start)
    q, k, v = (proj[:, o:o + n].double().view(T, H, -1) for o, n in ((0, H * d), (H * d, H * d), (2 * H * d, H * dv)))
    i, f = (cap * torch.tanh((proj[:, o:o + H] + bias[o:o + H]).double() / cap) for o in (cols, cols + H))
    f = torch.nn.functional.logsigmoid(f)

    def unpack(b, fresh):
        if fresh:
            return [torch.zeros(s, dtype=torch.float64) for s in ((H, d, dv), (H, d), (H,))]
        s = state[slots[b]].double()
        return [s[:, :d * dv].reshape(H, d, dv), s[:, d * dv:d * dv + d], s[:, d * dv + d]]

    def step(s, t):
        S, n, m = s
        top = torch.maximum(f[t] + m, i[t])
        keep, take = torch.exp(f[t] + m - top), torch.exp(i[t] - top)
        S = S * keep[:, None, None] + take[:, None, None] * k[t][..., None] * v[t][:, None]
        n = n * keep[:, None] + take[:, None] * k[t]
        below = torch.maximum((n * q[t]).sum(-1).abs() * d ** -0.5, torch.exp(-top)) + 1e-6
        # a sum n . q that nearly cancels is divided by: its terms' errors come out enlarged
        magnified[t] = ((n * q[t]).abs().sum(-1) * d ** -0.5 / below).clamp_min(1.0)
        return [S, n, top], ((S * q[t][..., None]).sum(1) * d ** -0.5 / below[:, None]).reshape(-1)
    magnified = torch.ones(T, H, dtype=torch.float64)
    want, ends = walk(cu, past, unpack, step, H * dv)
    ends = torch.stack([torch.cat([S.reshape(H, -1)] + [n, m[:, None]] * copies, 1) for S, n, m in ends])

    def run():
        dev = state.to(DEV)
        out = kernels.matrix_memory(proj.to(DEV), (0, H * d, 2 * H * d), dev, i32(cu), i32(past), i32(slots), H, d, dv,
                                    kernels.MEM_EXPGATE, bias=bias.to(DEV), gate_offsets=(cols, cols + H), cap=cap,
                                    q_scale=d ** -0.5, max_q=max(LENS))
        return out, torch.stack([dev[s] for s in slots])
    got, state_got = run()
    monkeypatch.setenv("NV_MATRIX_MEMORY_STEPS", "1")
    steps, state_steps = run()
    magnified = magnified.repeat_interleave(dv, 1)
    close(got, want, "rows", magnified)
    close(got, steps, "rows against the walk", magnified)
    close(state_got, ends, "states")
    close(state_got, state_steps, "states against the walk")


@pytest.mark.parametrize("H,G,n,dv", [(4, 1, 128, 64), (4, 2, 64, 64), (2, 2, 16, 128), (2, 1, 20, 24), (6, 3, 4, 4), (2, 1, 100, 68)])
@pytest.mark.parametrize("scale", [0.1, 3.0, 100.0])
def test_state_space(H, G, n, dv, scale):
    from byox_vllm_amd import kernels
    torch.manual_seed(H * 1000 + n + dv)
    cu, past, slots = batch()
    T, inner = cu[-1], H * dv
    xbc, z, dt = torch.randn(T, inner + 2 * G * n), torch.randn(T, inner), torch.randn(T, H)
    dt_bias, A_log, D = torch.randn(H), torch.randn(H) + torch.tensor(scale).log(), torch.randn(H)
    state = pool(cu, past, slots, (H, n, dv), lambda: torch.randn(H, n, dv))
    x = xbc[:, :inner].double().view(T, H, dv)
    B, C = (xbc[:, inner + o:inner + o + G * n].double().view(T, G, n).repeat_interleave(H // G, 1) for o in (0, G * n))
    step_size = torch.nn.functional.softplus(dt.double() + dt_bias.double())
    keep = torch.exp(-torch.exp(A_log.double()) * step_size)

    def step(S, t):
        S = S * keep[t][:, None, None] + (step_size[t][:, None] * B[t])[..., None] * x[t][:, None]
        y = ((S * C[t][..., None]).sum(1) + D.double()[:, None] * x[t]).reshape(-1)
        return S, y * torch.nn.functional.silu(z[t].double())
    want, ends = walk(cu, past, lambda b, fresh: torch.zeros(H, n, dv, dtype=torch.float64) if fresh else state[slots[b]].double(),
                      step, inner)
    runs = []
    for max_q in (max(LENS), 1):            # chunks; the walk
        dev = state.to(DEV)
        out = kernels.ssd_scan(xbc.to(DEV), z.to(DEV), dt.to(DEV), dt_bias.to(DEV), A_log.to(DEV), D.to(DEV), dev, i32(cu),
                               i32(past), i32(slots), H, G, n, dv, max_q=max_q)
        runs.append((out, torch.stack([dev[s] for s in slots])))
    close(runs[0][0], want, "rows")
    close(runs[0][1], torch.stack(ends), "states")
    close(runs[0][0], runs[1][0], "rows against the walk")


@pytest.mark.parametrize("H,n,dv", [(8, 128, 16), (8, 128, 64), (8, 32, 16), (8, 64, 32), (2, 128, 128)])
@pytest.mark.parametrize("longest", [2, 3, 17, 70])
def test_state_space_steps_of_single_tokens_and_a_piece(H, n, dv, longest):
    """Many decoding requests beside one piece, whichever of the two forms the step takes, against the walk asked for by max_q 1."""
    from byox_vllm_amd import kernels
    torch.manual_seed(n + dv + longest)
    lens = [1] * 70 + [longest]
    cu, past, slots = batch(lens)
    T, inner = cu[-1], H * dv
    data = [torch.randn(s, device=DEV) for s in ((T, inner + 2 * n), (T, inner), (T, H), (H,), (H,), (H,))]
    state = pool(cu, past, slots, (H, n, dv), lambda: torch.randn(H, n, dv)).to(DEV)
    runs = []
    for max_q in (longest, 1):
        dev = state.clone()
        out = kernels.ssd_scan(*data, dev, i32(cu), i32(past), i32(slots), H, 1, n, dv, max_q=max_q)
        runs.append((out, torch.stack([dev[s] for s in slots])))
    close(runs[0][0], runs[1][0], "rows")
    close(runs[0][1], runs[1][1], "states")


@pytest.mark.parametrize("lens,past", [([256], [0]), ([257, 3], [5, 0]), ([511, 128, 129, 1], [0, 9, 0, 4])])
def test_state_space_runs(lens, past):
    """Few requests with long prompts: runs side by side against one walk over the same tokens."""
    from byox_vllm_amd import kernels
    torch.manual_seed(sum(lens))
    H, G, n, dv = 2, 1, 64, 64
    cu = [0]
    for m in lens:
        cu.append(cu[-1] + m)
    T, inner = cu[-1], H * dv
    data = [torch.randn(s, device=DEV) for s in ((T, inner + 2 * G * n), (T, inner), (T, H), (H,), (H,), (H,))]
    data[4] = data[4] - 2.0
    state = torch.randn(len(lens), H, n, dv, device=DEV)
    runs = []
    for max_q in (max(lens), 1):
        dev = state.clone()
        out = kernels.ssd_scan(*data, dev, i32(cu), i32(past), i32(list(range(len(lens)))), H, G, n, dv, max_q=max_q)
        runs.append((out, dev))
    close(runs[0][0], runs[1][0], "rows")
    close(runs[0][1], runs[1][1], "states")


@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("at", [0, 5, 15, 20, 38])
def test_a_value_that_is_not_finite_stays_out_of_earlier_rows(bad, at):
    """One number of one token's value row is an infinity or a NaN: the rows ahead of it, and the other request's, are what they
    are without it; the token's own row is not finite."""
    from byox_vllm_amd import kernels
    torch.manual_seed(at)
    H, d, dv, lens = 2, 64, 64, [39, 20]
    cu, T = [0, 39, 59], 59
    ints = i32(cu), i32([0, 0]), i32([0, 1])
    rows = torch.randn(T, 2 * H * d + 2 * H * dv + 2 * H, device=DEV)
    z, w = torch.randn(T, H * d, device=DEV), torch.ones(dv, device=DEV)
    vectors = [torch.randn(H, device=DEV) for _ in range(3)]
    at_v = 2 * H * d

    def gla(p):
        return kernels.gla_recurrent(p, (0, H * d, at_v, at_v + H * dv), z, torch.zeros(2, H, d, dv, device=DEV), *ints, w, H, d, dv,
                                     4.0, 1.0, 1e-5, max_q=39)

    def gates(p):
        state = torch.zeros(2, H, d * dv + d + 1, device=DEV)
        return kernels.matrix_memory(p, (0, H * d, at_v), state, *ints, H, d, dv, kernels.MEM_EXPGATE, max_q=39, cap=15.0,
                                     gate_offsets=(at_v + 2 * H * dv, at_v + 2 * H * dv + H))

    def ssd(p):          # values first in this layout
        xbc = torch.cat([p[:, at_v:at_v + H * dv], p[:, :2 * d]], 1).contiguous()
        return kernels.ssd_scan(xbc, p[:, at_v + H * dv:at_v + 2 * H * dv], p[:, -H:], *vectors, torch.zeros(2, H, d, dv, device=DEV),
                                *ints, H, 1, d, dv, max_q=39)
    for name, f in (("channel decays", gla), ("exponential gates", gates), ("state space", ssd)):
        want = f(rows)
        spoilt = rows.clone()
        spoilt[at, at_v + 3] = bad
        got = f(spoilt)
        close(got[:at] if at else got[39:], want[:at] if at else want[39:], f"{name}: rows ahead")
        close(got[39:], want[39:], f"{name}: the other request")
        assert not torch.isfinite(got[at]).all(), name


def test_one_row_for_every_token():
    """Rows expanded over the tokens (a row stride of 0) give what copies of the row give."""
    from byox_vllm_amd import kernels
    torch.manual_seed(2)
    H, d, dv, lens = 2, 64, 64, [21, 5]
    cu, T = [0, 21, 26], 26
    ints = i32(cu), i32([0, 0]), i32([0, 1])
    row = torch.randn(1, 2 * H * d + 2 * H * dv, device=DEV).expand(T, -1)
    xbc = torch.randn(1, H * dv + 2 * d, device=DEV).expand(T, -1)
    z, dt, w = torch.randn(T, H * d, device=DEV), torch.randn(T, H, device=DEV), torch.ones(dv, device=DEV)
    vectors = [torch.randn(H, device=DEV) for _ in range(3)]
    gates = torch.randn(T, H * dv, device=DEV)
    for name in ("channel decays", "state space"):
        runs = []
        for copy in (False, True):
            state = torch.zeros(2, H, d, dv, device=DEV)
            if name == "state space":
                out = kernels.ssd_scan(xbc.contiguous() if copy else xbc, gates, dt, *vectors, state, *ints, H, 1, d, dv,
                                       max_q=max(lens))
            else:
                out = kernels.gla_recurrent(row.contiguous() if copy else row, (0, H * d, 2 * H * d, 2 * H * d + H * dv), z, state,
                                            *ints, w, H, d, dv, 4.0, 1.0, 1e-5, max_q=max(lens))
            runs.append((out, state))
        close(runs[0][0], runs[1][0], f"{name}: rows")
        close(runs[0][1], runs[1][1], f"{name}: states")
