"""Numbers for csrc/chunk_parts.h and its two recurrences in float64, in chunks of thirty-two tokens, each matrix product either whole or as
the sum of some of the nine products of three bf16 parts per number."""

import math

import torch

CHUNK = 32
KEPT = ((0, 0), (0, 1), (1, 0), (0, 2), (1, 1), (2, 0))      # parts of the two factors whose products the kernel adds up
# What may be off, of the norm.  A sum over K channels or tokens adds 6 K / 32 times what the matrix instruction summed exactly, each time to a
# number of at most the result's size here, where nothing cancels: their roundings add up as a random walk, K = 128 channels and then 32 tokens,
# and the chunks' states four times over.  Exponentials of sums of log decays, the steps or gates in front of them, SiLU or quotient: 8 units.
BOUND = (math.sqrt(6 * 128 / 32) + math.sqrt(6 * 32 / 32) * 2 + 8) * 2.0 ** -24


def positive(shape, seed):
    """Positive fp32 numbers whose second and third parts are nearly as large as can be, and positive: a product of parts that is left out
    shows in every sum with the same sign."""
    g = torch.Generator().manual_seed(seed)
    h = (torch.rand(shape, generator=g) + 0.5).to(torch.bfloat16).double()
    ulp = torch.exp2(torch.floor(torch.log2(h)) - 7)
    m = (0.49 * ulp).to(torch.bfloat16).double()
    return (h + m + 0.49 * torch.exp2(torch.floor(torch.log2(m)) - 7)).float()


def parts(x):
    x = x.float()
    h = x.to(torch.bfloat16).float()
    m = (x - h).to(torch.bfloat16).float()
    return [p.double() for p in (h, m, (x - h - m).to(torch.bfloat16).float())]


def product(a, b, kept):
    if kept is None:
        return a @ b
    pa, pb = parts(a), parts(b)
    return sum(pa[i] @ pb[j] for i, j in kept)


def recurrence(q, k, v, state, lf, weight, log_gate, m0=None, n0=None, kept=None):
    """One head, float64: q, k [T, d], v [T, dv], log decays lf [T].  ``log_gate`` False: weights are step sizes, -> (rows, state).  True: logs
    of exponential gates, with the running maximum m0 and the normaliser n0, -> (normalised rows, state, normaliser, maximum)."""
    q, k, v, S, lf, weight = (x.double() for x in (q, k, v, state, lf, weight))
    rows = []
    for c in range(0, q.size(0), CHUNK):
        a, b, x, F, g = q[c:c + CHUNK], k[c:c + CHUNK], v[c:c + CHUNK], lf[c:c + CHUNK].cumsum(0), weight[c:c + CHUNK]
        later = torch.ones(len(F), len(F), dtype=torch.bool).triu(1)
        if log_gate:
            m = F + torch.maximum(m0, torch.cummax(g - F, 0).values)
            between = torch.exp(F[:, None] - F[None] + g[None] - m[:, None])
            front, w, whole = torch.exp(F + m0 - m), torch.exp(F[-1] - F + g - m[-1]), torch.exp(F[-1] + m0 - m[-1])
        else:
            between, front, w, whole = torch.exp(F[:, None] - F[None]) * g[None], torch.exp(F), g * torch.exp(F[-1] - F), torch.exp(F[-1])
        P = product(a, b.t(), kept).mul(between).masked_fill(later, 0.0)
        o = front[:, None] * product(a, S, kept) + product(P, x, kept)
        if log_gate:
            below = torch.maximum((P.sum(1) + front * (a @ n0.double())).abs(), torch.exp(-m)) + 1e-6
            o = o / below[:, None]
            n0, m0 = whole * n0 + (w[:, None] * b).sum(0), m[-1]
        rows.append(o)
        S = whole * S + product(b.t(), w[:, None] * x, kept)
    return (torch.cat(rows), S, n0, m0) if log_gate else (torch.cat(rows), S)


def error(got, want):
    return ((got.double().cpu() - want).norm() / want.norm()).item()


def over(v, w):
    """v, divided by what weighs it into the state: there its parts are as large as v's own."""
    return (v.double() / w[:, None]).float()


def into_state(lf, weight, log_gate, m0):
    """What a token's value is multiplied by on its way into the state behind its chunk."""
    out = []
    for c in range(0, len(lf), CHUNK):
        F, g = lf[c:c + CHUNK].cumsum(0), weight[c:c + CHUNK]
        if log_gate:
            m = F[-1] + torch.maximum(m0, (g - F).max())
            out.append(torch.exp(F[-1] - F + g - m))
            m0 = m
        else:
            out.append(g * torch.exp(F[-1] - F))
    return torch.cat(out)


def state_space_case(weighted):
    """One head of 128 x 64, 97 tokens: q, k, v, state, raw step sizes, their bias, A_log, all fp32.  ``weighted``: values over their weights."""
    T, d, dv = 97, 128, 64
    q, k, v, state = (positive(s, i) for i, s in enumerate(((T, d), (T, d), (T, dv), (d, dv))))
    dt = torch.randn(T, generator=torch.Generator().manual_seed(9)) - 2.0
    bias, A_log = torch.tensor(0.3), torch.tensor(-0.7)
    step, lf = steps_and_decays(dt, bias, A_log)
    return q, k, over(v, into_state(lf, step, False, None)) if weighted else v, state, dt, bias, A_log


def steps_and_decays(dt, bias, A_log):
    step = torch.nn.functional.softplus(dt.double() + bias.double())
    return step, -torch.exp(A_log.double()) * step


def gates_case(weighted):
    """One head of 128 x 64, 97 tokens: q (scaled), k, v, state, normaliser, maximum, input- and forget-gate logits, fp32, and their cap."""
    T, d, dv, cap = 97, 128, 64, 15.0
    q, k, v, state, n = (positive(s, 10 + i) for i, s in enumerate(((T, d), (T, d), (T, dv), (d, dv), (d,))))
    g = torch.Generator().manual_seed(19)
    m, i, f = torch.tensor(0.25), torch.randn(T, generator=g), torch.randn(T, generator=g) + 2.0
    gate, lf = capped_gates(i, f, cap)
    return q, k, over(v, into_state(lf, gate, True, m.double())) if weighted else v, state, n, m, i, f, cap


def capped_gates(i, f, cap):
    return cap * torch.tanh(i.double() / cap), torch.nn.functional.logsigmoid(cap * torch.tanh(f.double() / cap))
