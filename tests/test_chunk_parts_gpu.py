"""Scalar decays in chunks of thirty-two tokens (csrc/chunk_parts.h), which the launches take where they know of twenty tokens and more to
a request, against the chunks of sixteen, which they take where they know nothing; at the edges of both, and which steps go where."""

import pytest
import torch

import chunk_parts_cases as C

pytestmark = pytest.mark.gpu
DEV = "cuda"
LENS = [1, 31, 32, 33, 63, 64, 65, 97]
# fp32 products and sums of up to 128 terms in two orders, and exponentials of sums of 32 and of 16 log decays: twice that of one against
# float64 (test_chunk_scan_gpu.py)
TOL = 2 * 4 * (128 + 32) * 2.0 ** -24


def i32(v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


def close(got, want, magnified=1.0):
    got, want = got.double(), want.double()
    off = ((got - want).abs() / torch.maximum(want.pow(2).mean().sqrt(), want.abs()) / magnified).max().item()
    assert torch.isfinite(got).all() and off < TOL, off


def state_space(xbc, z, dt, dt_bias, A_log, D, state, ints, lens, H, G, n, dv, tokens, runs=False):
    """nv_ssd_scan_batch -> rows; the state in place."""
    from byox_vllm_amd._C import check, lib, ptr, stream
    from byox_vllm_amd.kernels import workspace
    need = lib().nv_ssd_scan_workspace_bytes(len(lens), H, n, dv, max(lens)) if runs else 0
    ws = workspace(need, torch.device(DEV, 0), "ssd_scan") if need else None
    out = torch.empty(xbc.size(0), H * dv, device=DEV)
    check(lib().nv_ssd_scan_batch(ptr(xbc), xbc.stride(0), ptr(z), z.stride(0), ptr(dt), dt.stride(0), ptr(dt_bias), ptr(A_log), ptr(D),
                                  ptr(state), *map(ptr, ints), ptr(out), tokens, len(lens), H, G, n, dv, max(lens), ptr(ws), need, 2,
                                  stream()), "nv_ssd_scan_batch")
    return out


def gated(proj, bias, state, ints, lens, H, d, dv, tokens, q_scale=1.0):
    """nv_matrix_memory_batch with exponential gates, rows q | k | v | i | f -> rows; the state in place."""
    from byox_vllm_amd import kernels
    from byox_vllm_amd._C import check, lib, ptr, stream
    cols, out = 2 * H * d + H * dv, torch.empty(proj.size(0), H * dv, device=DEV)
    check(lib().nv_matrix_memory_batch(ptr(proj), proj.stride(0), 0, H * d, 2 * H * d, cols, cols + H, ptr(bias), None, ptr(state),
                                       *map(ptr, ints), ptr(out), out.stride(0), tokens, len(lens), H, d, dv, kernels.MEM_EXPGATE, 0,
                                       q_scale, 1.0, None, 0, 15.0, max(lens), 2, stream()), "nv_matrix_memory_batch")
    return out


def padded(*columns):
    """Columns side by side, rows of a multiple of four numbers."""
    x = torch.cat(columns, 1)
    return torch.cat([x, x.new_zeros(x.size(0), -x.size(1) % 4)], 1).to(DEV)


def both(run, lens, state):
    """``run(tokens, state, ints)`` -> rows; without the number of tokens and with it."""
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    past = [0 if i % 3 else 7 for i in range(len(lens))]
    ints = [i32(cu), i32(past), i32([len(lens) - 1 - i for i in range(len(lens))])]
    results = []
    for tokens in (0, cu[-1]):
        s = state.clone()
        results.append((run(tokens, s, ints), s))
    return results


@pytest.mark.parametrize("H,G,n,dv", [(4, 1, 128, 64), (4, 2, 64, 64), (2, 2, 16, 128), (2, 1, 20, 24), (3, 3, 4, 4), (2, 1, 100, 68),
                                      (2, 1, 128, 128)])
@pytest.mark.parametrize("lens", [LENS, [300, 257]])       # the last: runs side by side
def test_state_space(H, G, n, dv, lens):
    from byox_vllm_amd._C import check, lib, ptr, stream
    from byox_vllm_amd.kernels import workspace
    torch.manual_seed(n + dv)
    T, inner = sum(lens), H * dv
    xbc, z, dt = (torch.randn(T, c, device=DEV) for c in (inner + 2 * G * n, inner, H))
    dt_bias, A_log, D = (torch.randn(H, device=DEV) for _ in range(3))
    need = lib().nv_ssd_scan_workspace_bytes(len(lens), H, n, dv, max(lens))
    ws = workspace(need, torch.device(DEV, 0), "ssd_scan") if need else None

    def run(tokens, state, ints):
        out = torch.empty(T, inner, device=DEV)
        check(lib().nv_ssd_scan_batch(ptr(xbc), xbc.stride(0), ptr(z), z.stride(0), ptr(dt), dt.stride(0), ptr(dt_bias), ptr(A_log), ptr(D),
                                      ptr(state), *map(ptr, ints), ptr(out), tokens, len(lens), H, G, n, dv, max(lens), ptr(ws), need, 2,
                                      stream()), "nv_ssd_scan_batch")
        return out
    (rows, state), (rows_parts, state_parts) = both(run, lens, torch.randn(len(lens), H, n, dv, device=DEV))
    close(rows_parts, rows)
    close(state_parts, state)
    assert not torch.equal(rows_parts, rows)       # two forms indeed


@pytest.mark.parametrize("H,d,dv", [(2, 64, 128), (1, 128, 128), (3, 32, 64), (2, 20, 24), (1, 4, 4), (2, 100, 68), (1, 36, 128), (2, 64, 64)])
@pytest.mark.parametrize("forget", [4.0, -30.0])
def test_exponential_gates(H, d, dv, forget):
    from byox_vllm_amd import kernels
    from byox_vllm_amd._C import check, lib, ptr, stream
    torch.manual_seed(d + dv)
    T, cols = sum(LENS), 2 * H * d + H * dv
    proj = torch.randn(T, cols + 2 * H + (-(cols + 2 * H)) % 4, device=DEV)
    proj[:, cols:] *= 3.0
    bias = torch.zeros(cols + 2 * H, device=DEV)
    bias[cols:cols + H], bias[cols + H:] = -1.0, forget
    per_head = kernels.matrix_memory_state_size(kernels.MEM_EXPGATE, d, dv)
    state = torch.randn(len(LENS), H, per_head, device=DEV)
    slices = -(-dv // 64)
    for c in range(1, slices):      # the normaliser and the maximum lie there once per slice of 64 columns
        state[..., d * dv + c * (d + 1):d * dv + (c + 1) * (d + 1)] = state[..., d * dv:d * dv + d + 1]

    def run(tokens, s, ints):
        out = torch.empty(T, H * dv, device=DEV)
        check(lib().nv_matrix_memory_batch(ptr(proj), proj.stride(0), 0, H * d, 2 * H * d, cols, cols + H, ptr(bias), None, ptr(s),
                                           *map(ptr, ints), ptr(out), out.stride(0), tokens, len(LENS), H, d, dv, kernels.MEM_EXPGATE, 0,
                                           d ** -0.5, 1.0, None, 0, 15.0, max(LENS), 2, stream()), "nv_matrix_memory_batch")
        return out
    (rows, end), (rows_parts, end_parts) = both(run, LENS, state)
    # a row is divided by a sum n . q that may nearly cancel, which enlarges its errors: rows of like size
    calm = (rows.abs() < 8.0).view(T, H, dv).all(-1, keepdim=True).expand(-1, -1, dv).reshape(T, -1)
    assert calm.float().mean() > 0.5
    close(torch.where(calm, rows_parts, 0.0), torch.where(calm, rows, 0.0), 16.0)
    close(end_parts, end)
    assert not torch.equal(rows_parts, rows)


def test_the_line_between_them():
    """Steps of 20 tokens to a request on average and more."""
    from byox_vllm_amd import kernels
    torch.manual_seed(1)
    H, n, dv = 2, 64, 64
    for lens, parts in (([20, 20], True), ([20, 19], False), ([59, 1], True), ([58, 1, 1], True), ([57, 1, 1], False)):
        T, B = sum(lens), len(lens)
        cu = [0]
        for m in lens:
            cu.append(cu[-1] + m)
        data = [torch.randn(s, device=DEV) for s in ((T, H * dv + 2 * n), (T, H * dv), (T, H), (H,), (H,), (H,))]
        state, ints = torch.randn(B, H, n, dv, device=DEV), (i32(cu), i32([3] * B), i32(list(range(B))))
        got = kernels.ssd_scan(*data, state.clone(), *ints, H, 1, n, dv, max_q=max(lens))
        from byox_vllm_amd._C import check, lib, ptr, stream
        sixteen, s = torch.empty_like(got), state.clone()
        check(lib().nv_ssd_scan(*(a for x in data[:3] for a in (ptr(x), x.stride(0))), *map(ptr, data[3:]), ptr(s), *map(ptr, ints),
                                ptr(sixteen), B, H, 1, n, dv, max(lens), None, 0, 2, stream()), "nv_ssd_scan")
        assert torch.equal(got, sixteen) != parts, lens


# powers of two that q, k and v are multiplied by: numbers whose second and third parts would lie below the range of bf16
SCALES = [(0, 0, 0), (110, -118, 0), (-118, 60, 0), (0, 0, -119), (100, -70, -60)]


@pytest.mark.parametrize("scales", SCALES)
@pytest.mark.parametrize("weighted", [False, True])
def test_state_space_as_close_as_fp32(scales, weighted):
    q, k, v, state, dt, bias, A_log = C.state_space_case(weighted)
    a, b, c = (2.0 ** e for e in scales)
    q, k, v, state = q * a, k * b, v * c, state * b * c
    step, lf = C.steps_and_decays(dt, bias, A_log)
    want, end = C.recurrence(q, k, v, state, lf, step, False)
    T, (d, dv) = q.size(0), state.shape
    z, s = torch.ones(T, dv, device=DEV), state.to(DEV).view(1, 1, d, dv).clone()
    got = state_space(padded(v, k, q), z, dt.view(T, 1).to(DEV), bias.view(1).to(DEV), A_log.view(1).to(DEV), torch.zeros(1, device=DEV), s,
                      [i32([0, T]), i32([5]), i32([0])], [T], 1, 1, d, dv, T)
    errors = C.error(got, want * torch.nn.functional.silu(torch.ones((), dtype=torch.float64))), C.error(s.view(d, dv), end)
    assert max(errors) < C.BOUND, errors


@pytest.mark.parametrize("scales", SCALES)
@pytest.mark.parametrize("weighted", [False, True])
def test_exponential_gates_as_close_as_fp32(scales, weighted):
    q, k, v, state, n, m, i, f, cap = C.gates_case(weighted)
    a, b, c = (2.0 ** e for e in scales)
    q, k, v, state, n = q * a, k * b, v * c, state * b * c, n * b
    gate, lf = C.capped_gates(i, f, cap)
    want, end, n_end, m_end = C.recurrence(q, k, v, state, lf, gate, True, m.double(), n)
    T, (d, dv) = q.size(0), state.shape
    s = torch.cat([state.reshape(-1), n, m.view(1)]).to(DEV).view(1, 1, -1).clone()
    got = gated(padded(q, k, v, i.view(T, 1), f.view(T, 1)), None, s, [i32([0, T]), i32([5]), i32([0])], [T], 1, d, dv, T)
    s = s.view(-1)
    errors = C.error(got, want), C.error(s[:d * dv].view(d, dv), end), C.error(s[d * dv:-1], n_end)
    assert max(errors) < C.BOUND and abs(s[-1].item() - m_end.item()) < 2.0 ** -20, errors


def same(a, b):
    return torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(0.0), b.nan_to_num(0.0))


PLACES = [("q", float("inf")), ("k", float("-inf")), ("v", float("inf")), ("v", float("nan")), ("v", 3.4e38), ("k", 3.4e38), ("q", 1e34),
          ("state", float("inf")), ("state", 3.4e38)]


def numbers_without_parts(place, value, run, H, of):
    """``run(tokens, put)`` -> rows [T, H, *], states [B, H, *] with ``put`` ahead of it: one number of one request's second head.  That
    head's rows and states are those of the sixteen-token chunks, all others what they are without it."""
    clean, dirty, sixteen = (run(t, p) for t, p in ((True, False), (True, True), (False, True)))
    for (a, b, c), mine in zip(zip(clean, dirty, sixteen), of):
        mine = torch.stack([torch.zeros_like(mine), mine], 1).view(b.size(0), H)
        assert same(b[~mine], a[~mine]) and same(b[mine], c[mine]) and not same(b[mine], a[mine])
    assert not all(x.isfinite().all() for x in dirty) or abs(value) < float("inf")


@pytest.mark.parametrize("n,dv", [(64, 64), (128, 64), (128, 128), (32, 24)])
@pytest.mark.parametrize("place,value", PLACES)
def test_state_space_numbers_without_parts(n, dv, place, value):
    torch.manual_seed(n + dv)
    H, lens, hit = 2, [1, 97, 65, 40], 2
    B, T, inner, at = len(lens), sum(lens), H * dv, sum(lens[:hit]) + 37
    xbc, z, dt = (torch.randn(T, c, device=DEV) for c in (inner + 2 * H * n, inner, H))
    head, state = [torch.randn(H, device=DEV) for _ in range(3)], torch.randn(B, H, n, dv, device=DEV)
    cu = [sum(lens[:i]) for i in range(B + 1)]
    ints = [i32(cu), i32([3] * B), i32(list(range(B)))]

    def run(tokens, put):
        x, s = xbc.clone(), state.clone()
        if put and place == "state":
            s[hit, 1, 3, 5] = value
        elif put:
            x[at, {"v": dv, "k": inner + n, "q": inner + H * n + n}[place] + 5] = value
        rows = state_space(x, z, dt, *head, s, ints, lens, H, H, n, dv, T if tokens else 0)
        return rows.view(T, H, dv), s
    seq = torch.tensor([b for b, m in enumerate(lens) for _ in range(m)], device=DEV)
    request = torch.arange(B, device=DEV) == hit
    if place == "q":      # the state does not depend on it
        clean, dirty = run(True, False), run(True, True)
        assert same(dirty[1][request][:, 1], run(False, True)[1][request][:, 1]) and same(dirty[0][:, 0], clean[0][:, 0])
        assert same(dirty[0][seq == hit][:, 1], run(False, True)[0][seq == hit][:, 1]) and not same(dirty[0], clean[0])
        return
    numbers_without_parts(place, value, run, H, (seq == hit, request))


@pytest.mark.parametrize("d,dv", [(64, 64), (128, 64), (64, 128), (128, 128), (32, 24)])
@pytest.mark.parametrize("place,value", PLACES)
def test_exponential_gates_numbers_without_parts(d, dv, place, value):
    from byox_vllm_amd import kernels
    torch.manual_seed(d + dv)
    H, lens, hit = 2, [1, 97, 65, 40], 2
    B, T, at = len(lens), sum(lens), sum(lens[:hit]) + 37
    proj = padded(torch.randn(T, 2 * H * d + H * dv + 2 * H))
    state = torch.randn(B, H, kernels.matrix_memory_state_size(kernels.MEM_EXPGATE, d, dv), device=DEV)
    cu = [sum(lens[:i]) for i in range(B + 1)]
    ints = [i32(cu), i32([3] * B), i32(list(range(B)))]

    def run(tokens, put):
        x, s = proj.clone(), state.clone()
        if put and place == "state":
            s[hit, 1, 3 * dv + 5] = value
        elif put:
            x[at, {"q": d, "k": H * d + d, "v": 2 * H * d + dv}[place] + 5] = value
        rows = gated(x, None, s, ints, lens, H, d, dv, T if tokens else 0)
        return rows.view(T, H, dv), s
    seq = torch.tensor([b for b, m in enumerate(lens) for _ in range(m)], device=DEV)
    request = torch.arange(B, device=DEV) == hit
    if place == "q":
        clean, dirty, sixteen = run(True, False), run(True, True), run(False, True)
        assert same(dirty[1][request][:, 1], sixteen[1][request][:, 1]) and same(dirty[0][:, 0], clean[0][:, 0])
        assert same(dirty[0][seq == hit][:, 1], sixteen[0][seq == hit][:, 1]) and not same(dirty[0], clean[0])
        return
    numbers_without_parts(place, value, run, H, (seq == hit, request))


@pytest.mark.parametrize("place", ["k", "v", "state"])
def test_infinities_in_runs_side_by_side(place):
    """A run that meets one is walked again; what it leaves reaches the runs behind it."""
    torch.manual_seed(7)
    H, n, dv, lens = 2, 64, 64, [300, 257]
    T, inner = sum(lens), H * dv
    xbc, z, dt = (torch.randn(T, c, device=DEV) for c in (inner + 2 * H * n, inner, H))
    head, state = [torch.randn(H, device=DEV) - 2.0 for _ in range(3)], torch.randn(2, H, n, dv, device=DEV)
    if place == "state":
        state[0, 0, 5, 7] = float("inf")
    else:
        xbc[120, 7 if place == "v" else inner + 5] = float("inf")
    results = []
    for tokens in (T, 0):
        s = state.clone()
        results.append((state_space(xbc, z, dt, *head, s, [i32([0, 300, 557]), i32([3, 3]), i32([0, 1])], lens, H, H, n, dv, tokens, True), s))
    for got, want in zip(*results):
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf()) and not want.isfinite().all()
        assert torch.equal(got[got.isinf()], want[want.isinf()])
        close(torch.where(want.isfinite(), got, 0.0), torch.where(want.isfinite(), want, 0.0))
