"""What the float64 comparison of csrc/chunk_parts.h can see (chunk_parts_cases.py): the six products stay far inside its bound, and every one
of them left out goes past it."""

import pytest

import chunk_parts_cases as C


def results(kept):
    """Rows from values as they are, states from values over their weights."""
    out = []
    for weighted in (False, True):
        q, k, v, state, *raw = C.state_space_case(weighted)
        step, lf = C.steps_and_decays(*raw)
        out.append(C.recurrence(q, k, v, state, lf, step, False, kept=kept)[weighted])
        q, k, v, state, n, m, i, f, cap = C.gates_case(weighted)
        i, f = C.capped_gates(i, f, cap)
        out.append(C.recurrence(q, k, v, state, f, i, True, m.double(), n, kept=kept)[weighted])
    return out


def test_the_six_products():
    for got, want in zip(results(C.KEPT), results(None)):
        assert C.error(got, want) < 0.1 * C.BOUND


@pytest.mark.parametrize("left_out", C.KEPT)
def test_five_of_them(left_out):
    for got, want in zip(results([p for p in C.KEPT if p != left_out]), results(None)):
        assert C.error(got, want) > 1.5 * C.BOUND
