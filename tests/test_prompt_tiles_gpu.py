"""Prompt attention's walk over tiles of 64 keys (csrc/prompt_attn.h): kept first keys in a tile of their own or in the places ahead of
the window's first key, pages that hold whole tiles and pages that do not, last tiles that end inside a page nobody has filled, and
queries in bf16."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def i32(v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


@pytest.mark.parametrize("block", [64, 192, 256, 48])
@pytest.mark.parametrize("D,R", [(64, 1), (64, 4), (128, 1), (128, 2)])
@pytest.mark.parametrize("window,keep", [(0, 0), (64, 0), (100, 1), (128, 16), (65, 63), (90, 64), (70, 130), (300, 37)])
def test_windows_and_kept_keys(D, R, window, keep, block):
    from byox_vllm_amd import kernels
    torch.manual_seed(window + keep + D)
    new, past, G = [130, 1, 70, 200], [0, 511, 301, 64 * 5 + 33], 2
    H, pages = R * G, [-(-(a + b) // block) for a, b in zip(new, past)]
    order, tables, T = torch.randperm(sum(pages)).tolist(), [], sum(new)
    for n in pages:
        tables.append([order.pop() for _ in range(n)])
    cache = torch.randn(sum(pages) * block, 2 * G * D).to(torch.bfloat16)
    for b, t in enumerate(tables):      # rows that nobody has written
        filled = past[b] + new[b] - (pages[b] - 1) * block
        cache[t[-1] * block + filled:(t[-1] + 1) * block] = float("nan")
    cu = [0]
    for n in new:
        cu.append(cu[-1] + n)
    q = (torch.randn(T, H * D) * 2.0 * D ** -0.5).to(torch.bfloat16)
    want = torch.zeros(T, H, D, dtype=torch.float64)
    for b, t in enumerate(tables):
        n = past[b] + new[b]
        rows = torch.cat([cache[p * block:(p + 1) * block] for p in t])[:n].double()
        k, v = rows[:, :G * D].view(n, G, D), rows[:, G * D:].view(n, G, D)
        i, j = torch.arange(past[b], n)[:, None], torch.arange(n)[None]
        seen = j <= i
        if window:
            seen &= (i - j < window) | (j < keep)
        for h in range(H):
            s = (q[cu[b]:cu[b + 1]].double().view(-1, H, D)[:, h] @ k[:, h // R].t()).masked_fill(~seen, float("-inf"))
            want[cu[b]:cu[b + 1], h] = torch.softmax(s, -1) @ v[:, h // R]
    cache_d = cache.to(DEV)
    assert kernels.prompt_query_dtype(cache_d, T, max(new), H, G, D, D) == torch.bfloat16
    results = []
    for rows in (q, q.float()):
        out = torch.empty(T, H * D, dtype=torch.bfloat16, device=DEV)
        kernels.paged_softmax_attn(rows.to(DEV), cache_d, i32([t + [0] * (max(pages) - len(t)) for t in tables]), i32(cu), i32(past),
                                   i32([b for b, n in enumerate(new) for _ in range(n)]), max(new), H, G, D, D, block, out,
                                   window=window, keep_first=keep)
        results.append(out)
    assert torch.equal(*results)
    # probabilities rounded to 8 bits of mantissa (their sum is not), one rounding of the result
    got = results[0].double().cpu().view(T, H, D)
    assert torch.isfinite(got).all()
    assert ((got - want).abs().amax(-1) <= 2.0 ** -8 * want.abs().amax(-1) + 2.0 ** -9 * 4.0).all()
    assert (got - want).norm() <= 2.0 ** -8 * want.norm()


def test_queries_in_16_bits_are_refused_elsewhere():
    from byox_vllm_amd import kernels
    cache = torch.zeros(256, 2 * 64, dtype=torch.bfloat16, device=DEV)
    args = (cache, i32([[0]]), i32([0, 3]), i32([0]), i32([0, 0, 0]))
    for max_q, options in ((1, {}), (3, dict(softcap=20.0)), (3, dict(distance_term=True))):
        assert max_q > 1 or kernels.prompt_query_dtype(cache, 3, max_q, 1, 1, 64, 64) == torch.float32
        with pytest.raises(RuntimeError, match="does not take queries"):
            kernels.paged_softmax_attn(torch.zeros(3, 64, dtype=torch.bfloat16, device=DEV), *args, max_q, 1, 1, 64, 64, 256,
                                       torch.empty(3, 64, dtype=torch.bfloat16, device=DEV), **options)


@pytest.mark.parametrize("block", [16, 32, 48, 64, 80, 128])
@pytest.mark.parametrize("D,R", [(64, 1), (64, 4), (128, 2)])
@pytest.mark.parametrize("window,keep,chunk", [(64, 0, 0), (100, 1, 0), (65, 63, 0), (90, 64, 0), (70, 130, 0), (33, 16, 0), (0, 0, 100)])
def test_entries_of_the_table_that_nobody_sees_are_not_read(D, R, window, keep, chunk, block):
    """Blocks without a kept key and without one from the first new token's window on may have been given away: their entries are -1, and
    the page ahead of the cache, which such an entry stands for, holds NaNs that a read would carry into the results."""
    from byox_vllm_amd import kernels
    torch.manual_seed(window + keep + chunk + D)
    new, past, G = [130, 1, 70, 200], [0, 511, 301, 64 * 5 + 33], 2
    H, pages, T = R * G, [-(-(a + b) // block) for a, b in zip(new, past)], sum(new)
    held = torch.full(((sum(pages) + 1) * block, 2 * G * D), float("nan"), dtype=torch.bfloat16)
    cache = held[block:]
    cache[:] = torch.randn(cache.shape)
    order, tables, left = torch.randperm(sum(pages)).tolist(), [], []
    for n, before in zip(pages, past):
        tables.append([order.pop() for _ in range(n)])
        first = max(before - window + 1 if window else 0, before // chunk * chunk if chunk else 0, 0)
        left.append([page if (i + 1) * block > first or i * block < keep else -1 for i, page in enumerate(tables[-1])])
    assert any(-1 in t for t in left)
    cu = [0]
    for n in new:
        cu.append(cu[-1] + n)
    q = (torch.randn(T, H * D) * 2.0 * D ** -0.5).to(DEV)
    rows = held.to(DEV)[block:]
    results = []
    for shown in (tables, left):
        out = torch.empty(T, H * D, dtype=torch.bfloat16, device=DEV)
        kernels.paged_softmax_attn(q, rows, i32([t + [-1] * (max(pages) - len(t)) for t in shown]), i32(cu), i32(past),
                                   i32([b for b, n in enumerate(new) for _ in range(n)]), max(new), H, G, D, D, block, out,
                                   window=window, keep_first=keep, chunk=chunk)
        results.append(out)
    assert torch.isfinite(results[0]).all()
    assert torch.equal(*results)
