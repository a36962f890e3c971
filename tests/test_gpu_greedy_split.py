"""The full-rank greedy search with its cross terms from split operands
(csrc/ldlq.hip, greedy_plane_bytes): rows are searched independently, so the same
rows searched in pieces too short for that path give the general path's codes
for the same problem.

Bar: an fp32 search leaves the 64-bit one only where the cross terms' rounding
decides a code; the rest of that row then follows.  A cross term of K = cols
products carries a relative error of about 2^-24 sqrt(K) / 4 of its size, a few
grid steps, so each of the 2 x cols decisions goes the other way with a
probability of order 2e-6 sqrt(K / 4096) and a row with one of order 1 %: at
most that share of the rows may differ, in either path.  (Measured over 24
problems of these sizes: 50 rows of the split path, 69 of the general one, of
69000.)  A wrong element of a cross term would change nearly every row."""

from __future__ import annotations

import pytest
import torch

from tests.conftest import lognormal_hessian

pytestmark = pytest.mark.gpu

PIECE = 1100   # rows: below the split path's line
ROWS_COLS = [(2050, 2048), (2175, 2560), (2048, 4096)]   # its smallest, ragged rows, several K-blocks


def _problem(rows, cols, dev, seed):
    g = torch.Generator().manual_seed(seed)
    H = lognormal_hessian(cols, cols + 512, seed).to(dev)
    H = H + 0.01 * H.diagonal().mean() * torch.eye(cols, device=dev)
    W = torch.randn(rows, cols, generator=g).to(dev)
    s = W.abs().amax(1) / 7
    return W, (W / s[:, None]).round().clamp(-8, 7).to(torch.int8), s, H


def _search64(W, Q, s, H, passes):
    W, q, s, H = W.double(), Q.double(), s.double(), H.double()
    err = q * s[:, None] - W
    d = H.diagonal().tolist()
    for _ in range(passes):
        for j in range(W.shape[1]):
            cross = err @ H[j] - err[:, j] * d[j]
            new = ((W[:, j] - cross / d[j]) / s).round().clamp(-8, 7)
            q[:, j] = new
            err[:, j] = new * s - W[:, j]
    return q.to(torch.int8)


@pytest.mark.parametrize("rows,cols", ROWS_COLS)
def test_greedy_split_misses_no_more_than_general(gpu_dev, rows, cols):
    from int_crush_converter_amd.greedy import greedy_local_search
    W, Q, s, H = _problem(rows, cols, gpu_dev, rows + cols)
    want = _search64(W, Q, s, H, 2)
    got = greedy_local_search(W, Q, s, H, 2, -8, 7)
    gen = torch.cat([greedy_local_search(W[a:a + PIECE], Q[a:a + PIECE], s[a:a + PIECE], H, 2, -8, 7)
                     for a in range(0, rows, PIECE)])
    for name, x in (("split", got), ("general", gen)):
        differ = (x != want).any(1).sum().item()
        assert differ <= 0.01 * rows, (name, differ)


def test_greedy_split_infinite_rows(gpu_dev):
    # an infinite weight: its row gets the general path's codes, the others stay what they were
    from int_crush_converter_amd.greedy import greedy_local_search
    rows, cols = ROWS_COLS[0]
    W, Q, s, H = _problem(rows, cols, gpu_dev, 5)
    clean = greedy_local_search(W, Q, s, H, 1, -8, 7)
    W[3, 700], W[rows - 1, cols - 1], W[40, 0] = float("inf"), float("-inf"), float("nan")
    got = greedy_local_search(W, Q, s, H, 1, -8, 7)
    gen = torch.cat([greedy_local_search(W[a:a + PIECE], Q[a:a + PIECE], s[a:a + PIECE], H, 1, -8, 7)
                     for a in range(0, rows, PIECE)])
    for r in (3, 40, rows - 1):
        assert torch.equal(got[r], gen[r]), r
    assert torch.equal(got[64:rows - 64], clean[64:rows - 64])


def test_greedy_split_infinity_in_every_row(gpu_dev):
    # every cross term is formed again: the general path's codes, and in the time of a second product (1.7 times the
    # search without infinities), not of one thread summing each element (8.2 times)
    from int_crush_converter_amd.greedy import greedy_local_search
    rows, cols = ROWS_COLS[0]
    W, Q, s, H = _problem(rows, cols, gpu_dev, 6)

    def timed():
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        q = greedy_local_search(W, Q, s, H, 1, -8, 7)
        b.record()
        b.synchronize()
        return q, a.elapsed_time(b)

    timed()
    clean = timed()[1]
    W[torch.arange(rows), torch.randint(0, cols, (rows,), generator=torch.Generator().manual_seed(1))] = float("inf")
    got, t = timed()
    gen = torch.cat([greedy_local_search(W[a:a + PIECE], Q[a:a + PIECE], s[a:a + PIECE], H, 1, -8, 7)
                     for a in range(0, rows, PIECE)])
    assert torch.equal(got, gen)
    assert t < 4 * clean, (t, clean)
