"""GPU parity of hv_softmax_rows at the edges of its row split (sixteen lanes
per row, runs of four entries, 64 entries per step, the 255/256-entry
reciprocals, rows under four entries) and at the ends of int32, with rows at
every offset modulo four, against the CPU oracle, bit for bit."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EDGES = (1, 2, 3, 4, 5, 7, 8, 15, 16, 17, 60, 61, 63, 64, 65, 66, 67, 68, 127, 128, 129, 131, 191,
         192, 193, 197, 252, 253, 254, 255, 256)


@pytest.mark.parametrize("spread", (1, 1 << 10, 1 << 16, 1 << 20, 1 << 31))
def test_rows_of_every_edge_length(oracle, spread):
    from heatvit_amd import ops
    rng = np.random.default_rng(spread % 1013)
    rows = []
    for i in range(4):
        for n in rng.permutation(EDGES):
            r = rng.integers(-spread, spread, n)
            if i == 1:
                r[:] = r[0]  # a flat row: the largest sums
            if i == 2 and n > 1:
                r[rng.integers(n)] = spread - 1  # the maximum at any place
                r[rng.integers(n)] = -spread
            rows.append(r.tolist())
    att, sel = ops.softmax_rows(rows)
    for i, r in enumerate(rows):
        assert np.array_equal(att[i], oracle.softmax_attention(r)), (i, len(r))
        assert np.array_equal(sel[i], oracle.softmax_selector(r)), (i, len(r))


def test_one_output_and_nothing_outside_the_rows(oracle):
    """Either output alone; bytes around the rows keep their values, also
    with outputs at odd addresses."""
    import torch

    from heatvit_amd import _lib
    rng = np.random.default_rng(3)
    lens = [197, 5, 66, 3, 255, 1, 64]
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    total = int(off[-1])
    x = rng.integers(-(1 << 18), 1 << 18, total).astype(np.int32)
    xd, od = torch.from_numpy(x).cuda(), torch.from_numpy(off).cuda()
    stream = torch.cuda.current_stream().cuda_stream
    for shift in (0, 1, 3):
        att = torch.full((total + 16,), 77, dtype=torch.uint8, device="cuda")
        sel = torch.full((total + 16,), -77, dtype=torch.int32, device="cuda")
        _lib.check(_lib.lib().hv_softmax_rows(xd.data_ptr(), od.data_ptr(), len(lens),
                                              att.data_ptr() + 4 + shift, None, stream), "att")
        _lib.check(_lib.lib().hv_softmax_rows(xd.data_ptr(), od.data_ptr(), len(lens), None,
                                              sel.data_ptr() + 4 * shift, stream), "sel")
        a, s = att.cpu().numpy(), sel.cpu().numpy()
        for i in range(len(lens)):
            r = x[off[i]:off[i + 1]].tolist()
            lo, hi = off[i], off[i + 1]
            assert np.array_equal(a[4 + shift + lo:4 + shift + hi], oracle.softmax_attention(r)), i
            assert np.array_equal(s[shift + lo:shift + hi], oracle.softmax_selector(r)), i
        assert (a[:4 + shift] == 77).all() and (a[4 + shift + total:] == 77).all()
        assert (s[:shift] == -77).all() and (s[shift + total:] == -77).all()
