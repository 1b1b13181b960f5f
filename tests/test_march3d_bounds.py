"""CPU bounds model of the 3D velocity march in csrc/pda_box_kernels.hip
(vel_cc3_body): the box's x lines, each with one more cell at either end, laid
end to end over the planes, 64 consecutive cells to a wavefront of which it
owns 62, marched in y over strips.  For interior boxes and periodic axes, every
state read is a cell inside the grid and every box cell is stored once."""
import itertools

import numpy as np
import pytest

OWN = 62


def wrap(c, n, periodic):
    return np.where(c < 0, c + n, np.where(c >= n, c - n, c)) if periodic else c


def march(n, lo, hi, per, W, rps, own_of=OWN):
    """(reads outside the grid, flat ids of the cells stored)."""
    bw, line = hi[0] - lo[0], hi[0] - lo[0] + 2
    ncell = line * (hi[2] - lo[2])
    nwave = -(-(ncell - 2) // OWN)
    lane = np.arange(64)[None, :]
    s0 = np.arange(nwave)[:, None] * OWN + lane
    s = np.minimum(s0, ncell - 1)
    kz, e = lo[2] + s // line, s % line
    xe = lo[0] + e - 1
    own = (lane >= 1) & (lane <= own_of) & (s0 < ncell) & (e >= 1) & (e <= bw)
    i = wrap(xe, n[0], per[0])
    ic = np.where(i < n[0], i, n[0] - 1)
    bad, stores = 0, []

    def read(x, y, z):
        nonlocal bad
        ok = (x >= 0) & (x < n[0]) & (y >= 0) & (y < n[1]) & (z >= 0) & (z < n[2])
        bad += int(np.count_nonzero(~ok))

    for j0 in range(lo[1], hi[1], rps):
        j1 = min(j0 + rps, hi[1])
        for r in range(j0 - W, j1 - 1 + W + 1):  # the rows that enter the window
            read(ic, np.asarray(wrap(np.asarray(r), n[1], per[1])), kz)
        for r in range(j0, j1):
            for p in range(-(W - 1), W):
                read(ic + (wrap(xe + p, n[0], per[0]) - ic), np.asarray(r), kz)
            for p in range(-W, W + 1):
                read(ic, np.asarray(r), wrap(kz + p, n[2], per[2]))
            stores.append(((kz * n[1] + r) * n[0] + i)[own])
    return bad, np.concatenate(stores)


def boxes():
    for W, per in itertools.product((1, 2, 3), itertools.product((False, True), repeat=3)):
        for nx, ny, nz in ((2 * W + 1, 2 * W + 2, 2 * W + 1), (60, 8, 7), (61, 7, 8), (62, 7, 7), (66, 7, 9), (130, 8, 7)):
            n = (nx, ny, nz)
            lo = tuple(0 if p else W for p in per)
            hi = tuple(m if p else m - W for m, p in zip(n, per))
            yield n, lo, hi, per, W


@pytest.mark.parametrize("rps", [1, 3, 64])
def test_reads_inside_and_cells_stored_once(rps):
    for n, lo, hi, per, W in boxes():
        bad, stores = march(n, lo, hi, per, W, rps)
        want = [(k * n[1] + j) * n[0] + i for k in range(lo[2], hi[2]) for j in range(lo[1], hi[1])
                for i in range(lo[0], hi[0])]
        assert bad == 0, (n, per, W)
        assert np.array_equal(np.sort(stores), np.array(want)), (n, per, W)


def test_model_flags_planted_mistakes():
    n, lo, hi = (66, 11, 9), (3, 3, 3), (63, 8, 6)
    _, stores = march(n, lo, hi, (False,) * 3, 3, 2, own_of=63)  # a lane that its neighbour owns too
    assert len(stores) != len(np.unique(stores))
    assert march(n, (2, 3, 3), hi, (False,) * 3, 3, 2)[0] > 0     # a box whose stencils leave the grid
