"""The guess network's tiles on grids that are narrow or low.  Values: a field of
few columns (or rows) is periodic, so the network's output on it repeated to a
wide grid is its output on the narrow one, bit for bit (every pixel is the same
chain of products), and the gradients are the same but for the order of the
FP32 sums (at most 2^17 terms in blocks of 512 and more, relative 1e-4 of the
gradient's norm).  Cost: half a million pixels as 4 or 8 columns, or 4 rows, cost
no more than 1.4 times the same pixels as 1024 x 512 (1.2 to 2.8 times with 32
columns and 16 rows to every tile)."""
import time

import numpy as np
import pytest

import guessnet_oracle as G
import pressiodemoapps_amd as pda

pytestmark = pytest.mark.gpu
COSTS = np.array([9.0, 4.0, 1.0, 0.0, 2.5, 3.0, 7.0])


@pytest.fixture(scope="module")
def torch():
    import torch as _t
    if not _t.cuda.is_available():
        pytest.skip("no HIP device")
    return _t


def _net(nx, ny, w, scales):
    net = pda.GuessNet(nx, ny)
    net.set_scales(scales[0], scales[1], scales[2], scales[3])
    net.set_params(w)
    return net


# (columns, rows, repeats in x, repeats in y): 8-column tiles with one and four
# rows per wave, a tile wider than the grid, partial tiles, grids lower than a
# tile; the last one's repetition has more bands of columns than the backward
# pass has workgroups
@pytest.mark.parametrize("nx,ny,rx,ry", [(4, 128, 8, 1), (4, 32768, 8, 1), (5, 512, 32, 1), (8, 64, 4, 1),
                                         (8, 16384, 8, 1), (12, 128, 8, 1), (40, 512, 4, 1), (512, 4, 1, 8),
                                         (16384, 4, 1, 8), (4096, 12, 1, 4), (32768, 4, 2, 1)])
def test_narrow_grid_equals_its_periodic_repetition(nx, ny, rx, ry, torch):
    print(f"[gpu-nn-tiles] {nx} x {ny}", flush=True)
    rng = np.random.default_rng(nx + ny)
    w = (rng.standard_normal(pda.GuessNet(32, 16).nparams) * 0.1).astype(np.float32)
    f0 = rng.standard_normal(2 * nx * ny)
    f = [f0 + 0.08 * k * rng.standard_normal(f0.shape) for k in range(5)]
    scales = (5e-3, tuple(float(np.std(5e-3 * d)) for d in G.diffs(f)), 5.5e-3, 4.5e-3)

    def run(mx, my, fields):
        net = _net(mx, my, w, scales)
        t = [torch.from_numpy(x).cuda() for x in fields]
        loss, g, o = net.gradients(t, 4e-3, COSTS)
        return loss, g.astype(np.float64), o.reshape(my, mx, -1), net.policy()[0]

    loss, g, o, order = run(nx, ny, f)
    rep = [np.tile(x.reshape(ny, nx, 2), (ry, rx, 1)).ravel() for x in f]
    wloss, wg, wo, worder = run(nx * rx, ny * ry, rep)
    assert np.array_equal(wo, np.tile(o, (ry, rx, 1)))
    err = float(np.linalg.norm(g - wg) / np.linalg.norm(wg))
    print(f"[gpu-nn-tiles] gradients {err:.1e}, loss {loss:.6g} {wloss:.6g}, order {order:.6g} {worder:.6g}", flush=True)
    assert err <= 1e-4 and abs(loss - wloss) <= 1e-4 * wloss and abs(order - worder) <= 1e-4


def test_cost_of_narrow_and_low_grids(torch):
    def cost(nx, ny):
        net = pda.GuessNet(nx, ny)
        net.set_params((np.random.default_rng(0).standard_normal(net.nparams) * 0.05).astype(np.float32))
        u = torch.rand(2 * nx * ny, dtype=torch.float64, device="cuda")
        f = [torch.rand_like(u) for _ in range(5)]
        out = torch.empty_like(u)
        best = float("inf")
        for _ in range(6):
            torch.cuda.synchronize()
            t = time.perf_counter()
            for _ in range(10):
                net.predict(u, u, f, 5e-3, out=out)
            torch.cuda.synchronize()
            best = min(best, (time.perf_counter() - t) / 10 * 1e6)
        return best

    wide = cost(1024, 512)
    for nx, ny in ((4, 131072), (8, 65536), (131072, 4)):
        us = cost(nx, ny)
        print(f"[gpu-nn-tiles] {nx} x {ny}: {us:.0f} us, 1024 x 512: {wide:.0f} us", flush=True)
        assert us <= 1.4 * wide


def test_memory_of_a_wide_grid(torch):
    """The backward pass's partial sums are bounded: a grid of 131072 columns takes
    what the same pixels take as 1024 columns, to 32 MB of 430 (177 MB of partial
    sums with a workgroup for every band of 64 columns, 44 with 512 at most)."""
    def taken(nx, ny):
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        net = pda.GuessNet(nx, ny)
        return before - torch.cuda.mem_get_info()[0], net

    a, keep = taken(1024, 512)
    b, other = taken(131072, 4)
    print(f"[gpu-nn-tiles] 1024 x 512: {a / 1e6:.0f} MB, 131072 x 4: {b / 1e6:.0f} MB", flush=True)
    assert a > 300e6 and b <= a + 32e6
