"""The index lines of the 3D velocity march (vel_cc3_body and the launch's count of
wavefronts) are those that the bounds model in test_march3d_bounds.py restates:
a change to one of them must come with a change of the model."""
import os
import re

import pytest

import test_march3d_bounds as model

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "pressio-demoapps_amd", "csrc", "pda_box_kernels.hip")

# (line of the kernel, what the model restates by it)
BODY = [
    ("const int bw = int(B.hi[0] - B.lo[0]), line = bw + 2;", "line"),
    ("const int64_t ncell = int64_t(line) * (B.hi[2] - B.lo[2]);", "ncell"),
    ("const int64_t nwave = (ncell - 2 + V3OWN - 1) / V3OWN;", "nwave"),
    ("const int64_t strip = bid / nwave, wave = bid - strip * nwave;", "the grid"),
    ("const int j0 = int(B.lo[1] + strip * rows_per_strip);", "j0"),
    ("const int j1 = j0 + rows_per_strip < int(B.hi[1]) ? j0 + rows_per_strip : int(B.hi[1]);", "j1"),
    ("const int64_t s0 = wave * V3OWN + lane, s = s0 < ncell ? s0 : ncell - 1;", "s0, s"),
    ("const int plane = int(s / line), e = int(s - int64_t(plane) * line);", "kz, e"),
    ("const int kz = int(B.lo[2]) + plane, xe = int(B.lo[0]) + e - 1;", "kz, xe"),
    ("const int64_t i = wrap_axis<0>(B, xe);", "i"),
    ("const int64_t ic = i < nx ? i : nx - 1;", "ic"),
    ("const bool own = lane >= 1 && lane <= V3OWN && s0 < ncell && e >= 1 && e <= bw;", "own"),
    ("for (int p = 0; p < NR; ++p) dx[p] = wrap_axis<0>(B, xe + p - (W - 1)) - int(ic);", "x reads"),
    ("for (int p = 0; p <= 2 * W; ++p) dz[p] = (wrap_axis<2>(B, kz + p - W) - kz) * int(nx) * ny;", "z reads"),
    ("const double *col = U + (int64_t(kz) * nx * ny + ic) * M;", "the column"),
    ("if (r + 1 < j1) load(col + wrap_axis<1>(B, r + 1 + W) * row, nxt);", "the last rows of the window"),
    ("for (int p = 0; p < NR; ++p) load(col + wrap_axis<1>(B, j0 - W + p) * row, win[p]);", "its first rows"),
    ("for (int r = j0 - 2; r < j1; ++r) {", "rows"),
    ("const double *at = col + r * row;", "the row's cell"),
    ("if (p != W - 1) load(at + int64_t(dx[p]) * M, xs[p]);", "x reads"),
    ("if (p != W) load(at + int64_t(dz[p]) * M, zs[p]);", "z reads"),
    ("const int64_t c = (int64_t(kz) * ny + r) * nx + i;", "stores"),
]
LAUNCH = [
    "if (dim == 3) return ((bw + 2) * (B.hi[2] - B.lo[2]) - 2 + V3OWN - 1) / V3OWN;",
    "return velocity_waves(B, dim, w) * ((bh + rows_per_strip - 1) / rows_per_strip);",
]
WRAP = ["if (B.mode[A] != 1) return c;", "return c < 0 ? c + n : (c >= n ? c - n : c);"]


def _source():
    txt = open(SRC).read()
    start = txt.index("vel_cc3_body(")
    return txt, txt[start:txt.index("\n}\n", start)]


def _lacking(txt, body):
    lacking = [line for line, _ in BODY if line not in body]
    lacking += [line for line in LAUNCH + WRAP if line not in txt]
    seg = int(re.search(r"constexpr int VSEG = (\d+);", txt).group(1))
    own = re.search(r"constexpr int V3OWN = VSEG - (\d+);", txt)
    if own is None or seg - int(own.group(1)) != model.OWN:
        lacking.append("V3OWN")
    return lacking


def test_model_restates_the_kernel():
    assert _lacking(*_source()) == []


@pytest.mark.parametrize("line", [b for b, _ in BODY])
def test_a_changed_line_is_seen(line):
    txt, body = _source()
    other = line.replace("+ 1", "+ 2").replace("- 1", "- 2").replace("<", "<=").replace(" W", " (W)").replace("=", "= 0 +")
    assert _lacking(txt.replace(line, other), body.replace(line, other)) == [line]


def test_a_changed_width_is_seen():
    txt, body = _source()
    assert _lacking(txt.replace("V3OWN = VSEG - 1;", "V3OWN = VSEG;"), body) == ["V3OWN"]
