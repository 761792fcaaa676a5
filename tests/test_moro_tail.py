"""The FP64 kernels' inverse-normal tail table (compfinance_amd/csrc/
moro_tail_f64.inc) and the shared-memory layout that holds its upper rows.
CPU only.

The table's values are compared with Moro's tail in extended precision.  The
bound is the rounding of the last multiply-add (1 half-ulp) plus that of the
product before it and of the leading coefficient, each at most 1 half-ulp of a
smaller number: 3 half-ulps of the result."""
import json
import os
import subprocess
import sys

import numpy as np

import pyoracle as po

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "compfinance_amd", "csrc")
sys.path.insert(0, CSRC)
import gen_moro_tail_f64 as gen  # noqa: E402

BIAS = (1023 - 33) << 2


def _committed():
    rows = []
    for line in open(os.path.join(CSRC, "moro_tail_f64.inc")):
        if not line.strip().startswith("//"):
            rows.append([float(x) for x in line.split("//")[0].split(",") if x.strip()])
    return np.array(rows)


def _eval(rows, v):
    """The kernel's steps: row from the upper 14 bits, exact distance to the
    midpoint, Horner with one rounding per step."""
    u = v.view(np.int64)
    r = (u >> 50) - BIAS
    mid = ((u >> 50 << 50) | (1 << 49)).view(np.float64)
    d = (v - mid).astype(np.longdouble)
    p = rows[r, 11]
    for k in range(10, -1, -1):
        p = (rows[r, k].astype(np.longdouble) + p.astype(np.longdouble) * d).astype(np.float64)
    return p, r


def test_committed_table_is_the_generated_one():
    np.testing.assert_array_equal(_committed(), gen.table())


def test_table_is_the_tail():
    rows = _committed()
    rng = np.random.default_rng(20261206)
    # row edges from both sides, the Sobol words' masses, the smallest masses of
    # both generators (1 - p of the largest uniform is a little under 2^-32)
    edges = np.array([(1.0 + q / 4.0) * 2.0 ** e for e in range(-33, -3) for q in range(4)])
    words = np.concatenate([np.arange(1, 50_000), rng.integers(1, int(0.08 * 2 ** 32), 300_000)])
    v = np.concatenate([edges, np.nextafter(edges, 0.0)[1:], words * 2.3283064365387E-10,
                        [1.0 - 2.3283064365387E-10 * 4294967295.0, 1.0 - 4294967087.0 / 4294967088.0]])
    v = v[v < 0.08]
    z, row = _eval(rows, v)
    assert row.min() >= 0 and row.max() <= 119
    t = gen.tail(v)
    err = np.abs((z.astype(np.longdouble) - t) / t) / np.longdouble(2.0 ** -53)
    assert err.max() < 3.0, float(err.max())
    np.testing.assert_allclose(z, -po.inv_normal(v), rtol=1e-14)


SRC = r"""
#include <cstdio>
#include "../../compfinance_amd/csrc/cf_internal.h"
using namespace cfk;
int main()
{
    long bad = 0, n_checked = 0;
    for (int n : {1, 2, 3, 4, 5, 59, 60, 156, 157, 261})
        for (int m : {1, 2, 30, 60, 255})
            for (int w : {1, 4, 16}) {
                const SmemLayout L = smem_layout(n, m, n + 1, 2, w, 8, true, false, true, false, 2 * m + 3, 2, true);
                const size_t off[] = {L.lo, L.mtab, L.hi, L.hi_tail, L.step_sample, L.invn, L.knots, L.bucket, L.iv,
                                      L.acc, L.tails, L.ivbar, L.total};
                for (size_t o : off) bad += o % 16 != 0;
                // the last 16-byte word of LO: dimension group (n - 1) / 4, entry 15
                bad += (size_t(n - 1) / 4 * 16 + 16) * 16 > L.mtab - L.lo;
                bad += kMoroLdsBytes > L.hi - L.mtab;
                bad += size_t(w) * sobol_hi_stride(n) * 4 > L.hi_tail - L.hi;
                bad += size_t(n) * lv_cols(m) * 8 > L.drift - L.iv;
                bad += size_t(w) * tail_row(false) * 8 > L.ivbar - L.tails;
                bad += (size_t(ivbar_copy_stride(n, m)) + size_t(n) * lv_cols(m)) * 8 > L.total - L.ivbar;
                ++n_checked;
            }
    std::printf("{\"bad\": %ld, \"checked\": %ld, \"c3\": %zu}\n", bad, n_checked,
                smem_layout(156, 30, 157, 2, 16, 8, true, false, true, false, 107, 2, true).total);
    return 0;
}
"""


def test_split_layout_holds_its_regions(tmp_path):
    src = os.path.join(ROOT, "tests", "cpp")
    exe = str(tmp_path / "split_layout")
    subprocess.run(["g++", "-std=c++17", "-O1", "-x", "c++", "-", "-I", src, "-o", exe],
                   input=SRC.replace("../../", ROOT + "/"), text=True, check=True)
    out = json.loads(subprocess.run([exe], capture_output=True, text=True, check=True).stdout)
    assert out["bad"] == 0 and out["checked"] == 150, out
    assert out["c3"] <= 160 * 1024      # two adjoint grids beside the 30 x 36 grid's tables
