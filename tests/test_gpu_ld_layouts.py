"""The row-parallel LD solves (k_tri_chain_rp, k_tri_chain_rpf) in the layouts
at the ends of the plan's range: one wave and 9-16 waves, 1-64 lanes per row,
far dependencies over one and several lanes, levels cut into pieces, a single
chain with levels of more than 1,024 rows, odd sizes; integer layouts on single
vectors and on blocks.  Every LD solve equals the oracle's bit for bit (whole
numbers, or FP sums in stored order: no tolerance)."""
from __future__ import annotations

import os
import re

import numpy as np
import pytest

import oracle as O
import sc23ad as S
from helpers import export

pytestmark = pytest.mark.gpu


LAYOUT = re.compile(r"\[sc23ad plan\] kind 0 n (\d+) .*rp waves (\d+) entries (\d+) rows \d+ "
                    r"lanes (\d+) .*rp: pieces (\d+) far (\d+) fence \d+(.*)")


def _check(a, smoother, monkeypatch, capfd, prec=S.INT, block=0):
    """LD solves of every level against the oracle; the layouts picked: (rows,
    waves, entries, lanes, pieces, far entries, single vectors entry-parallel).
    block: V-cycles of so many vectors in one call too (integers)."""
    a.lmax1_scaling(np.zeros(a.n))
    return _check_hierarchy(S.Hierarchy(a, prec, S.amg_param(smoother)), monkeypatch, capfd, prec,
                            block)


def _check_hierarchy(h, monkeypatch, capfd, prec, block):
    monkeypatch.setenv("SC23AD_VERBOSE", "1")
    capfd.readouterr()
    amg = S.Amg(h)
    plans = [(*map(int, m.groups()[:-1]), "entry-parallel" in m.group(7))
             for m in LAYOUT.finditer(capfd.readouterr().err)]
    print("[ld layouts] (n, waves, entries, lanes, pieces, far, ep):", plans, flush=True)
    path = export(h)
    try:
        oh = O.OracleHier(path)
    finally:
        os.unlink(path)
    rng = np.random.default_rng(7)
    for lv in range(amg.depth):
        n = oh.level_n(lv)
        if prec == S.INT:
            x = rng.integers(-2**29, 2**29, n).astype(np.int32)
        else:  # signed zeros and subnormals among them: compared bit for bit
            x = rng.standard_normal(n).astype(np.float64 if prec == S.FP64 else np.float32)
            x[::7] = -0.0
            x[3::11] = 1e-310 if prec == S.FP64 else 1e-40
        y, yo = amg.level_op(lv, S.OP_TRSV_LD, x, n), oh.level_op(lv, S.OP_TRSV_LD, x, n)
        assert y.tobytes() == yo.tobytes(), lv
    if block:
        v = rng.integers(-2**29, 2**29, (block, oh.level_n(0))).astype(np.int32)
        out = S.precondition_block(amg, v)
        for k in range(block):
            assert np.array_equal(out[k], oh.vcycle(v[k])), k
    return plans


@pytest.mark.parametrize("kind,params,smoother,waves,lanes", [
    (S.GEN_POISSON2D, (3,), S.SOR, 1, 1),
    (S.GEN_LAPLACE3D, (61,), S.SOR, 9, 32),
    (S.GEN_DIFFUSION27, (33, 5, 1.0, 1.0, 1e-3, 3), S.BLOCK_SOR, 1, 8),
], ids=["poisson2d_3", "laplace3d_61_sor", "diffusion27_33_block"])
def test_layouts_of_the_plan(kind, params, smoother, waves, lanes, monkeypatch, capfd):
    plans = _check(S.CsrMat.generate(kind, *params), smoother, monkeypatch, capfd)
    assert max(p[1] for p in plans) >= waves and max(p[3] for p in plans) >= lanes


def test_entry_parallel_where_few_rows_are_long(monkeypatch, capfd):
    """27-point SOR levels whose longest row is many times their mean: single
    vectors take the entry-parallel kernel, blocks the row-parallel one."""
    a = S.CsrMat.generate(S.GEN_DIFFUSION27, 64, 8, 1.0, 1.0, 1e-3, 2)
    plans = _check(a, S.SOR, monkeypatch, capfd, block=2)
    assert not plans[0][6] and any(p[6] for p in plans)
    assert all(p[1] > 0 for p in plans)


def _wide_level_short_reach(n=1000, first=970, reach=25):
    """`first` rows without dependencies, then rows that depend on the last
    `reach` of them: a level many times wider than any dependency reaches."""
    rng = np.random.default_rng(5)
    at = [(k, int(d)) for k in range(first, n)
          for d in rng.choice(np.arange(first - reach, first), 3, replace=False)]
    m = np.zeros((n, n))
    for k, d in at:
        m[k, d] = m[d, k] = -rng.uniform(0.5, 1.0)
    m[np.arange(n), np.arange(n)] = 1.0 - m.sum(1)
    i, j = np.nonzero(m)
    rptr = np.searchsorted(i, np.arange(n + 1)).astype(np.int32)
    return S.CsrMat.from_arrays(n, rptr, j.astype(np.int32), m[i, j])


@pytest.mark.parametrize("prec", [S.INT, S.FP64, S.FP32], ids=["int", "fp64", "fp32"])
@pytest.mark.parametrize("knobs", [{}, {"SC23AD_TRI_RP": "0"}, {"SC23AD_RP_WAVES": "1"},
                                   {"SC23AD_RP_WAVES": "8"}, {"SC23AD_RP_RING_FAR": "1",
                                                              "SC23AD_FP_RING_FAR": "1"}],
                         ids=["plan", "other-kernels", "one-wave", "eight-waves", "least-ring"])
def test_level_wider_than_the_reach(knobs, prec, monkeypatch, capfd):
    """The ring holds at least the rows that are solved between two barriers,
    also where the dependencies need less: rows a ring apart share a slot."""
    for k, v in knobs.items():
        monkeypatch.setenv(k, v)
    a = _wide_level_short_reach()
    a.lmax1_scaling(np.zeros(a.n))
    h = S.Hierarchy(a, prec, S.amg_param(S.SOR, coarse_n=64))
    for _ in range(4):
        _check_hierarchy(h, monkeypatch, capfd, prec, 3 if prec == S.INT else 0)


@pytest.mark.parametrize("prec", [S.INT, S.FP64, S.FP32], ids=["int", "fp64", "fp32"])
def test_jacobi_sor_levels_wider_than_the_reach(prec, monkeypatch, capfd):
    """JacobiSOR blocks of 1,200 rows: two levels, the second of 31 rows that
    depend on the last of the first."""
    a = S.CsrMat.generate(S.GEN_CONVDIFF2D, 94, 24.14150207068065, 5.948711626198889)
    a.lmax1_scaling(np.zeros(a.n))
    h = S.Hierarchy(a, prec, S.amg_param(S.JACOBI_SOR, coarse_n=300))
    for _ in range(4):
        _check_hierarchy(h, monkeypatch, capfd, prec, 0)


@pytest.mark.parametrize("prec", [S.INT, S.FP64, S.FP32], ids=["int", "fp64", "fp32"])
def test_one_long_row_is_not_padded_to(prec, monkeypatch, capfd):
    """A 5-point system of 48,400 rows whose last row has 400 entries more (in
    its BlockSOR block): a layout padded to it would take 200-300 MB for 1-2 MB of
    entries."""
    n = 220 * 220
    rptr, cind, val = S.CsrMat.generate(S.GEN_POISSON2D, 220).arrays()
    rng = np.random.default_rng(17)
    old = cind[rptr[n - 1]:]
    extra = np.setdiff1d(n - 1200 + rng.choice(1199, 400, replace=False), old).astype(np.int32)
    cols = np.concatenate([old, extra])
    vals = np.concatenate([val[rptr[n - 1]:], np.full(len(extra), -2.0**-9)])
    order = np.argsort(cols)
    rptr = rptr.copy()
    rptr[n] += len(extra)
    a = S.CsrMat.from_arrays(n, rptr, np.concatenate([cind[:len(cind) - len(old)], cols[order]]),
                             np.concatenate([val[:len(val) - len(old)], vals[order]]))
    plans = _check(a, S.BLOCK_SOR, monkeypatch, capfd, prec)
    assert plans[0][0] == n and plans[0][1] == 0


@pytest.mark.parametrize("prec", [S.FP64, S.FP32], ids=["fp64", "fp32"])
def test_fp_level_pipelined_where_few_rows_are_long(prec, monkeypatch, capfd):
    """Short rows in levels of about 100 and one row of 150 entries: a thread per
    row beats 32 lanes per row, which would cut every level into ten pieces."""
    n = 120
    rptr, cind, val = S.CsrMat.generate(S.GEN_POISSON2D, n).arrays()
    old = cind[rptr[-2]:]
    extra = np.setdiff1d(np.arange(n * n - 200, n * n - 50), old).astype(np.int32)
    cols = np.concatenate([old, extra])
    order = np.argsort(cols)
    vals = np.concatenate([val[rptr[-2]:], np.full(len(extra), -2.0**-9)])[order]
    rptr = rptr.copy()
    rptr[-1] += len(extra)
    cut = len(cind) - len(old)
    a = S.CsrMat.from_arrays(n * n, rptr, np.concatenate([cind[:cut], cols[order]]),
                             np.concatenate([val[:cut], vals]))
    plans = _check(a, S.SOR, monkeypatch, capfd, prec)
    assert plans[0][0] == n * n and plans[0][1] == 0


@pytest.mark.parametrize("lanes", [1, 2, 4, 8, 16, 32, 64])
@pytest.mark.parametrize("waves", [1, 3])
def test_forced_layouts(lanes, waves, monkeypatch, capfd):
    monkeypatch.setenv("SC23AD_RP_LANES", str(lanes))
    monkeypatch.setenv("SC23AD_RP_WAVES", str(waves))
    a = (S.CsrMat.generate(S.GEN_POISSON2D, 67) if lanes == 1 else
         S.CsrMat.generate(S.GEN_DIFFUSION27, 17, 5, 1.0, 1.0, 1e-3, 3))
    plans = _check(a, S.SOR, monkeypatch, capfd, block=3)
    assert any(p[1] == waves and p[3] == lanes for p in plans)


@pytest.mark.parametrize("waves", [9, 16])
def test_sixteen_waves(waves, monkeypatch, capfd):
    monkeypatch.setenv("SC23AD_RP_WAVES", str(waves))
    plans = _check(S.CsrMat.generate(S.GEN_POISSON2D, 67), S.SOR, monkeypatch, capfd, block=3)
    assert any(p[1] == waves for p in plans)


@pytest.fixture(scope="module")
def far_hierarchy():
    """BlockSOR blocks of 7 1/2 grid lines: the rows of a line's second half
    depend on the line before, up to 299 levels back.  Entries per row 2, 4,
    10, 11, 10 on the five levels, far ones 1, 2, 5, 3, 5."""
    a = S.CsrMat.generate(S.GEN_POISSON2D, 300)
    a.lmax1_scaling(np.zeros(a.n))
    return S.Hierarchy(a, S.INT, S.amg_param(S.BLOCK_SOR))


@pytest.mark.parametrize("lanes,entries,waves", [
    (1, 4, 1), (1, 4, 3), (1, 4, 9), (1, 4, 16), (1, 8, 2), (1, 10, 1), (1, 12, 8),
    (2, 8, 1), (2, 10, 3), (2, 12, 8), (4, 8, 3), (4, 10, 1), (4, 12, 2), (8, 8, 8), (8, 10, 2),
    (8, 12, 1)])
def test_far_layouts(lanes, entries, waves, far_hierarchy, monkeypatch, capfd):
    """Far dependencies over 1-8 lanes, single vectors and blocks (a ring of
    only what the far rule leaves to it; factors whose rows are longer than the
    forced layout take other kernels)."""
    monkeypatch.setenv("SC23AD_RP_RING_FAR", "1")
    monkeypatch.setenv("SC23AD_RP_LANES", str(lanes))
    monkeypatch.setenv("SC23AD_RP_ENTRIES", str(entries))
    monkeypatch.setenv("SC23AD_RP_WAVES", str(waves))
    plans = _check_hierarchy(far_hierarchy, monkeypatch, capfd, S.INT, 5)
    got = [p[5] for p in plans if (p[1], p[2], p[3]) == (waves, entries, lanes)]
    assert 1 in got and 2 in got  # one far entry per row has kernels of its own
    assert lanes * entries < 10 or 5 in got


@pytest.mark.parametrize("prec", [S.FP64, S.FP32], ids=["fp64", "fp32"])
@pytest.mark.parametrize("lanes", [1, 2, 4, 8, 16, 32, 64])
@pytest.mark.parametrize("waves", [1, 3, 8])
def test_forced_fp_layouts(lanes, waves, prec, monkeypatch, capfd):
    """One lane per row on the 2D factor (2-4 entries per row), several on the
    27-point one (up to 13 and more), whose pieces subtract 8 to 64 products."""
    monkeypatch.setenv("SC23AD_RP_LANES", str(lanes))
    monkeypatch.setenv("SC23AD_RP_WAVES", str(waves))
    a = (S.CsrMat.generate(S.GEN_POISSON2D, 67) if lanes == 1 else
         S.CsrMat.generate(S.GEN_DIFFUSION27, 17, 5, 1.0, 1.0, 1e-3, 3))
    plans = _check(a, S.SOR, monkeypatch, capfd, prec)
    assert any(p[1] == waves and p[3] == lanes for p in plans)


@pytest.mark.parametrize("prec", [S.FP64, S.FP32], ids=["fp64", "fp32"])
@pytest.mark.parametrize("smoother", [S.SOR, S.BLOCK_SOR], ids=["sor", "block"])
def test_fp_far_dependencies_small_ring(smoother, prec, monkeypatch, capfd):
    monkeypatch.setenv("SC23AD_FP_RING_FAR", "1")
    # 1.2 planes per BlockSOR block: rows in the second one depend on rows of the
    # first many levels back, as the coarse levels of the SOR hierarchy do
    plans = _check(S.CsrMat.generate(S.GEN_DIFFUSION27, 48 if smoother == S.BLOCK_SOR else 29, 5,
                                     1.0, 1.0, 1e-3, 3), smoother, monkeypatch, capfd, prec)
    assert any(p[5] > 0 for p in plans)


@pytest.mark.parametrize("prec", [S.FP64, S.FP32], ids=["fp64", "fp32"])
@pytest.mark.parametrize("lanes", [1, 2, 4, 8, 16])
def test_fp_far_layouts(lanes, prec, monkeypatch, capfd):
    monkeypatch.setenv("SC23AD_FP_RING_FAR", "1")
    monkeypatch.setenv("SC23AD_RP_LANES", str(lanes))
    plans = _check(S.CsrMat.generate(S.GEN_POISSON2D, 300), S.BLOCK_SOR, monkeypatch, capfd, prec)
    got = {p[5] for p in plans if p[3] == lanes and p[1] > 0}
    assert {1, 2} <= got and (lanes == 1 or 5 in got)
