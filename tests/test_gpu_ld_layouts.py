"""The row-parallel LD solves (k_tri_chain_rp, k_tri_chain_rpf) in the layouts
that the plan picks at the ends of its range: one wave and 9-16 waves, 1-64 lanes per
row, levels cut into pieces, a single chain with levels of more than 1,024
rows, odd sizes.  Every LD solve equals the oracle's bit for bit (whole
numbers: no tolerance)."""
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

def _check(a, smoother, monkeypatch, capfd, prec=S.INT):
    """LD solves of every level against the oracle; the layouts picked: (rows,
    waves, entries, lanes, pieces, far entries, single vectors entry-parallel)."""
    monkeypatch.setenv("SC23AD_VERBOSE", "1")
    a.lmax1_scaling(np.zeros(a.n))
    h = S.Hierarchy(a, prec, S.amg_param(smoother))
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
    plans = _check(a, S.SOR, monkeypatch, capfd)
    assert not plans[0][6] and any(p[6] for p in plans)
    assert all(p[1] > 0 for p in plans)
    h = S.Hierarchy(a, S.INT, S.amg_param(S.SOR))
    path = export(h)
    amg, oh = S.Amg(h), O.OracleHier(path)
    os.unlink(path)
    assert S.block_native(amg)
    v = np.random.default_rng(3).integers(-2**29, 2**29, (2, a.n)).astype(np.int32)
    out = S.precondition_block(amg, v)
    for k in range(2):
        assert np.array_equal(out[k], oh.vcycle(v[k]))
        assert np.array_equal(out[k], amg.precondition(v[k]))


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


@pytest.mark.parametrize("lanes", [1, 2, 4, 8, 16, 32, 64])
@pytest.mark.parametrize("waves", [1, 3])
def test_forced_layouts(lanes, waves, monkeypatch, capfd):
    monkeypatch.setenv("SC23AD_RP_LANES", str(lanes))
    monkeypatch.setenv("SC23AD_RP_WAVES", str(waves))
    plans = _check(S.CsrMat.generate(S.GEN_DIFFUSION27, 17, 5, 1.0, 1.0, 1e-3, 3), S.SOR,
                   monkeypatch, capfd)
    assert any(p[1] == waves and p[3] == lanes for p in plans) or lanes == 1


def test_sixteen_waves(monkeypatch, capfd):
    monkeypatch.setenv("SC23AD_RP_WAVES", "16")
    plans = _check(S.CsrMat.generate(S.GEN_POISSON2D, 67), S.SOR, monkeypatch, capfd)
    assert any(p[1] == 16 for p in plans)


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
    _check(S.CsrMat.generate(S.GEN_DIFFUSION27, 29, 5, 1.0, 1.0, 1e-3, 3), smoother, monkeypatch,
           capfd, prec)
