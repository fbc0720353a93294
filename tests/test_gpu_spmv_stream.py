"""The CSR products streamed through LDS (k_spmv_stream_int, _fp): every row
count per workgroup, rows shorter and longer than a tile of 2,048 entries,
empty rows and workgroups without entries, sizes off the workgroup's.  Whole
numbers, or FP sums in stored order: no tolerance."""
from __future__ import annotations

import os

import numpy as np
import pytest

import oracle as O
import sc23ad as S
from helpers import export

pytestmark = pytest.mark.gpu


def _reference(rptr, cind, val, bit, x):
    with np.errstate(over="ignore"):  # 64-bit sums wrap
        p = np.concatenate([[0], np.cumsum(val.astype(np.int64) * x[cind].astype(np.int64))])
        return ((p[rptr[1:]] - p[rptr[:-1]]) >> bit).astype(np.int32)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 1023, 1024, 1041, 32 * 512 - 1, 32 * 512, 128 * 512, 128 * 512 + 77])
def test_rows_per_workgroup(n):
    """4, 16, 32 and 128 rows per workgroup, by the number of rows."""
    rng = np.random.default_rng(n)
    lens = rng.integers(0, 12, n)
    lens[rng.integers(0, n, 3)] = [2047, 2048, 5001]
    lens[n // 3:n // 3 + 300] = 0
    rptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    m = 3001
    cind = rng.integers(0, m, rptr[-1]).astype(np.int32)
    val = rng.integers(-2**31, 2**31, rptr[-1]).astype(np.int32)
    x = rng.integers(-2**31, 2**31, m).astype(np.int32)
    for bit in (0, 30):
        assert np.array_equal(S.spmv_int(rptr, cind, val, bit, x),
                              _reference(rptr, cind, val, bit, x)), bit


@pytest.mark.parametrize("n", [1, 3, 4, 5, 1023, 1024, 32 * 512, 128 * 512 + 77])
@pytest.mark.parametrize("kind", ["all long", "one", "every 50th", "around the bound"])
def test_long_rows(n, kind):
    """Rows of more than 32 entries per lane, whose workgroups share each tile's
    products: alone, among short and empty rows, across many tiles, and rows of
    exactly the bound and one more (64 to 2,048 entries)."""
    rng = np.random.default_rng(n)
    if kind == "all long":
        lens = np.full(n, max(300, min(40000, 2000000 // n)) + n % 3)
    else:
        lens = rng.integers(0, 5, n)
        if kind == "one":
            lens[n // 2] = 100001
        elif kind == "every 50th":
            lens[::50] = rng.integers(300, 4000, len(lens[::50]))
        else:
            at = rng.permutation(n)[:64]
            lens[at] = np.resize([64, 65, 256, 257, 512, 513, 2048, 2049], len(at))
    rptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    m = 5003
    cind = rng.integers(0, m, rptr[-1]).astype(np.int32)
    val = rng.integers(-2**31, 2**31, rptr[-1]).astype(np.int32)
    x = rng.integers(-2**31, 2**31, m).astype(np.int32)
    for bit in (0, 30):
        assert np.array_equal(S.spmv_int(rptr, cind, val, bit, x),
                              _reference(rptr, cind, val, bit, x)), bit


@pytest.mark.parametrize("prec", [S.INT, S.FP64, S.FP32], ids=["int", "fp64", "fp32"])
def test_fused_modes_on_a_hierarchy(prec, monkeypatch):
    """Forced on every matrix that has a streamed candidate: each level's
    products and one V-cycle, whose residuals and corrections are fused.  FP
    rows are added in stored order: the same bits, signed zeros included."""
    monkeypatch.setenv("SC23AD_SPMV_FORMAT", "stream")
    sy = S.make_system(S.GEN_INCLUSIONS3D, (24, 8, 2.0, 4.0, 1e4, 3), 5)
    h = S.Hierarchy(sy.a, prec, S.amg_param(S.BLOCK_SOR))
    path = export(h)
    amg, oh = S.Amg(h), O.OracleHier(path)
    os.unlink(path)
    rng = np.random.default_rng(31)

    def vector(n):
        if prec == S.INT:
            return rng.integers(-2**20, 2**20, n).astype(np.int32)
        v = rng.standard_normal(n).astype(np.float64 if prec == S.FP64 else np.float32)
        v[::3] = -0.0
        return v

    for lv in range(amg.depth):
        n, nxt = oh.level_n(lv), oh.level_n(lv + 1)
        x, xc = vector(n), vector(nxt)
        for op in (S.OP_SPMV_A, S.OP_SPMV_U):
            assert amg.level_op(lv, op, x, n).tobytes() == oh.level_op(lv, op, x, n).tobytes(), lv
        assert (amg.level_op(lv, S.OP_SPMV_R, x, nxt).tobytes()
                == oh.level_op(lv, S.OP_SPMV_R, x, nxt).tobytes()), lv
        assert (amg.level_op(lv, S.OP_SPMV_P, xc, n).tobytes()
                == oh.level_op(lv, S.OP_SPMV_P, xc, n).tobytes()), lv
    v = vector(sy.a.n)
    assert amg.precondition(v).tobytes() == oh.vcycle(v).tobytes()
