"""CPU: the by-value tables the Python calls fill (RowIdx, DSampArgs) take what ctypes takes, element by element: integers that wrap
into their field, numbers beyond float32's range, any iterable."""
import ctypes as C

import pytest

import gpu_cases

ROW = dict(top_k=20, qoff=72, inv_t=1.25, top_p=0.95, min_p=0.02, key=0x123456789abcdef0)


def one_by_one(m, args):
    da = m.DSampArgs()
    for i, a in enumerate(args):
        da.on[i], da.top_k[i], da.qoff[i] = a.get("on", 1), a["top_k"], a["qoff"]
        da.inv_t[i], da.top_p[i], da.min_p[i] = a["inv_t"], a["top_p"], a["min_p"]
        da.key_lo[i], da.key_hi[i] = a["key"] & 0xFFFFFFFF, a["key"] >> 32
    return bytes(da)


@pytest.mark.parametrize("change", [dict(), dict(on=0), dict(key=-1), dict(key=-(1 << 63)), dict(key=(1 << 64) - 1), dict(top_k=(1 << 32) - 1),
                                    dict(qoff=-72), dict(inv_t=1e300), dict(inv_t=float("inf"), min_p=1), dict(top_p=True)])
@pytest.mark.parametrize("rows", [1, 7, 32])
def test_draft_arguments(change, rows):
    m = gpu_cases.pkg()
    args = [dict(ROW, key=ROW["key"] + i) for i in range(rows)]
    args[rows // 2].update(change)
    want = one_by_one(m, args)
    assert bytes(m._dsamp_args(args)) == want
    assert bytes(m._dsamp_args(iter(args))) == want and bytes(m._dsamp_args(tuple(args))) == want


def test_draft_arguments_that_are_refused():
    m = gpu_cases.pkg()
    assert bytes(m._dsamp_args([])) == bytes(m.DSampArgs())
    with pytest.raises(IndexError):
        m._dsamp_args([ROW] * 33)
    with pytest.raises(KeyError):
        m._dsamp_args([dict(ROW), {k: v for k, v in ROW.items() if k != "min_p"}])
    with pytest.raises(TypeError):
        m._dsamp_args([dict(ROW, top_k=1.5)])


def test_row_tables_from_any_iterable():
    m = gpu_cases.pkg()
    want = (C.c_int32 * 32)(*range(5, 25))
    for values in (list(range(5, 25)), tuple(range(5, 25)), range(5, 25), iter(range(5, 25)), {v: 0 for v in range(5, 25)}):
        assert list(m._row_idx(values).v) == list(want)
    for values in (list(range(33)), iter(range(33))):
        with pytest.raises(IndexError):
            m._row_idx(values)
