"""C ABI of gnn_rows_product / gnn_reduce_parts on a CPU-only host: the ctypes mirrors have the C
layout and argument errors come back before any GPU work."""

import ctypes
import pathlib
import subprocess

import pytest

from geometric_nn_ops_torch import _lib

ROOT = pathlib.Path(__file__).resolve().parent.parent


def test_structs_match_c_layout(tmp_path):
    fields = {"gnn_rows_product_item": _lib.RowsProductItem, "gnn_rows_product_args": _lib.RowsProductArgs,
              "gnn_reduce_segment": _lib.ReduceSegment, "gnn_reduce_args": _lib.ReduceArgs}
    body = "".join(f'printf("%zu\\n", sizeof({name}));' + "".join(
        f'printf("%zu\\n", offsetof({name}, {f}));' for f, *_ in cls._fields_) for name, cls in fields.items())
    c = tmp_path / "layout.c"
    c.write_text('#include <stdio.h>\n#include <stddef.h>\n#include "gnn_triangle.h"\nint main(void) {' + body + "}")
    subprocess.run(["gcc", "-std=c11", f"-I{ROOT / 'include'}", str(c), "-o", str(tmp_path / "layout")], check=True)
    got = subprocess.run([str(tmp_path / "layout")], capture_output=True, text=True, check=True).stdout.split()
    want = [v for cls in fields.values() for v in (ctypes.sizeof(cls), *(getattr(cls, f).offset for f, *_ in cls._fields_))]
    assert [int(v) for v in got] == want


def _product(**kw):
    a = _lib.RowsProductArgs()
    a.rows, a.count, a.dtype = 64, 1, _lib.GNN_BF16
    p = a.p[0]
    p.d, p.t, p.partial, p.d_ld, p.t_ld, p.O, p.I = 4096, 8192, 4096, 32, 16, 32, 16
    for k, v in kw.items():
        setattr(a if hasattr(a, k) else p, k, v)
    return a


@pytest.mark.parametrize("bad", [{"rows": 0}, {"count": 0}, {"count": 5}, {"dtype": 9}, {"O": 12}, {"I": 0},
                                 {"d_ld": 24}, {"t_ld": 20}, {"d": None}, {"partial": None}, {"t": 8200}])
def test_rows_product_argument_errors(bad):
    lib = _lib.load()
    assert lib.gnn_rows_product(ctypes.byref(_product(**bad)), None) == _lib.GNN_ERR_ARG
    assert lib.gnn_last_error()


def test_null_args():
    lib = _lib.load()
    assert lib.gnn_rows_product(None, None) == _lib.GNN_ERR_ARG
    assert lib.gnn_reduce_parts(None, None) == _lib.GNN_ERR_ARG
    assert lib.gnn_rows_product_slices(None) == 0


@pytest.mark.parametrize("bad", [{"parts": 0}, {"n": 0}, {"stride": 3}, {"dtype": 7}, {"src": None}, {"dst": 4098}])
def test_reduce_argument_errors(bad):
    a = _lib.ReduceArgs()
    a.count = 1
    s = a.seg[0]
    s.src, s.dst, s.parts, s.stride, s.n, s.dtype = 4096, 8192, 2, 16, 16, _lib.GNN_F32
    for k, v in bad.items():
        setattr(s, k, v)
    assert _lib.load().gnn_reduce_parts(ctypes.byref(a), None) == _lib.GNN_ERR_ARG


@pytest.mark.parametrize("rows", [1, 31, 257, 5000, 40401, 147456])
@pytest.mark.parametrize("cus", [1, 32, 256])
def test_the_launch_is_held_to_the_slices_that_were_allocated(rows, cus, monkeypatch):
    """The number of slices follows the compute units of whichever device is current when it is asked
    for; the tensors' own device must not decide again. The wrapper passes the split on."""
    import torch

    from geometric_nn_ops_torch.triangle._kernels import trimul as K

    per = max(-(-rows // max(1, 2 * cus)), 256)
    chosen = -(-rows // (-(-per // 32) * 32))

    class Lib:
        def gnn_rows_product_slices(self, args):
            return chosen

    launched = []
    monkeypatch.setattr(_lib, "load", lambda: Lib())
    monkeypatch.setattr(_lib, "call", lambda fn, a, device: launched.append((fn, a.slice_rows)))
    (part,) = K.rows_products_hip([(torch.empty(rows, 8, dtype=torch.bfloat16), torch.empty(rows, 8, dtype=torch.bfloat16))])
    monkeypatch.undo()
    assert part.shape[0] == chosen and launched[0][0] == "gnn_rows_product"
    again = _product(rows=rows, slice_rows=launched[0][1])
    assert launched[0][1] > 0 and _lib.load().gnn_rows_product_slices(ctypes.byref(again)) == chosen
