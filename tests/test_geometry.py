"""Launch rules shared by the host and the kernels (kernel_geometry.h), checked
on the CPU against the memory that the kernels' rows really cover, and the
kernels that the GPU tests' shapes reach by them."""
import ctypes
import os
import subprocess

import pytest

import test_hip_fp8
import test_hip_ops
from support import BF16, ELEM_BYTES, FP16, FP32, ROOT

# the kernels by smx_route's index; "main" holds rows whole (fp8: prefetches),
# "stream" and "element" are the main kernels' other paths
ROUTES = ["main", "rows", "wide", "long", "split", "any", "stream", "element"]


def compiled(out, *flags):
    subprocess.run(["gcc", "-O2", "-Wall", "-Werror", "-Wno-unused-function", "-I", os.path.join(ROOT, "dataflow_lib_amd", "csrc", "kernels"),
                    os.path.join(ROOT, "tests", "geometry_check.c"), "-o", out, *flags], check=True)
    return out


def test_softmax_row_windows_fit_their_launch(tmp_path):
    res = subprocess.run([compiled(str(tmp_path / "geometry_check"))], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout


@pytest.fixture(scope="module")
def route(tmp_path_factory):
    lib = ctypes.CDLL(compiled(str(tmp_path_factory.mktemp("geometry") / "libgeometry.so"), "-shared", "-fPIC"))
    lib.smx_route.argtypes = [ctypes.c_int] * 3 + [ctypes.c_ulonglong] * 2

    def of(elem, shape, x=0, out=0):
        return ROUTES[lib.smx_route(shape[0], shape[1], elem, 4096 + x, 8192 + out)]

    return of


@pytest.mark.parametrize("dt", [FP32, FP16, BF16], ids=test_hip_ops.dt_id)
def test_softmax_test_shapes_reach_every_kernel(route, dt):
    """Plain, special and shifted rows of the GPU tests each run on every kernel
    that their type has (split and unaligned ones among the offset shapes)."""
    T, es = test_hip_ops, ELEM_BYTES[dt]
    every = {"main", "rows", "wide", "split", "any", "stream"} | ({"long"} if es == 2 else set())
    plain = {route(es, s) for s in T.SMX_SHAPES} | {route(es, s, s[2] * es, s[2] * es) for s in T.ROW_SHAPES}
    special = {route(es, s) for s in T.SPECIAL_ROWS + T.MANY_ROWS}
    shifted = {route(es, s) for s in T.SHIFTED_SHAPES + T.WHOLE_ROW_SHAPES}
    assert plain >= every and special >= every and shifted >= every - {"wide"}
    assert {route(es, (600 if c[0] <= 1000 else 66, c[0])) for c in T.FAR_CASES} >= {"main", "rows"} | ({"stream"} if es == 4 else set())
    assert {route(es, s) for s in T.MARGIN_SHAPES} >= {"rows", "any"} | ({"main", "long"} if es == 2 else {"stream"})
    assert route(es, (66, 128256), 0, es) == "element"


def test_softmax_counter_test_takes_tickets(route):
    """more than two rows per workgroup where rows are held whole, more than
    one where they are streamed, and small grids and split rows between"""
    taken = [(route(ELEM_BYTES[dt], s), s[0]) for dt, _, s in test_hip_ops.COUNTER_CASES]
    ticketed = {r for r, n in taken if n > (512 if r in ("main", "long") else 256)}
    assert ticketed >= {"main", "long", "any", "stream"} and {r for r, _ in taken} >= {"rows", "split"}


def test_softmax_fp8_test_shapes_reach_every_kernel(route):
    T = test_hip_fp8
    every = {"main", "rows", "wide", "split", "element"}
    assert {route(1, s) for s in T.SMX_SPECIAL} == every
    assert {route(1, s, 5 if s in T.SMX_UNALIGNED else 0) for s in T.SMX_SHAPES} == every
    assert route(1, (600, 65552)) == "main" and route(2, (600, 66000)) == "main"   # the two-stream test
