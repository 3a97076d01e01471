"""The library's planning, scratch and dispatch on the CPU: tests/cpp/fake_hip.cpp stands in for the HIP
runtime (no device, launches run nothing), in a process of its own with it preloaded. The profiler's
keys then name the plan of a call, and allocations can be refused."""
from __future__ import annotations

import os
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
SRC = ROOT / "tests" / "cpp" / "fake_hip.cpp"

PRELUDE = """
import ctypes as C
import irontensor_amd as it
from irontensor_amd import _lib, profiler
fake = C.CDLL(None)
fake.fake_hip_limit.argtypes = [C.c_size_t]
fake.fake_hip_launches.restype = C.c_char_p
ctx = it.Context.global_()
def launches():
    return fake.fake_hip_launches().decode().split()
def buf(elements):
    return it.Tensor.empty([elements])
def gemm(bf16, ta, tb, m, n, k, a, b, c, batch=1, sa=0, sb=0, sc=0, lda=None, ldb=None, epi=None):
    return ctx.lib.it_gemm(ctx.handle, 2 if bf16 else 0, 0, ta, tb, m, n, k, 1.0, C.c_void_p(a), lda or (m if ta else k),
                           sa, C.c_void_p(b), ldb or (k if tb else n), sb, 0.0, C.c_void_p(c), n, sc, batch,
                           C.byref(epi) if epi is not None else None)
def keys(f):
    profiler.reset(ctx)
    profiler.enable(ctx)
    assert f() == 0, ctx.lib.it_last_error()
    got = list(profiler.stats(ctx))
    profiler.enable(ctx, False)
    return got
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    lib = tmp_path_factory.mktemp("fake") / "fake_hip.so"
    res = subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                          str(SRC), "-o", str(lib)], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert res.returncode == 0, res.stdout
    return lib


def _run(fake, body):
    preload = ":".join([str(fake)] + [p for p in [os.environ.get("LD_PRELOAD")] if p])
    res = subprocess.run([sys.executable, "-c", PRELUDE + body], stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                         text=True, timeout=300, cwd=ROOT, env=dict(os.environ, LD_PRELOAD=preload))
    print(res.stdout)
    assert res.returncode == 0, res.stdout[-3000:]


def test_refused_scratch_falls_back(fake):
    """A product whose faster plan needs scratch that cannot be had runs on the plan without, and nothing
    reports the refused allocation afterwards: BF16 operands that need padded copies take the plain
    tiles, an FP32 product is not split, and a group of FP32 products runs as separate ones."""
    _run(fake, """
A, B, Cc = buf(1999 * 1237), buf(3001 * 1237), buf(1999 * 3001)
ragged = lambda: gemm(1, 0, 1, 1999, 3001, 1237, A.ptr, B.ptr, Cc.ptr)
split = lambda: gemm(0, 1, 0, 256, 256, 4096, A.ptr, B.ptr, Cc.ptr)
call = lambda c: _lib.GemmCall(1, 0, 256, 256, 4096, 1.0, A.ptr, 256, 0, B.ptr, 256, 0, 0.0, c, 256, 0, 1, None)
calls = (_lib.GemmCall * 2)(call(Cc.ptr), call(Cc.ptr + 4 * 65536))
group = lambda: ctx.lib.it_gemm_group(ctx.handle, 0, 0, 2, calls)
fake.fake_hip_limit(1 << 20)
for f, needs in ((ragged, '_dtl_edge'), (split, None), (group, '_group')):
    got = keys(f)
    print('refused:', got, flush=True)
    assert got and all(k.endswith(' s1') for k in got) and not any(needs and needs in k for k in got), got
    assert not any('reduce' in k for k in launches())
fake.fake_hip_limit((1 << 64) - 1)
for f, needs in ((ragged, '_dtl_edge'), (split, ' s'), (group, '_group')):
    got = keys(f)
    print('granted:', got, flush=True)
    assert any(needs in k for k in got), got
assert not keys(split)[0].endswith(' s1')
""")


def test_shared_operand_is_padded_once(fake):
    """A ragged BF16 B that a batch shares (stride 0) takes one padded copy: forty of this one would pass the
    1 GB that such copies may take, and the product would stay on the plain tiles."""
    _run(fake, """
bt, m, n, k = 40, 128, 4097, 4001
A, B, Cc = buf(bt * m * k // 2 + 1), buf(n * k // 2 + 1), buf(bt * m * n)
got = keys(lambda: gemm(1, 0, 1, m, n, k, A.ptr, B.ptr, Cc.ptr, bt, m * k, 0, m * n))
print(got)
assert '_dtl_edge' in got[0], got
""")


def test_operands_beyond_the_edge_tiles_offsets(fake):
    """A ragged product over a B whose k rows span more than 2 GiB a split has no edge-tile plan and stays on
    the plain tiles (launched on nothing here: the buffer is not that large)."""
    _run(fake, """
X = buf(1 << 22)
got = keys(lambda: gemm(1, 0, 0, 1000, 1000, 4096, X.ptr, X.ptr, X.ptr, ldb=1 << 23))
print(got)
assert '_edge' not in got[0], got
""")


def test_padded_copies_are_given_back(fake):
    """it_empty_cache frees the scratch of a ragged BF16 product's padded copies; while a graph is alive, which
    may hold its address, it stays, and later products take it again."""
    _run(fake, """
A, B, Cc = buf(8001 * 4001 // 2 + 1), buf(4001 * 8003 // 2 + 1), buf(8001 * 8003)
f = lambda: gemm(1, 0, 1, 8001, 8003, 4001, A.ptr, B.ptr, Cc.ptr)
scratch = lambda: ctx.lib.it_mem_scratch(ctx.handle)
before = scratch()
assert '_dtl_edge' in keys(f)[0] and scratch() - before > 100e6
assert ctx.lib.it_empty_cache(ctx.handle) == 0 and scratch() == before
assert '_dtl_edge' in keys(f)[0] and scratch() - before > 100e6
g = C.c_void_p()
assert ctx.lib.it_capture_begin(ctx.handle) == 0 and f() == 0
assert 'pad_bf16' in ' '.join(launches())
assert ctx.lib.it_capture_end(ctx.handle, C.byref(g)) == 0
assert ctx.lib.it_empty_cache(ctx.handle) == 0 and scratch() - before > 100e6
assert ctx.lib.it_graph_destroy(g) == 0
assert ctx.lib.it_empty_cache(ctx.handle) == 0 and scratch() == before
""")


def test_small_ragged_products_stay_on_the_plain_tiles(fake):
    """Ragged BF16 products of whole 16-byte vectors and little work are faster on the plain tiles' masked loads
    (7.0 against 12.7 us, 10.9 against 16.5); long or unaligned ones on the edge tiles."""
    _run(fake, """
X = buf(1 << 24)
for ta, tb, m, n, k, edge in ((1, 0, 448, 1776, 64, 0), (0, 0, 7840, 392, 152, 0), (0, 0, 104, 104, 280, 0),
                              (0, 1, 1999, 3001, 1237, 1), (0, 1, 2000, 3000, 1240, 1), (1, 0, 529, 210, 6306, 1)):
    got = keys(lambda: gemm(1, ta, tb, m, n, k, X.ptr, X.ptr, X.ptr))
    print(got, flush=True)
    assert ('_dtl_edge' in got[0]) == bool(edge), got
""")
