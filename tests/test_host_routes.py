"""The host library's own decisions, without a GPU: zlm_gpu_hip.cpp built
against a HIP runtime that allocates host memory under a limit and runs no
kernels (tests/fake_hip.cpp).  What a call launches comes from the launch log,
what it allocates, frees, copies and waits for from the runtime's counters.
Numerical results of the same routes are the GPU tests' part."""
import ctypes
import importlib.util
import os
import subprocess
import sys

import numpy as np
import pytest

from zlm_amd import device as zd
from zlm_amd import synth

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIVE, MALLOCS, REFUSED, FREES, SYNCS, H2D, D2H, MISUSE = range(8)
NO_LIMIT = (1 << 64) - 1


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    """The package's device module over the library built with the stand-in runtime."""
    lib = tmp_path_factory.mktemp("fake_hip") / "libzlm_gpu_hip.so"
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-w", "-D__HIP_PLATFORM_AMD__", f"-I{rocm}/include",
                    f"-I{ROOT}/include", f"-I{ROOT}/zlm_amd/csrc", f"{ROOT}/zlm_amd/csrc/zlm_gpu_hip.cpp",
                    f"{ROOT}/tests/fake_hip.cpp", "-Wl,-Bsymbolic", "-ldl", "-o", str(lib)], check=True)
    spec = importlib.util.spec_from_file_location("zlm_device_fake_hip", zd.__file__)
    mod = importlib.util.module_from_spec(spec)
    sys.modules[spec.name] = mod
    spec.loader.exec_module(mod)
    mod.LIB_PATH = str(lib)
    raw = mod.lib()
    raw.fake_hip_stat.restype = ctypes.c_uint64
    raw.fake_hip_limit.argtypes = [ctypes.c_uint64]
    return mod


class _Box:
    """A device over the stand-in runtime, with device buffers for x and out."""

    def __init__(self, mod, x_floats, out_floats):
        self.raw = mod.lib()
        self.raw.fake_hip_limit(NO_LIMIT)
        self.dev = mod.Device()
        assert self.dev.available(), self.dev.last_error()
        self.misuse = self.stat(MISUSE)
        self.x, self.out = self.dev.dev_malloc(4 * x_floats), self.dev.dev_malloc(4 * out_floats)

    def stat(self, i):
        return int(self.raw.fake_hip_stat(i))

    def resident(self, qt, rows, k):
        res = self.dev.upload_resident(np.zeros(rows * synth.row_bytes(qt, k), np.uint8))
        assert res is not None
        return res

    def run(self, res, qt, rows, k, m):
        """(accepted, the launches that do not convert weights)"""
        assert self.dev.launch_log(True)
        ok = self.dev.mat_mul_enqueue(res, zd.quant(qt), rows, k, m, self.x, self.out)
        log = [r for r in self.dev.launch_log_read() if r["what"] not in ("repack", "repack records", "tile weights")]
        return ok, log

    def whats(self, *call):
        ok, log = self.run(*call)
        assert ok, self.dev.last_error()
        return [r["what"] for r in log]


@pytest.fixture
def box(fake):
    made = []

    def make(x_floats, out_floats):
        made.append(_Box(fake, x_floats, out_floats))
        return made[-1]

    yield make
    for b in made:
        assert b.stat(MISUSE) == b.misuse
        b.raw.fake_hip_limit(NO_LIMIT)
        b.dev.deinit()


def test_wide_gemm_where_memory_is_spent(box):
    """The wide GEMM's activations take more scratch than the tiled form's.  A
    refused growth costs nothing that the call or a later one needs."""
    qt, k, m = synth.Q4_1, 1536, 512
    rows = 56 * 192
    b = box(m * k, m * rows)
    res = b.resident(qt, rows, k)
    spare = b.dev.dev_malloc(1 << 20)
    assert b.whats(res, qt, 640, k, m)[0] == "quantize tiled"  # the tiles and the tiled form's scratch
    scratch = b.dev.scratch_device_bytes()
    b.raw.fake_hip_limit(b.stat(LIVE))
    freed, synced, refused = b.stat(FREES), b.stat(SYNCS), b.stat(REFUSED)
    for _ in range(3):
        assert b.whats(res, qt, rows, k, m) == ["quantize tiled", "gemm"]
        assert b.dev.last_error() == ""
    assert (b.stat(FREES), b.stat(SYNCS)) == (freed, synced)
    assert b.stat(REFUSED) == refused + 1  # asked once
    assert b.dev.scratch_device_bytes() == scratch
    # memory that this library gives back is a reason to ask again; here it is still too little
    b.dev.dev_free(spare)
    assert b.whats(res, qt, rows, k, m) == ["quantize tiled", "gemm"]
    assert b.stat(REFUSED) == refused + 2
    b.raw.fake_hip_limit(NO_LIMIT)
    assert b.whats(res, qt, rows, k, m) == ["quantize tiled", "gemm"]
    b.dev.free_resident(b.resident(qt, 32, k))
    assert b.whats(res, qt, rows, k, m) == ["quantize tiled", "gemm wide"]
    assert b.dev.scratch_device_bytes() > scratch
    b.dev.free_resident(res)


# Eager 5 to 8 tokens by a tall weight are the whole preparation that a capture
# of up to 32 tokens needs, as they are where the small-M GEMM runs them: the
# tall kernel itself builds neither tiles nor scratch, so the capture's begin does.
TALL = [(synth.Q4_0, 65536, 64), (synth.Q4_1, 32768, 4160), (synth.Q4_K, 32768, 256)]


@pytest.mark.parametrize("qt,rows,k", TALL)
def test_capture_after_eager_tall_tokens(box, qt, rows, k):
    b = box(32 * k, 32 * rows)
    res = b.resident(qt, rows, k)
    assert b.whats(res, qt, rows, k, 8) == ["gemm tall"]
    held = b.dev.resident_device_bytes(res)
    assert held == zd.layout_bytes(zd.quant(qt), rows, k, False)  # no tiled copy yet
    assert b.dev.capture_begin(), b.dev.last_error()
    assert b.dev.resident_device_bytes(res) == zd.layout_bytes(zd.quant(qt), rows, k, True)
    for m in (9, 32):
        assert b.whats(res, qt, rows, k, m) == ["quantize tiled", "gemm small"]
    assert b.whats(res, qt, rows, k, 8) == ["gemm tall"]
    assert not b.run(res, qt, rows, k, 33)[0]  # more scratch than eight eager tokens ask for
    assert "eager call before capture" in b.dev.last_error()
    graph = b.dev.capture_end()
    assert graph
    b.dev.graph_destroy(graph)
    mallocs = b.stat(MALLOCS)
    assert b.dev.capture_begin()  # once is enough
    b.dev.graph_destroy(b.dev.capture_end())
    assert b.stat(MALLOCS) == mallocs
    b.dev.free_resident(res)


def test_capture_without_eager_tokens_is_refused(box):
    qt, rows, k = TALL[0]
    b = box(32 * k, 32 * rows)
    few, released, freed = (b.resident(qt, rows, k) for _ in range(3))
    assert b.whats(few, qt, rows, k, 4) == ["gemm tall"]  # 3 and 4 tokens never prepared a GEMM
    for r in (released, freed):
        assert b.whats(r, qt, rows, k, 8) == ["gemm tall"]
    assert b.dev.release_gemm_tiles(released)
    b.dev.free_resident(freed)
    assert b.dev.capture_begin(), b.dev.last_error()
    for r in (few, released):
        assert not b.run(r, qt, rows, k, 16)[0]
        assert "tiles must be built by an eager matMul" in b.dev.last_error()
    b.dev.graph_destroy(b.dev.capture_end())
    b.dev.free_resident(few)
    b.dev.free_resident(released)


def test_capture_begins_where_memory_for_the_tiles_is_spent(box):
    qt, rows, k = TALL[0]
    b = box(32 * k, 32 * rows)
    res = b.resident(qt, rows, k)
    assert b.whats(res, qt, rows, k, 8) == ["gemm tall"]
    b.raw.fake_hip_limit(b.stat(LIVE))
    assert b.dev.capture_begin()
    assert b.dev.last_error() == ""
    assert b.whats(res, qt, rows, k, 8) == ["gemm tall"]
    assert not b.run(res, qt, rows, k, 16)[0]
    b.dev.graph_destroy(b.dev.capture_end())
    b.dev.free_resident(res)


@pytest.mark.parametrize("qt,rows,k,m", [(synth.Q4_0, 64, 256, 16), (synth.Q4_K, 32768, 256, 8), (synth.Q8_0, 64, 64, 2)])
def test_streamed_weight_leaves_nothing_behind(box, qt, rows, k, m):
    """matMulBatch over a host weight: its tiled copy goes with the call."""
    b = box(m * k, m * rows)
    w = np.zeros(rows * synth.row_bytes(qt, k), np.uint8)
    x, out = np.zeros(m * k, np.float32), np.zeros(m * rows, np.float32)
    assert b.dev.mat_mul_batch(zd.quant(qt), w, rows, k, m, x, out), b.dev.last_error()
    live = b.stat(LIVE)
    for _ in range(3):
        assert b.dev.mat_mul_batch(zd.quant(qt), w, rows, k, m, x, out), b.dev.last_error()
    assert b.stat(LIVE) == live
    assert b.dev.capture_begin()  # and nothing of it is prepared for a capture
    b.dev.graph_destroy(b.dev.capture_end())
    assert b.stat(LIVE) == live


# How a host matMul's x and y cross, either side of each line: y stored by the
# product into pinned memory ("direct") or copied by DMA, x by the copy kernel or
# by DMA (q8_0, q4_0 / q4_1 and q4_k store at their own rates).
CROSS = [  # quant, rows, k, m, y direct, x by the copy kernel
    (synth.Q4_0, 40960, 2048, 1, True, True), (synth.Q4_0, 40961, 2048, 1, False, True),
    (synth.Q4_0, 131072, 1024, 1, False, True), (synth.Q4_K, 131072, 2048, 1, False, True),
    (synth.Q4_K, 65536, 3072, 1, True, True), (synth.Q8_0, 65536, 3072, 1, False, True),
    (synth.Q8_0, 65536, 3840, 1, True, True), (synth.Q4_0, 262145, 3072, 1, False, True),
    (synth.Q4_0, 65536, 64, 2, True, True), (synth.Q4_0, 65537, 64, 2, False, True),
    (synth.Q4_1, 131072, 64, 2, False, True), (synth.Q4_K, 131072, 256, 2, True, True),
    (synth.Q4_K, 131073, 256, 2, False, True), (synth.Q8_0, 65537, 1024, 2, False, True),
    (synth.Q8_0, 65537, 2048, 2, True, True),
    (synth.Q8_0, 196608, 64, 4, True, True), (synth.Q8_0, 196609, 64, 4, False, True),
    (synth.Q8_0, 49153, 4096, 4, True, True), (synth.Q4_1, 98305, 96, 8, False, True),
    (synth.Q4_0, 131072, 64, 8, True, True), (synth.Q4_0, 131073, 64, 8, False, True),
    (synth.Q4_0, 131073, 2048, 8, True, True),
    (synth.Q4_0, 64, 4096, 56, True, True), (synth.Q4_0, 64, 4096, 57, True, False),
    (synth.Q4_0, 98304, 32, 32, True, True), (synth.Q4_0, 98305, 32, 32, False, True),
    (synth.Q4_0, 98305, 544, 32, False, False), (synth.Q4_0, 4096, 512, 500, False, False),  # the second tiled
    (synth.Q4_K, 8192, 256, 64, False, True), (synth.Q4_K, 8192, 512, 64, False, False),
]


@pytest.mark.parametrize("qt,rows,k,m,direct,staged", CROSS)
def test_host_matmul_crossing(box, qt, rows, k, m, direct, staged):
    b = box(16, 16)
    res = b.resident(qt, rows, k)
    x, out = np.zeros(m * k, np.float32), np.zeros(m * rows, np.float32)
    h2d, d2h = b.stat(H2D), b.stat(D2H)
    assert b.dev.launch_log(True)
    assert b.dev.mat_mul_resident(res, zd.quant(qt), rows, k, m, x, out), b.dev.last_error()
    assert (b.stat(D2H) == d2h, b.stat(H2D) == h2d) == (direct, staged)
    assert ("stage x" in [r["what"] for r in b.dev.launch_log_read()]) == staged
    b.dev.free_resident(res)


# Where the wide fp6 GEMM runs: one round of its workgroups (128 tokens x 192 rows, 256
# CUs), or several where rows have 96 blocks and the rounds are 7/8 full.
@pytest.mark.parametrize("qt,rows,k,m,what", [
    (synth.Q4_1, 56 * 192, 1536, 512, "gemm wide"), (synth.Q4_1, 55 * 192, 1536, 512, "gemm"),
    (synth.Q4_1, 49152, 42 * 32, 128, "gemm"), (synth.Q4_1, 49152, 43 * 32, 128, "gemm wide"),  # the shortest rows
    (synth.Q4_1, 49152, 96 * 32 - 32, 256, "gemm"), (synth.Q4_1, 49152, 96 * 32, 256, "gemm wide"),
    (synth.Q4_K, 12288, 2816, 1024, "gemm"), (synth.Q4_K, 12288, 3072, 1024, "gemm wide"),
    (synth.Q4_K, 49152, 256, 1024, "gemm"), (synth.Q4_0, 12288, 3072, 1024, "gemm")])
def test_wide_gemm_route(box, qt, rows, k, m, what):
    b = box(16, 16)
    res = b.resident(qt, rows, k)
    assert b.whats(res, qt, rows, k, m) == ["quantize tiled", what]
    b.dev.free_resident(res)


@pytest.mark.parametrize("qt,rows,m", [(synth.Q4_K, 32768, 5), (synth.Q4_1, 40001, 8), (synth.Q4_0, 65536, 3)])
def test_tall_kernel_covers_the_chip(box, qt, rows, m):
    """One workgroup per CU, also where that leaves some of its 16 waves without a 16-row tile."""
    b = box(16, 16)
    res = b.resident(qt, rows, 256)
    ok, log = b.run(res, qt, rows, 256, m)
    assert ok, b.dev.last_error()
    assert [(r["what"], r["grid_x"], r["block"]) for r in log] == [("gemm tall", 256, 1024)]
    b.dev.free_resident(res)
