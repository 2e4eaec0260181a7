"""What the library asks the runtime to launch, without a device: launch_recorder.cpp stands in for the HIP runtime."""
import os
import subprocess
import sys

import pytest

from effective_transformer_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))

# a line of output per launch (no device memory is touched, so any address does)
PREFIX = """
import ctypes as C, sys
recorder = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
recorder.recorded_launches.restype = C.c_char_p
sys.path.insert(0, sys.argv[2])
from effective_transformer_amd import _lib
lib = _lib.load()
handle = C.c_void_p()
assert lib.et_create(C.byref(handle), 0) == 0, lib.et_last_error(None)
some = C.c_void_p(1 << 40)
"""
# fp32 layers in the order given
LAYERS = PREFIX + """
weights = _lib.LayerWeights(*[1 << 40] * len(_lib.WEIGHT_FIELDS))
for heads, batch, seq, rows in eval(sys.argv[3]):
    nbytes = lib.et_layer_workspace_bytes(_lib.ET_FP32, batch, seq, heads, 64)
    s = lib.et_layer(handle, _lib.ET_FP32, C.byref(weights), some, some, some, some, some, some, C.c_void_p(1 << 41), batch, seq, seq,
                     heads, 64, rows, C.c_void_p(1 << 42), nbytes, None)
    assert s == 0, lib.et_last_error(handle)
print(recorder.recorded_launches().decode(), end="")
"""
# fp16 products on k-contiguous weights
PRODUCTS = PREFIX + """
for m, n, k, off in eval(sys.argv[3]):
    s = lib.et_gemm_bt(handle, _lib.ET_FP16, some, some, C.c_void_p((1 << 41) + off), None, m, n, k, None, None)
    assert s == 0, lib.et_last_error(handle)
print(recorder.recorded_launches().decode(), end="")
"""


@pytest.fixture(scope="module")
def recorder(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("recorder") / "librecorder.so")
    # (host code alone, and no runtime of its own beside it)
    subprocess.run([build.hipcc(), "-std=c++17", "-O1", "-shared", "-fPIC", "--offload-host-only", "-no-hip-rt", "-x", "hip",
                    os.path.join(HERE, "launch_recorder.cpp"), "-o", out], check=True, capture_output=True)
    return out


def _run(recorder, program, calls, cus=256):
    """[(kernel, workgroups, dynamic LDS, size raised)] of the calls in a process of their own."""
    r = subprocess.run([sys.executable, "-c", program, recorder, os.path.dirname(HERE), repr(calls)], capture_output=True, text=True,
                       env=dict(os.environ, RECORDER_CUS=str(cus)), timeout=120)
    assert r.returncode == 0, r.stderr
    found = [line.split() for line in r.stdout.splitlines()]
    return [(name, int(wgs), int(lds), int(raised)) for name, wgs, lds, raised in found]


def _launches(recorder, layers, cus=256):
    """The same of fp32 layers (heads, batch, seq, rows)."""
    found = _run(recorder, LAYERS, layers, cus)
    assert len(found) >= 8 * len(layers)
    return found


# rows for every height of tile
@pytest.mark.parametrize("rows", [30, 200, 900, 3000, 8000, 30000])
@pytest.mark.parametrize("heads", [(8, 12, 29, 30, 31, 32), (32, 31, 30, 8)])
def test_no_launch_takes_more_lds_than_its_kernel_was_given(recorder, heads, rows):
    """The output product's LDS grows with the hidden size: whatever size came first, the next one's must have been asked for."""
    for name, _, lds, raised in _launches(recorder, [(h, 1000, 32, rows) for h in heads]):
        assert lds <= max(raised, 64 * 1024), "%s: %d bytes of LDS, %d asked for" % (name, lds, raised)


@pytest.mark.parametrize("cus", [64, 256])
def test_blocks_without_queries_come_last_beyond_four_workgroups_a_cu(recorder, cus):
    """8 heads and 192 positions, three blocks of queries: on both sides of four workgroups a CU."""
    most = 4 * cus // 24
    for batch in (most, most + 1):
        attention = [name for name, *_ in _launches(recorder, [(8, batch, 192, batch * 100)], cus) if "attention_flash_f32" in name]
        assert len(attention) == 1 and ("ILb1E" in attention[0]) == (batch > most)


# rows on both sides of 2^32 threads in wavefronts of 16 x 16 tiles; the longest rows a matrix of 288 GB has; the last of shorter rows
@pytest.mark.parametrize("m,n", [(1008, 1 << 24), (1009, 1 << 24), (8192, 1 << 24), (33, (1 << 26) + 8), (2, 2 ** 31 - 4096), (1024, (1 << 24) - 8)])
@pytest.mark.parametrize("off", [0, 2])
def test_longest_rows_of_products_go_to_large_tiles(recorder, m, n, off):
    """A C of rows from 2^24 values on, 8-byte aligned or not: a workgroup to a tile of 128 x 128, in a grid that a launch takes."""
    (name, wgs, _, _), = _run(recorder, PRODUCTS, [(m, n, 64, off)])
    assert "gemm_f16_bt_kernelILi4ELi4ELi2E" in name
    tiles = (m + 127) // 128 * ((n + 127) // 128)
    assert tiles <= wgs < tiles + 8 and wgs * 256 < 1 << 32
