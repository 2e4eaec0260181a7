"""Bytes of arguments that a kernel's launches hand over, as the built library's metadata states them.

Encoders of few rows are issued by the host, and the size of a launch's arguments is part of what that costs: with 16 bytes more
that only fp32 launches read, the 12 attention launches of one query (1 x 32, fp16) took the encoder 3 % longer."""
import os
import struct

import msgpack

from effective_transformer_amd import _lib


def _kernels():
    """name -> metadata of every kernel: the code objects lie in the library as they are, each with one AMDGPU note."""
    with open(_lib.LIB_PATH, "rb") as f:
        data = f.read()
    found, at = {}, data.find(b"AMDGPU\0\0")
    while at >= 0:
        name_size, size, kind = struct.unpack_from("<III", data, at - 12)
        if name_size == 7 and kind == 32:
            for kernel in msgpack.unpackb(data[at + 8:at + 8 + size], strict_map_key=False)["amdhsa.kernels"]:
                found[kernel[".name"]] = kernel
        at = data.find(b"AMDGPU\0\0", at + 8)
    return found


def _argument_bytes(kernel):
    return max(a[".offset"] + a[".size"] for a in kernel[".args"] if not a[".value_kind"].startswith("hidden_"))


def test_fp16_attention_is_handed_nothing_of_fp32():
    assert os.path.exists(_lib.LIB_PATH)
    short = {n: k for n, k in _kernels().items() if "16attention_kernelI" in n}
    half = [k for n, k in short.items() if "attention_kernelIDF16_" in n]
    full = [k for n, k in short.items() if "attention_kernelIf" in n]
    assert half and full
    # seven pointers, six sizes, the scale and the form of the result
    assert {_argument_bytes(k) for k in half} == {7 * 8 + 6 * 4 + 2 * 4}
    # and where the exponents of the heads go
    assert {_argument_bytes(k) for k in full} == {7 * 8 + 6 * 4 + 2 * 4 + 16}
