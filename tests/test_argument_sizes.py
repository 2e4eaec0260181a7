"""What the launches of an fp16 encoder of few rows hand over: up to 112 bytes of arguments each, from 116 on the host takes 0.8 us longer."""
import pytest

from test_kernel_arguments import _argument_bytes, _kernels

FEW_ROWS = ("gemm_f16_bt_kernel", "gemm_f16_bt_wave_kernel", "gemm_f16_bt_quad_kernel", "bias_residual_layernorm_kernelIDF16_", "16attention_kernelIDF16_",
            "attention_flash_kernel", "compress_rows_kernel", "mapped_restore_rows_kernel", "scan_index_kernel", "mask_class_kernel")


@pytest.mark.parametrize("name", FEW_ROWS)
def test_arguments_of_few_rows(name):
    kernels = {n: k for n, k in _kernels().items() if name in n}
    assert kernels
    for n, k in kernels.items():
        assert _argument_bytes(k) <= 112, n
        assert k[".kernarg_segment_size"] <= 112, n       # (the size of the grid, where a kernel asks for it, is 256 bytes of it)
