"""The form in which HipBackend hands activations to the quantized products:
fp32 rows as they are where rounding them in the kernel is no slower than one
cast first, fp16 rows elsewhere (no GPU: the choice is the host's)."""
import types

import pytest
import torch

from versenext_amd import _lib
from versenext_amd.hip_backend import HipBackend


def _form(x, N):
    be = types.SimpleNamespace(_torch_device=torch.device("cpu"))
    be._acts = lambda t, K: HipBackend._acts(be, t, K)
    lead, rows, code = HipBackend._linear_x(be, x, x.shape[-1], N)
    assert lead == x.shape[:-1] and rows.shape == (x[..., 0].numel(), x.shape[-1]) and rows.stride(1) == 1
    assert rows.dtype == (torch.float32 if code == _lib.VNX_F32 else torch.float16)
    assert torch.equal(rows.half(), x.reshape(rows.shape).half())
    return code


# both sides of each line: outputs x K of a workgroup per 16 weight rows, K
# alone, outputs of the tiled GEMM; an LM head's weight rows
@pytest.mark.parametrize("rows,N,K,direct", [
    (1, 1024, 1024, True), (16, 8192, 5120, True), (17, 8192, 4096, False), (32, 4096, 5120, True),
    (32, 8192, 5120, False), (8, 16384, 4096, False), (16, 2048, 8192, True), (16, 2048, 16384, False),
    (17, 128, 8192, False), (32, 32768, 1024, True), (1, 248320, 1024, True), (33, 8192, 5120, True),
    (1024, 4096, 256, False), (1023, 4096, 256, True)])
def test_rule(rows, N, K, direct):
    assert (_form(torch.randn(rows, K), N) == _lib.VNX_F32) == direct


def test_rows_the_kernel_cannot_read_in_place():
    x = torch.randn(4, 260)
    assert _form(x[:, :256], 64) == _lib.VNX_F32
    assert _form(x[:, 1:257], 64) == _lib.VNX_F16             # off a 16-byte boundary
    assert _form(torch.randn(4, 261)[:, :256], 64) == _lib.VNX_F16
    assert _form(torch.randn(256, 4).t(), 64) == _lib.VNX_F16
    assert _form(torch.randn(1, 256).expand(4, 256), 64) == _lib.VNX_F16
    assert _form(x[:, :256].half(), 64) == _form(x[:, :256].double(), 64) == _lib.VNX_F16
