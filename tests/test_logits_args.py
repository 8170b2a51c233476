"""What CometSparkGPU.logits hands its bf16 head: the kernel is given rows of the
head's own width and a destination that it can write, and nothing else reaches
it (no GPU: the entry is replaced by one that notes its arguments)."""
import types

import pytest
import torch

from versenext_amd import _lib
from versenext_amd.model import CometSparkGPU

D, V = 64, 96


def _model():
    calls = []

    def gemm(x, ldx, sxb, w, swb, M, N, K, batch, epi, comb, ldc, y, y_dtype, ldy, syb, stream):
        calls.append(dict(M=M, N=N, K=K, y=y, y_dtype=y_dtype, ldy=ldy))
        return _lib.VNX_OK

    m = types.SimpleNamespace(cfg=types.SimpleNamespace(vocab_size=V, dim=D), head=None, dtype=torch.bfloat16,
                              dev=torch.device("cpu"), head_p=torch.zeros(V * D, dtype=torch.bfloat16),
                              head_w=torch.zeros((V, D), dtype=torch.bfloat16), _st=lambda: 0,
                              hip=types.SimpleNamespace(_L=types.SimpleNamespace(vnx_gemm_bf16=gemm)))
    return m, calls


@pytest.mark.parametrize("rows", [2, 300])
@pytest.mark.parametrize("width", [D // 2, D + 64])
def test_hidden_of_another_width_is_refused(rows, width):
    m, calls = _model()
    with pytest.raises(ValueError):
        CometSparkGPU.logits(m, torch.zeros((1, rows, width)))
    with pytest.raises(ValueError):
        CometSparkGPU.logits(m, torch.zeros((1, rows, width)), out=torch.zeros((1, rows, V)))
    assert not calls


def test_a_destination_the_kernel_can_write():
    for dtype in (torch.float32, torch.bfloat16):
        m, calls = _model()
        out = torch.zeros((2, 3, 2 * V), dtype=dtype)[..., :V]
        assert CometSparkGPU.logits(m, torch.zeros((2, 3, D)), out=out) is out
        assert calls == [dict(M=6, N=V, K=D, y=out.data_ptr(), y_dtype=_lib.DTYPE_CODES[dtype], ldy=2 * V)]
    m, calls = _model()
    assert CometSparkGPU.logits(m, torch.zeros((2, 3, D))).shape == (2, 3, V)


def _others(rows):
    """Destinations that have the right shape but not the kernel's form."""
    yield torch.zeros((V, rows)).t().view(1, rows, V)                                # columns a row apart
    yield torch.zeros((1, rows, 2 * V))[..., ::2]
    yield torch.zeros((1, rows, V), device="meta")                                   # memory of another device


@pytest.mark.parametrize("which", range(3))
def test_other_destinations_are_refused_or_copied_to(which):
    # up to 256 rows a destination without unit last stride is refused; longer
    # ones, and those of another device, receive a copy
    m, calls = _model()
    few, many = list(_others(4))[which], list(_others(300))[which]
    if which < 2:
        with pytest.raises(ValueError):
            CometSparkGPU.logits(m, torch.zeros((1, 4, D)), out=few)
        assert not calls
    assert CometSparkGPU.logits(m, torch.zeros((1, 300, D)), out=many) is many
    for c in calls:
        assert c["ldy"] == V and c["y"] != (many.data_ptr() if which < 2 else 0)


def test_a_half_precision_destination():
    m, calls = _model()
    out = torch.full((1, 4, V), 3.0, dtype=torch.float16)
    assert CometSparkGPU.logits(m, torch.zeros((1, 4, D)), out=out) is out
    assert all(c["y"] != out.data_ptr() for c in calls)
