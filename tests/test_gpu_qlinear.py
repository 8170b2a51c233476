"""GPU parity of the quantized products of any row count (vnx_linear_w4 / _w8;
the tiled GEMM from 33 rows on) against fp64.

Bar: |y - ref| <= RTOL * sum_k |x_k w_k| + one fp32 rounding, ref the fp64
product of the fp16 activations and the exact q * s.  The fp32 sums run over
at most 128 products, then over chunks of 128 in three levels: a few roundings
of 2^-24 of the running sums, well inside RTOL = 2^-20."""
import pytest
import torch

from versenext_amd import _lib
from versenext_amd import quant as VQ

pytestmark = pytest.mark.gpu

RTOL = 2.0 ** -20


def _layer(hip, N, K, qtype, seed, bias=False):
    g = torch.Generator(device=hip.torch_device).manual_seed(seed)
    w = torch.randn((N, K), generator=g, device=hip.torch_device) * 0.02
    b = torch.randn(N, generator=g, device=hip.torch_device) if bias else None
    return VQ.QuantizedLinear(w, b, qtype, "rocm"), g


def _check(lin, x, y):
    w, x = lin.dequantize().double(), x.half().double().reshape(-1, lin.in_features)
    y = y.double().reshape(-1, lin.out_features)
    ref, mag = x @ w.t().contiguous(), x.abs() @ w.abs().t().contiguous()
    if lin.bias is not None:
        ref = ref + lin.bias.double()
    err = (y - ref).abs()
    assert bool((err <= RTOL * mag + 2.0 ** -23 * ref.abs() + 1e-30).all()), float((err / (mag + 1e-30)).max())


# 32 | 33 rows (the narrow kernels' last, the GEMM's first), remainders of the
# row and column tiles, one chunk and odd chunk counts, each tile shape (64 x
# 128, 32 x 128, 32 x 64, 32 x 32), 64 | 65 rows of an LM head
@pytest.mark.parametrize("rows,N,K", [
    (1, 130, 128), (32, 130, 384), (33, 130, 384), (33, 31, 128), (100, 300, 640), (257, 2049, 256),
    (512, 1000, 1152), (1000, 2080, 384), (1024, 4097, 256), (64, 33000, 128), (65, 33000, 128), (40, 8192, 640)])
@pytest.mark.parametrize("qtype", ["int8", "int4", "int4_g128"])
def test_rows(hip, rows, N, K, qtype):
    print("qlinear", rows, N, K, qtype, flush=True)
    lin, g = _layer(hip, N, K, qtype, seed=rows + N + K)
    x = torch.randn((rows, K), generator=g, device=hip.torch_device)
    y = lin(x)
    assert y.shape == (rows, N) and y.dtype == torch.float32
    _check(lin, x, y)
    assert torch.equal(y, lin(x.half()))                    # fp32 activations round as a cast does


@pytest.mark.parametrize("rows,N,K", [(5, 130, 256), (96, 130, 256), (24, 32800, 512), (70, 4096, 128)])
@pytest.mark.parametrize("qtype", ["int8", "int4", "int4_g128"])
def test_bias_strides_and_special_values(hip, rows, N, K, qtype):
    lin, g = _layer(hip, N, K, qtype, seed=K, bias=True)
    x = torch.randn((rows, K), generator=g, device=hip.torch_device)
    y = lin(x)
    _check(lin, x, y)
    plain = VQ.QuantizedLinear.forward
    b, lin.bias = lin.bias, None
    assert torch.equal(y, plain(lin, x) + b)                # one rounding, as a separate add
    wide = torch.randn((rows, K + 4), generator=g, device=hip.torch_device)
    assert torch.equal(lin(wide[:, :K]), lin(wide[:, :K].contiguous()))       # strided fp32 rows
    odd = torch.randn((rows, K + 1), generator=g, device=hip.torch_device)
    assert torch.equal(lin(odd[:, 1:]), lin(odd[:, 1:].contiguous()))         # rows off a 16-byte boundary
    x[0, 3], x[rows - 1, 0], x[rows // 2, 7] = float("inf"), 1e30, float("nan")
    torch.testing.assert_close(lin(x), lin(x.half()), rtol=0, atol=0, equal_nan=True)
    assert bool(torch.isnan(lin(x)[rows // 2]).all())


def test_refusals(hip):
    lin, _ = _layer(hip, 64, 128, "int8", seed=1)
    with pytest.raises(ValueError):
        lin(torch.zeros((3, 100), device=hip.torch_device))
    with pytest.raises(ValueError):
        hip.gemv_w8(torch.zeros((3, 128)), lin.wq, lin.scale, bias=torch.zeros(63))
    L = hip._L
    assert L.vnx_linear_w8(lin.wq.data_ptr(), _lib.VNX_BF16, 128, lin.wq.data_ptr(), 128, lin.scale.data_ptr(), 1, 64, 128,
                           None, lin.scale.data_ptr(), 64, None) == _lib.VNX_ERR_UNSUPPORTED


@pytest.mark.parametrize("rows", [3, 40])
def test_lazily_negated_operands(hip, rows):
    """The imaginary part of a conjugate is a view whose memory holds the
    other sign: the product and the bias are those of its values."""
    lin, g = _layer(hip, 128, 256, "int8", seed=rows, bias=True)
    z = torch.complex(torch.randn((256, rows), generator=g, device=hip.torch_device),
                      torch.randn((256, rows), generator=g, device=hip.torch_device))
    planes = torch.stack([z.real.t(), z.imag.t()]).contiguous()
    x = torch.view_as_complex(planes.permute(1, 2, 0).contiguous()).conj().imag
    assert x.is_neg() and torch.equal(lin(x), lin(x.resolve_neg().contiguous()))
    neg = torch._neg_view(planes[0].contiguous())          # unit strides: the form that is read in place
    assert neg.is_neg() and torch.equal(lin(neg), lin(neg.resolve_neg()))
    want = lin(planes[0]) - lin.bias - lin.bias
    lin.bias = torch._neg_view(lin.bias)
    torch.testing.assert_close(lin(planes[0]), want, rtol=1e-5, atol=1e-5)


def test_the_bias_of_a_user(hip):
    """A bias set on the layer keeps PyTorch's rules: its type promotes, its
    tangent and its batching pass through, another device is refused."""
    lin, g = _layer(hip, 128, 256, "int4_g128", seed=5, bias=True)
    x = torch.randn((5, 256), generator=g, device=hip.torch_device)
    b, lin.bias = lin.bias, None
    y = lin(x)
    lin.bias = b.double()
    assert lin(x).dtype == torch.float64 and torch.equal(lin(x), y + b.double())
    lin.bias = b.half()
    assert torch.equal(lin(x), y + b.half())
    lin.bias = b.cpu()
    with pytest.raises(RuntimeError):
        lin(x)
    import torch.autograd.forward_ad as fwd

    with fwd.dual_level():
        lin.bias = fwd.make_dual(b, torch.ones_like(b))
        out = fwd.unpack_dual(lin(x))
        assert torch.equal(out.primal, y + b) and torch.equal(out.tangent, torch.ones_like(y))

    def call(v):
        lin.bias = v
        return lin(x)

    bs = torch.stack([b, 2 * b])
    assert torch.equal(torch.func.vmap(call)(bs), torch.stack([y + b, y + 2 * b]))
    lin.bias = None


@pytest.mark.parametrize("rows,N,K", [(3, 32905, 1024), (30, 32905, 1024), (16, 40001, 512), (45, 33000, 512)])
def test_head_with_bias(hip, rows, N, K):
    """The streaming kernel of a head's many weight rows: the bias travels with
    the tiles' loads, fp16 and fp32 activations alike."""
    lin, g = _layer(hip, N, K, "int4_g128", seed=rows, bias=True)
    x = torch.randn((rows, K), generator=g, device=hip.torch_device)
    y = lin(x)
    _check(lin, x, y)
    b, lin.bias = lin.bias, None
    assert torch.equal(y, lin(x) + b) and torch.equal(lin(x), lin(x.half()))
    lin.bias = b
    assert torch.equal(y, lin(x.half()))
