"""GPU parity of the prefill-size GEMM (vnx_gemm_bf16 / _residual past 2,048
output tiles) and of the routed products of any row count (vnx_mod_lists,
vnx_expert_gemm_bf16_rows), against the fp64 products of the same bf16 inputs.

Bars as in tests/test_gpu_gemm.py: RTOL * sum_k |x_k w_k| per element plus one
rounding of the output type; SwiGLU's bound is propagated through silu(g) * u;
the residual form adds one fp32 rounding of the result.  Row lists are exact."""
import ctypes

import pytest
import torch

from versenext_amd import _lib

pytestmark = pytest.mark.gpu

RTOL = 1e-5
ROUND = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}
TINY = 2.0 ** -25                        # half the spacing of fp16's subnormals
P = lambda t: ctypes.c_void_p(t.data_ptr()) if t is not None else None


def _st():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _pack(w):
    L = _lib.lib()
    E, N, K = w.shape
    out = torch.empty((E, L.vnx_pack_bf16_size(N, K) // 2), dtype=torch.bfloat16, device=w.device)
    for z in range(E):
        _lib.check(L.vnx_pack_bf16(P(w[z]), K, N, K, P(out[z]), _st()))
    return out


def _inputs(hip, M, N, K, E, seed):
    g = torch.Generator(device=hip.torch_device).manual_seed(seed)
    x = torch.randn((M, K), generator=g, device=hip.torch_device).to(torch.bfloat16)
    w = (torch.randn((E, N, K), generator=g, device=hip.torch_device) * 0.05).to(torch.bfloat16)
    return x, w


def _check(y, x, w, epi, cw=None):
    """y (rows, cols) against x (rows, K) . w (N, K)^T on the GPU in fp64."""
    x, w = x.double(), w.double()
    acc, mag = x @ w.t().contiguous(), x.abs() @ w.abs().t().contiguous()
    if epi:
        blk = torch.arange(w.shape[0], device=w.device).view(-1, 32)
        gi, ui = blk[:, :16].reshape(-1), blk[:, 16:].reshape(-1)
        g, u = acc[:, gi], acc[:, ui]
        silu = g * torch.sigmoid(g)
        c = 1.0 if cw is None else cw.double()[:, None]
        ref = c * silu * u
        bound = c * RTOL * (1.1 * mag[:, gi] * u.abs() + silu.abs() * mag[:, ui])
    else:
        ref, bound = acc, RTOL * mag
    err = (y.double() - ref).abs()
    assert bool((err <= bound + ROUND[y.dtype] * ref.abs() + TINY).all()), float((err / (bound + 1e-30)).max())


# the three tile shapes (128 x 256, 64 x 256, 64 x 128), remainders of rows,
# columns (element stores past N % 32) and chunks (odd and a single one), the
# line of the dispatch (2,048 tiles) from both sides, one row tile of a W past
# 64 MB (read past the caches)
@pytest.mark.parametrize("M,N,K,epi,dtype", [
    (4099, 2080, 192, 0, torch.bfloat16), (16384, 1024, 64, 1, torch.bfloat16),
    (2048, 2048, 128, 0, torch.float32), (2017, 2080, 320, 1, torch.float16), (1000, 2053, 64, 0, torch.bfloat16),
    (1030, 1985, 448, 0, torch.float32), (1024, 2048, 1024, 0, torch.bfloat16), (1024, 2016, 1024, 0, torch.bfloat16),
    (97, 131105, 320, 0, torch.float32), (128, 131072, 320, 0, torch.bfloat16)])
def test_wide_gemm(hip, M, N, K, epi, dtype):
    print("wide gemm", M, N, K, epi, dtype, flush=True)
    x, w = _inputs(hip, M, N, K, 1, seed=M + N)
    nc = N // 2 if epi else N
    ldy = (nc + 7) // 8 * 8 + 8
    y = torch.full((M + 1, ldy), 7.0, dtype=dtype, device=hip.torch_device)
    _lib.check(hip._L.vnx_gemm_bf16(P(x), K, 0, P(_pack(w)), 0, M, N, K, 1, epi, None, 0, P(y), _lib.DTYPE_CODES[dtype],
                                    ldy, 0, _st()))
    _check(y[:M, :nc], x, w[0], epi)
    assert bool((y[M] == 7).all()) and bool((y[:, nc:] == 7).all())         # nothing past the result


@pytest.mark.parametrize("M,N,K", [(2048, 1024, 192), (1016, 2085, 64), (8200, 1024, 128)])
def test_wide_residual(hip, M, N, K):
    x, w = _inputs(hip, M, N, K, 1, seed=K)
    ldr = (N + 7) // 8 * 8
    res = torch.randn((M, ldr), device=hip.torch_device)
    old = res.clone()
    _lib.check(hip._L.vnx_gemm_bf16_residual(P(x), K, P(_pack(w)), M, N, K, P(res), ldr, _st()))
    xd, wd = x.double(), w[0].double()
    ref = old[:, :N].double() + xd @ wd.t().contiguous()
    tol = RTOL * (xd.abs() @ wd.abs().t().contiguous()) + 2.0 ** -24 * ref.abs()
    assert bool(((res[:, :N].double() - ref).abs() <= tol).all()) and torch.equal(res[:, N:], old[:, N:])


def _routing(hip, M, E, kind):
    g = torch.Generator().manual_seed(M + E)
    comb = torch.rand((M, E), generator=g) + 0.05
    if kind == "half":
        comb[torch.rand((M, E), generator=g) < 0.5] = 0.0
    elif kind == "skewed":                 # all rows to expert 1, none to expert 0, one to expert 2
        comb[:, 0] = 0.0
        comb[:, 2:] = 0.0
        comb[M - 1, 2] = 0.25
    else:
        comb.zero_()
    return comb.to(hip.torch_device)


@pytest.mark.parametrize("M,N,K,E,kind,epi,dtype", [
    (2048, 5376, 1024, 16, "half", 1, torch.bfloat16), (700, 512, 192, 16, "half", 0, torch.bfloat16),
    (257, 96, 64, 3, "skewed", 1, torch.float32), (3000, 1024, 128, 5, "skewed", 0, torch.float16),
    (300, 64, 128, 4, "none", 0, torch.float32), (1, 40, 64, 2, "half", 0, torch.float32)])
def test_routed_rows(hip, M, N, K, E, kind, epi, dtype):
    print("routed rows", M, N, K, E, kind, epi, dtype, flush=True)
    dev, L = hip.torch_device, hip._L
    x, w = _inputs(hip, M, N, K, E, seed=M + K)
    comb = _routing(hip, M, E, kind)
    rows = torch.full((E, M), -7, dtype=torch.int32, device=dev)
    counts = torch.full((E,), -7, dtype=torch.int32, device=dev)
    slots = torch.full((M, E), -7, dtype=torch.int32, device=dev)
    _lib.check(L.vnx_mod_lists(P(comb), E, M, E, P(rows), P(counts), P(slots), _st()))
    ref = [torch.nonzero(comb[:, z] != 0).flatten() for z in range(E)]
    assert counts.tolist() == [t.numel() for t in ref]
    want = torch.full((M, E), -1, dtype=torch.int32, device=dev)
    for z, t in enumerate(ref):
        assert torch.equal(rows[z, :t.numel()].long(), t)
        want[t, z] = torch.arange(t.numel(), dtype=torch.int32, device=dev)
    assert torch.equal(slots, want)
    total, wp, nc = int(counts.sum()), _pack(w), N // 2 if epi else N
    for bound in (0, total):
        y = torch.full((E, M, nc), 9.0, dtype=dtype, device=dev)
        _lib.check(L.vnx_expert_gemm_bf16_rows(P(x), K, 0, P(wp), wp.stride(0), M, N, K, E, epi, P(comb) if epi else None,
                                               E, P(rows), P(counts), bound, P(y), _lib.DTYPE_CODES[dtype], nc, M * nc,
                                               _st()))
        for z, t in enumerate(ref):
            _check(y[z, :t.numel()], x[t], w[z], epi, comb[t, z] if epi else None)
            assert bool((y[z, t.numel():] == 9).all())


@pytest.mark.parametrize("M,N,K,E", [(2048, 5376, 128, 16), (1024, 512, 192, 16), (300, 96, 64, 3)])
def test_routed_rows_past_the_callers_bound(hip, M, N, K, E):
    """total_rows below the counts' sum (rows whose router logits are NaN
    select every expert): every listed row is computed all the same."""
    print("routed rows past the bound", M, N, K, E, flush=True)
    dev, L = hip.torch_device, hip._L
    x, w = _inputs(hip, M, N, K, E, seed=M + K)
    comb = torch.full((M, E), float("nan"), device=dev)
    comb[M // 2:] = _routing(hip, M, E, "half")[M // 2:]
    rows = torch.empty((E, M), dtype=torch.int32, device=dev)
    counts = torch.empty((E,), dtype=torch.int32, device=dev)
    slots = torch.empty((M, E), dtype=torch.int32, device=dev)
    _lib.check(L.vnx_mod_lists(P(comb), E, M, E, P(rows), P(counts), P(slots), _st()))
    wp, n = _pack(w), counts.tolist()
    assert min(n) >= M // 2                                # a NaN weight is not 0: the row is on every list
    for bound in (M * E // 2, 1):
        y = torch.full((E, M, N), 9.0, dtype=torch.bfloat16, device=dev)
        _lib.check(L.vnx_expert_gemm_bf16_rows(P(x), K, 0, P(wp), wp.stride(0), M, N, K, E, 0, None, E, P(rows), P(counts),
                                               bound, P(y), _lib.DTYPE_CODES[torch.bfloat16], N, M * N, _st()))
        for z in range(E):
            _check(y[z, :n[z]], x[rows[z, :n[z]].long()], w[z], 0)
            assert bool((y[z, n[z]:] == 9).all())


# a head's columns: one and two row tiles with both tile shapes, a W that the
# last-level cache holds beside the logits, one that it does not, and one that
# streams (fp32 and 16-bit logits past the caches each, and not)
@pytest.mark.parametrize("M,N,K,dtype", [
    (224, 64000, 64, torch.bfloat16), (150, 64000, 64, torch.float32), (129, 100352, 64, torch.float16),
    (256, 32768, 64, torch.float32), (131, 65536, 1984, torch.bfloat16), (97, 131104, 1088, torch.float32),
    (128, 131104, 1088, torch.bfloat16), (33, 131111, 1088, torch.bfloat16)])
def test_head_gemm(hip, M, N, K, dtype):
    print("head gemm", M, N, K, dtype, flush=True)
    x, w = _inputs(hip, M, N, K, 1, seed=M + K)
    ldy = (N + 7) // 8 * 8 + 8
    y = torch.full((M + 1, ldy), 7.0, dtype=dtype, device=hip.torch_device)
    _lib.check(hip._L.vnx_gemm_bf16(P(x), K, 0, P(_pack(w)), 0, M, N, K, 1, 0, None, 0, P(y), _lib.DTYPE_CODES[dtype],
                                    ldy, 0, _st()))
    for n in range(0, N, 16384):
        _check(y[:M, n:min(n + 16384, N)], x, w[0][n:n + 16384], 0)
    assert bool((y[M] == 7).all()) and bool((y[:, N:] == 7).all())
