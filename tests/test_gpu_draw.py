"""GPU parity of the draws' inverse-CDF walk and of the nucleus passes where
their loops can go wrong: rows shorter than a sub-block, partial last
sub-blocks, odd numbers of sub-blocks per wave, rows without residual mass
(recomputed by the drawing workgroup), arrival counters packed for want of
room, nucleus cuts inside long runs of ties, rows that nothing is drawn from.

Bar as in tests/test_gpu_spec_accept.py and tests/test_gpu_sampler.py: ids,
accept_len and the nucleus bit-exact against the CPU oracle, save rows that a
flag marks on either side."""
import ctypes

import numpy as np
import pytest
import torch

from oracle.speculative import spec_accept
from spec_inputs import make_inputs
from test_gpu_sampler import _check
from test_gpu_spec_accept import compare, run_gpu
from versenext_amd import _lib

pytestmark = pytest.mark.gpu


# sub-blocks are 256 fp32 / 512 bf16 elements; four waves take them in turn
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V", [5, 255, 256, 517, 1024, 2304, 9 * 512 + 1, 70003])
def test_walk_edges(hip, V, dtype):
    print("walk", V, dtype, flush=True)
    B, k, T = 6, 3, 0.9
    tgt, dft, ids, u = make_inputs(B, k, V, T, seed_t=V, seed_d=V + 1, seed_x=V + 2, seed_u=V + 3)
    dft[:3] = tgt[:3, :k]              # p == q ...
    ids[0, 0] = ids[1, 1] = -1         # ... rejected: no residual mass
    u[4, k], u[5, k] = 0.0, np.float32(1.0 - 2.0 ** -24)
    if dtype == torch.bfloat16:
        tgt, dft = (torch.from_numpy(a).to(dtype).float().numpy() for a in (tgt, dft))
    g, o = run_gpu(hip, tgt, dft, ids, u, T, dtype=dtype), spec_accept(tgt, dft, ids, u, T)
    _, bad, _ = compare(g, o, k)
    assert not bad, bad
    assert np.array_equal(g["flags"] & 8, o["flags"] & 8)


def test_packed_counters(hip):
    """The fixed scratch near its limit: no room for a line per counter."""
    B, k, V, T = 100000, 1, 7, 0.8
    g = torch.Generator(device=hip.torch_device).manual_seed(3)
    tgt = torch.randn((B, k + 1, 8), generator=g, device=hip.torch_device)
    dft = torch.randn((B, k, 8), generator=g, device=hip.torch_device)
    ids = torch.randint(0, V, (B, k), generator=g, device=hip.torch_device)
    u = torch.rand((B, k + 1), generator=g, device=hip.torch_device)
    L, P = hip._L, lambda t: ctypes.c_void_p(t.data_ptr())
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    need = L.vnx_spec_accept_workspace(B, k, V)
    assert need > L.vnx_spec_accept_noalloc_max_bytes()
    outs = []
    for packed in (False, True):
        acc = torch.full((B,), -7, dtype=torch.int32, device=hip.torch_device)
        out = torch.full((B, k + 1), -7, dtype=torch.int64, device=hip.torch_device)
        args = (P(tgt), P(dft), _lib.DTYPE_CODES[torch.float32], B, k, V, 8, 16, 8, 8, P(ids), P(u), T, None, None,
                P(acc), P(out), None, None, None)
        if packed:
            _lib.check(L.vnx_spec_accept_noalloc(*args, st))
        else:
            ws = torch.empty((need,), dtype=torch.uint8, device=hip.torch_device)
            _lib.check(L.vnx_spec_accept(*args, P(ws), need, st))
        outs.append((acc, out))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
    assert int(outs[0][1].min()) >= -1 and int(outs[0][1].max()) < V


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V", [3, 256, 1025, 33 * 512 + 8, 151936])
def test_nucleus_edges(hip, V, dtype):
    """Rows: one value (every cut is a tie), a few values, spread values, one
    dominant value, NaN, +inf, all -inf, all but one -inf."""
    rng = np.random.default_rng(V)
    x = rng.normal(0, 3.0, (8, V)).astype(np.float32)
    x[0] = 0.5
    x[1] = np.round(x[1])
    x[3, V // 2] = 60.0
    x[4, V - 1] = np.nan
    x[5, [0, V // 2]] = np.inf
    x[6] = -np.inf
    x[7] = -np.inf
    x[7, V // 3] = -2.0
    x = torch.from_numpy(x).to(dtype).float().numpy()
    u = rng.random(8).astype(np.float32)
    for T, p in ((1.0, 0.9), (0.7, 0.35), (1.0, 1e-4), (1.0, 0.99999), (0.8, 1.0), (0.0, 1.0)):
        print("nucleus", V, dtype, T, p, flush=True)
        _, _, bad = _check(hip, x, T, 0, p, u, dtype=dtype)
        assert bad <= 1, (T, p)
