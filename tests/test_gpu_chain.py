"""GPU parity of the chain attention kernel (vnx_chain_attn) against fp64.

Bar: |out - ref| <= RTOL * mag, mag = sum over the paths of gate * sum_j p_j
|v_j|, plus one rounding of the output type.  The kernel's errors are those
of vnx_tree_attn (tests/test_gpu_tree.py): fp32 sums of exact bf16 products,
exp2 on the transcendental unit, P as bf16 hi + lo (2^-17 relative); ALiBi
adds one fp32 rounding of a bias of up to ~1000 in the exp2 domain's scores
(2^-14 absolute in the exponent), so its bar is 2^-13."""
import ctypes

import numpy as np
import pytest
import torch

from versenext_amd import _lib

pytestmark = pytest.mark.gpu

RTOL = 2e-5
ROUND = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _args(q, kc, vc, out, Tp, tp, window, seg2, gates, slopes, amax):
    B, H, N, d = q.shape
    a = _lib.TreeAttnArgs()
    a.q = q.data_ptr(); a.q_strides[:] = list(q.stride()[:3])
    a.k_cache = kc.data_ptr(); a.v_cache = vc.data_ptr(); a.cache_strides[:] = list(kc.stride()[:3])
    a.out = out.data_ptr(); a.out_dtype = _lib.DTYPE_CODES[out.dtype]; a.out_strides[:] = list(out.stride()[:3])
    a.B, a.H, a.Hkv, a.Tp, a.N, a.d = B, H, kc.shape[1], Tp, N, d
    a.scale = 1.0 / np.sqrt(d)
    a.tp_batch = tp.data_ptr() if tp is not None else None
    a.window = window
    if seg2 is not None:
        a.k_seg2, a.v_seg2 = seg2[0].data_ptr(), seg2[1].data_ptr()
        a.seg2_strides[:] = [0 if seg2[0].shape[0] == 1 else seg2[0].stride(0)] + list(seg2[0].stride()[1:3])
        a.T2 = seg2[0].shape[2]
    a.gates = gates.data_ptr() if gates is not None else None
    if slopes is not None:
        a.alibi_slopes = slopes.data_ptr(); a.alibi_max_keys = amax
    return a


def _reference(q, kc, vc, Tp, tp, window, seg2, gates, slopes, amax):
    """fp64 on the CPU: (out, mag), both (B, H, N, d)."""
    q, kc, vc = (t.double().cpu() for t in (q, kc, vc))
    B, H, N, d = q.shape
    rep = H // kc.shape[1]
    g = gates.double().cpu() if gates is not None else torch.ones(3, dtype=torch.float64)
    out, mag = torch.zeros_like(q), torch.zeros_like(q)

    def add(b, s, v, gate):
        p = torch.softmax(s, -1)
        out[b] += gate * (p @ v)
        mag[b] += gate.abs() * (p @ v.abs())

    for b in range(B):
        t = Tp if tp is None else int(tp[b].clamp(0, Tp))
        k, v = kc[b, :, :t + N].repeat_interleave(rep, 0), vc[b, :, :t + N].repeat_interleave(rep, 0)
        s = q[b] @ k.transpose(-1, -2) / np.sqrt(d)
        dist = (t + torch.arange(N))[:, None] - torch.arange(t + N)[None]
        hide = dist < 0
        add(b, s.masked_fill(hide | (dist >= window) if window else hide, -np.inf), v,
            g[0] if gates is not None else torch.tensor(1.0, dtype=torch.float64))
        if seg2 is not None:
            z = 0 if seg2[0].shape[0] == 1 else b
            k2, v2 = (x[z].double().cpu().repeat_interleave(rep, 0) for x in seg2)
            add(b, q[b] @ k2.transpose(-1, -2) / np.sqrt(d), v2, g[1])
        if slopes is not None and t + N <= amax:
            bias = -slopes.double().cpu()[:, None, None] * dist.double()
            add(b, (s + bias).masked_fill(hide, -np.inf), v, g[2])
    return out, mag


# edges: one column, one short of / one past a 32-column wave, a 64- and a
# 128-column workgroup, windows shorter than a step and than N, prefixes that
# start off a 64-key step, heads that divide by 8 (XCD order) and do not, all
# three workgroup shapes (few, some and many tiles), three heads to a KV head
CASES = [
    dict(B=1, H=2, Hkv=1, d=64, N=1, tp=[0]),
    dict(B=2, H=4, Hkv=2, d=64, N=33, tp=[5, 63], window=7),
    dict(B=1, H=6, Hkv=2, d=64, N=43, tp=None, Tp=10, T2=5),
    dict(B=1, H=16, Hkv=8, d=64, N=65, tp=[0], window=1024, T2=128),
    dict(B=3, H=8, Hkv=8, d=64, N=200, tp=[0, 129, 70], window=64, T2=65, shared=False),
    dict(B=2, H=4, Hkv=2, d=64, N=131, tp=[0, 900], window=100, T2=3, amax=1024),
    dict(B=4, H=16, Hkv=8, d=64, N=512, tp=[0, 0, 0, 0], window=1024, T2=128, out=torch.bfloat16),
    dict(B=8, H=16, Hkv=8, d=64, N=1030, tp=[0, 1, 2, 3, 4, 5, 6, 7], window=1024, T2=128, out=torch.float16),
    dict(B=1, H=2, Hkv=1, d=128, N=129, tp=[31], window=50, T2=31, amax=4096),
    dict(B=8, H=16, Hkv=8, d=128, N=260, tp=[17] * 8, T2=64, out=torch.bfloat16),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"B{c['B']}H{c['H']}kv{c['Hkv']}d{c['d']}N{c['N']}")
def test_chain_attention(hip, case):
    c = dict(window=0, T2=0, amax=0, shared=True, out=torch.float32)
    c.update(case)
    B, H, Hkv, d, N = (c[x] for x in ("B", "H", "Hkv", "d", "N"))
    print("chain_attn", case, flush=True)
    dev = hip.torch_device
    g = torch.Generator().manual_seed(N * 131 + d)
    rnd = lambda *s: torch.randn(s, generator=g).to(torch.bfloat16).to(dev)
    Tp = c.get("Tp", max(c["tp"]) if c["tp"] else 0)
    tp = torch.tensor(c["tp"], dtype=torch.int32, device=dev) if c["tp"] else None
    q = rnd(B, N, H, d).transpose(1, 2)                     # heads strided, as a projection leaves them
    kc, vc = rnd(B, Hkv, Tp + N + 3, d), rnd(B, Hkv, Tp + N + 3, d)
    kc[:, :, Tp + N:] = float("nan")                        # rows past every sequence are never used
    vc[:, :, Tp + N:] = float("nan")
    z = 1 if c["shared"] else B
    seg2 = (rnd(z, Hkv, c["T2"], d), rnd(z, Hkv, c["T2"], d)) if c["T2"] else None
    slopes = torch.rand(H, generator=g).to(dev) if c["amax"] else None
    gates = torch.tensor([0.7, 0.4, 0.55], device=dev) if seg2 is not None or slopes is not None else None
    out = torch.full((B, N, H, d), float("nan"), dtype=c["out"], device=dev).transpose(1, 2)
    a = _args(q, kc, vc, out, Tp, tp, c["window"], seg2, gates, slopes, c["amax"])
    _lib.check(hip._L.vnx_chain_attn(ctypes.byref(a), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    ref, mag = _reference(q, kc, vc, Tp, tp, c["window"], seg2, gates, slopes, c["amax"])
    err = (out.double().cpu() - ref).abs()
    tol = (2.0 ** -13 if slopes is not None else RTOL) * mag + ROUND[c["out"]] * ref.abs()
    print(f"  worst err / mag {float((err / mag).max()):.2e}", flush=True)
    assert torch.isfinite(out).all() and bool((err <= tol).all())


def test_chain_attention_refusals(hip):
    dev = hip.torch_device
    q = torch.zeros((1, 2, 4, 64), dtype=torch.bfloat16, device=dev)
    kc = torch.zeros((1, 1, 8, 64), dtype=torch.bfloat16, device=dev)
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    call = lambda a: hip._L.vnx_chain_attn(ctypes.byref(a), st)
    make = lambda: _args(q, kc, kc, torch.empty_like(q), 4, None, 0, None, None, None, 0)
    assert call(make()) == _lib.VNX_OK
    for field, value, status in (("d", 32, _lib.VNX_ERR_UNSUPPORTED), ("N", 0, _lib.VNX_ERR_INVALID_ARG),
                                 ("f32_rows", 1, _lib.VNX_ERR_UNSUPPORTED), ("T2", 3, _lib.VNX_ERR_INVALID_ARG),
                                 ("k_tree", kc.data_ptr(), _lib.VNX_ERR_UNSUPPORTED),
                                 ("q", q.data_ptr() + 2, _lib.VNX_ERR_UNSUPPORTED), ("scale", 0.0, _lib.VNX_ERR_INVALID_ARG)):
        a = make()
        setattr(a, field, value)
        assert call(a) == status, field
