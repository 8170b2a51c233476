"""GPU parity of the row norm around its two widths (4 and 16 columns per
thread, split at 1,024 columns) and of the routing weights with equal logits.

Norm: the fp32 sum of D squares in partial sums of at most 16 terms and a
butterfly is within 32 * 2^-24 of the exact sum, the result within half of
that and four roundings: 20 * 2^-24 relative, plus the output's rounding.
Routing: the selected set is exact; a weight has at most E + P exps and as many
roundings in its two sums, so 64 * 2^-24."""
import ctypes

import pytest
import torch

from versenext_amd import _lib

pytestmark = pytest.mark.gpu

P = lambda t: ctypes.c_void_p(t.data_ptr()) if t is not None else None


def _st():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


@pytest.mark.parametrize("D", [1, 255, 257, 1023, 1024, 1025, 4095])
@pytest.mark.parametrize("embed", [False, True])
def test_norm_widths(hip, D, embed):
    print("norm", D, embed, flush=True)
    M, V, eps, scale = 9, 11, 1e-6, 1.5
    g = torch.Generator(device=hip.torch_device).manual_seed(D)
    rnd = lambda *s: torch.randn(s, generator=g, device=hip.torch_device)
    w = rnd(D)
    xo, y = torch.full((M, D + 3), 7.0, device=hip.torch_device), torch.full((M, D + 5), 7.0, device=hip.torch_device)
    if embed:
        emb = rnd(V, D).to(torch.bfloat16)
        ids = torch.randint(-1, V + 1, (M,), generator=g, device=hip.torch_device)     # clamped into the table
        _lib.check(hip._L.vnx_embed_rmsnorm(P(ids), P(emb), _lib.VNX_BF16, D, V, scale, P(w), eps, M, D, P(xo), D + 3,
                                            P(y), _lib.VNX_F32, D + 5, _st()))
        s = emb[ids.clamp(0, V - 1)].float() * scale
    else:
        x, res = rnd(M, D), rnd(M, D).to(torch.float16)
        _lib.check(hip._L.vnx_rmsnorm(P(x), D, P(res), _lib.DTYPE_CODES[torch.float16], D, P(w), eps, M, D, P(xo),
                                      D + 3, P(y), _lib.VNX_F32, D + 5, _st()))
        s = x + res.float()
    assert torch.equal(xo[:, :D], s) and bool((xo[:, D:] == 7).all()) and bool((y[:, D:] == 7).all())
    sd = s.double()
    ref = sd / torch.sqrt((sd * sd).mean(dim=1, keepdim=True) + eps) * w.double()
    assert bool(((y[:, :D].double() - ref).abs() <= 21 * 2.0 ** -24 * ref.abs()).all())


@pytest.mark.parametrize("NP,NE,topk", [(4, 4, 2), (1, 16, 16), (2, 8, 5), (8, 7, 1), (3, 1, 1)])
def test_route_with_ties(hip, NP, NE, topk):
    M = 65
    g = torch.Generator().manual_seed(NP * 100 + NE)
    lg = torch.randint(-2, 3, (M, NP + NP * NE), generator=g).float() * 0.75           # mostly equal logits
    dev = lg.to(hip.torch_device)
    comb = torch.full((M, NP * NE + 1), 7.0, device=hip.torch_device)
    _lib.check(hip._L.vnx_mod_route(P(dev), lg.shape[1], M, NP, NE, topk, P(comb), NP * NE + 1, _st()))
    pw = torch.softmax(lg[:, :NP].double(), dim=-1)
    ref = torch.zeros((M, NP * NE), dtype=torch.float64)
    for p in range(NP):
        le = lg[:, NP + p * NE:NP + (p + 1) * NE].double()
        idx = torch.argsort(-le, dim=-1, stable=True)[:, :topk]
        ref[:, p * NE:(p + 1) * NE].scatter_(1, idx, torch.softmax(torch.gather(le, 1, idx), dim=-1) * pw[:, p:p + 1])
    got = comb.cpu()
    assert bool((got[:, -1] == 7).all()) and bool(((got[:, :-1] > 0) == (ref > 0)).all())
    assert bool(((got[:, :-1].double() - ref).abs() <= 64 * 2.0 ** -24 * ref).all())
