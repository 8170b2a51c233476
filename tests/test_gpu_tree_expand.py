"""vnx_tree_expand against the oracle and against the row top-b it replaces
(vnx_row_topk on every row, then each node's rank), and tree attention with the
ancestor words passed by value against the same words on the device: all bit
for bit."""
import numpy as np
import pytest
import torch

from oracle import tree as OT
from versenext_amd import tree as T

pytestmark = pytest.mark.gpu


def _by_topk(hip, draft, par):
    rows, rank, seen = np.where(par < 0, 0, par + 1), np.zeros(par.size, np.int64), {}
    for i, p in enumerate(par):
        rank[i] = seen.get(int(p), 0)
        seen[int(p)] = rank[i] + 1
    ids, _ = hip.topk(draft, int(rank.max()) + 1)
    return ids[:, torch.from_numpy(rows).to(ids.device), torch.from_numpy(rank).to(ids.device)]


# a chain, a wide root (16 children, the most), the (4, 3, 2) tree, parents out
# of order with interleaved siblings, 64 nodes; rows of a single short chunk,
# of odd lengths, of one element past a chunk and longer than 64 chunks
@pytest.mark.parametrize("par", [T.chain(6), [-1] * 16, T.tree_from_branching((4, 3, 2)),
                                 [-1, 0, -1, 0, 2, 1, 0, 2, 4], T.tree_from_branching((4, 3, 4))[:64], T.chain(64)],
                         ids=["chain", "wide", "432", "mixed", "large", "long"])
@pytest.mark.parametrize("V,dtype", [(17, torch.float32), (8193, torch.bfloat16), (50001, torch.float32),
                                     (530000, torch.bfloat16)])
def test_expand_equals_topk(hip, par, V, dtype):
    par = np.asarray(par, np.int32)
    B, R = 2, par.size + 1
    print("expand", par.size, V, dtype, flush=True)
    g = torch.Generator(device=hip.torch_device).manual_seed(V + R)
    buf = torch.randn((B, R + 2, (V + 15) // 8 * 8), generator=g, device=hip.torch_device).to(dtype)
    draft = buf[:, 1:R + 1, :V]                          # a strided view: no copy
    draft[0, 0, :min(V, 40)] = 9.0                       # ties go to the lower id
    draft[1, 0, 3], draft[1, R - 1, 5] = float("nan"), float("-inf")
    want = _by_topk(hip, draft, par)
    assert torch.equal(hip.expand_tree(draft, par), want)
    assert torch.equal(hip.expand_tree(draft.float().cpu().numpy(), par), want)


def test_expand_refusals(hip):
    d = torch.zeros((1, 3, 32), device=hip.torch_device)
    with pytest.raises(IndexError):
        hip.expand_tree(d, T.chain(4))                   # row 3 of 3
    with pytest.raises(ValueError):
        hip.expand_tree(torch.zeros((1, 18, 32)), [-1] * 17)
    with pytest.raises(ValueError):
        hip.expand_tree(d, [0])
    assert hip.expand_tree(d[:0], T.chain(2)).shape == (0, 2)


@pytest.mark.parametrize("N,Tp,d,window,alibi", [(1, 0, 64, 0, False), (40, 2048, 64, 0, False), (64, 100, 64, 80, False),
                                                 (7, 617, 128, 0, False), (40, 300, 64, 0, True), (63, 33, 128, 64, True)])
def test_ancestor_words_by_value(hip, N, Tp, d, window, alibi):
    print("words by value", N, Tp, d, window, alibi, flush=True)
    B, H, Hkv = 3, 8, 4
    par = np.concatenate([[-1], np.random.default_rng(N).integers(-1, np.arange(1, N))]) if N > 1 else np.array([-1])
    words = T.ancestor_words(par)
    g = torch.Generator(device=hip.torch_device).manual_seed(N + Tp)
    r = lambda *s: torch.randn(s, generator=g, device=hip.torch_device).to(torch.bfloat16)
    kc, vc = (r(B, Hkv, Tp, d), r(B, Hkv, Tp, d)) if Tp else (None, None)
    kw = dict(window=window)
    if alibi:
        kw.update(alibi_slopes=torch.rand(H, generator=g, device=hip.torch_device), gates=torch.tensor([0.5, 0.2, 0.9]))
    args = (r(B, H, N, d), kc, vc, r(B, Hkv, N, d), r(B, Hkv, N, d))
    assert torch.equal(hip.tree_attention(*args, words, **kw), hip.tree_attention(*args, np.tile(words, (B, 1)), **kw))


@pytest.mark.parametrize("par", [T.chain(6), [-1] * 16, T.tree_from_branching((4, 3, 2)), [-1, 0, -1, 0, 2, 1, 0, 2, 4]],
                         ids=["chain", "wide", "432", "mixed"])
@pytest.mark.parametrize("V,dtype", [(17, torch.float32), (8193, torch.bfloat16), (20011, torch.float32)])
def test_expand_equals_the_oracle(hip, par, V, dtype):
    par = np.asarray(par, np.int32)
    B, R = 3, par.size + 1
    print("expand against the oracle", par.size, V, dtype, flush=True)
    g = torch.Generator().manual_seed(V + R)
    draft = torch.randn((B, R, V), generator=g).to(dtype)
    draft[0, 0, V // 2:] = 9.0                           # ties go to the lower id
    draft[1, :, 1] = float("-inf")
    draft[1, 0, 3], draft[2, R // 2, 5], draft[2, 0, 7] = float("nan"), float("nan"), float("inf")
    got = hip.expand_tree(draft, par)
    assert np.array_equal(got.cpu().numpy(), OT.expand_tree(draft.float().numpy(), par))
