"""Infinities and NaN stay where the mathematics puts them.

A key that a query does not attend, a page that does not exist and a step that
a lane only pads its walk with must not touch the query's output; a key that it
does attend must show.  Every case compares with the same call on finite inputs
(bit for bit where nothing may change) or with the fp64 oracle's own infinities
and NaN."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import make_inputs, oracle_tree

pytestmark = pytest.mark.gpu
DEV = "cuda"


def say(*a):
    print(*a, flush=True)


@pytest.mark.parametrize("D,Hkv,b,md", [
    (64, 8, 4, 4),    # 4 heads per slot, 5 steps in chunks of 2: the last chunk holds a step without a key
    (64, 16, 4, 5),   # 2 heads per slot, 6 steps
    (128, 8, 4, 5),   # one step per chunk: only walks shorter than their wave's pad
    (32, 8, 3, 6),
])
def test_paged_heads_of_a_group_are_independent(D, Hkv, b, md):
    """An infinity or a NaN in one q head of a group leaves the others as they were."""
    from qattention_amd import _lib, ragged_attn as ra
    lens, Hq, ps = [2100, 1365], 32, 16
    Q, K, V, cu = make_inputs(lens, Hq, D, 9000 + D + Hkv, Hkv=Hkv)
    Kc, Vc, pt = ra.build_paged_kv(list(K.to(DEV).split(lens)), list(V.to(DEV).split(lens)), ps)
    pt = pt.clone()
    pt[1, 3] = -1  # a page missing from the second sequence
    pt = pt.to(DEV)
    call = lambda q: ra._paged_forward(q, Kc, Vc, pt, cu, b, md, max(lens), True, _lib.ALGO_GATHER)  # noqa: E731
    q = Q.to(DEV)
    say("paged group", D, Hkv, b, md)
    O, L = call(q)
    g = Hq // Hkv
    for bad in (float("inf"), float("nan")):
        for h in range(2):  # each group's first and second head
            q2 = q.clone()
            q2[:, h::g, 3] = bad
            O2, L2 = call(q2)
            keep = [i for i in range(Hq) if i % g != h]
            assert torch.equal(O2[:, keep], O[:, keep]) and torch.equal(L2[:, keep], L[:, keep]), (bad, h)


def _attends(cu, b, md, parents, node):
    """Tokens of the first sequence's batch row whose walk attends its node `node`."""
    from oracle import clib
    anc = (clib.ancestor_table_heap(cu.numpy(), b, md) if parents is None
           else clib.ancestor_table_parents(cu.numpy(), parents, md))
    first = np.zeros(anc.shape[0], dtype=bool)
    first[: int(cu[1])] = True
    return torch.from_numpy((anc == node).any(1) & first)


@pytest.mark.parametrize("walk", ["heap", "parents", "paged"])
@pytest.mark.parametrize("lens,Hq,Hkv,D", [
    ([2048, 30], 32, 8, 128),   # 4 heads per slot, one step per chunk
    ([2100, 30], 32, 16, 128),  # 2 heads per slot
    ([2100, 30], 32, 8, 64),    # 4 heads, two steps per chunk
    ([500], 32, 32, 128),       # one head, 16 lanes
    ([200], 32, 32, 64),        # one head, 8 lanes
    ([1500], 32, 32, 128),      # gather kernel
])
def test_nan_key_reaches_who_attends_it(lens, Hq, Hkv, D, walk):
    """NaN in a leaf's, an inner node's and a root's K row (of different kv heads):
    exactly the queries that attend the node become NaN, O and LSE."""
    from qattention_amd import _lib, ragged_attn as ra
    b, md = 4, 6
    Q, K, V, cu = make_inputs(lens, Hq, D, 9100 + D + Hkv, Hkv=Hkv)
    par = None
    if walk == "parents":
        par = np.concatenate([np.maximum(np.arange(n) - 1, 0) // b for n in lens]).astype(np.int32)
    nodes = [lens[0] - 1, 6, 0]
    K2 = K.clone()
    for h, node in enumerate(nodes):
        K2[node, h, 1] = float("nan")

    def call(k):
        q, k, v = Q.to(DEV), k.to(DEV), V.to(DEV)
        if walk == "heap":
            return ra._tree_forward(q, k, v, cu, b, md, max(lens), True, _lib.ALGO_GATHER)
        if walk == "parents":
            return ra.ragged_attention_with_parents(q, k, v, cu, torch.from_numpy(par).to(DEV), md, max(lens))
        Kc, Vc, pt = ra.build_paged_kv(list(k.split(lens)), list(v.split(lens)), 16)
        return ra._paged_forward(q, Kc, Vc, pt.to(DEV), cu, b, md, max(lens), True, _lib.ALGO_GATHER)

    say("nan key", walk, lens, Hq, Hkv, D)
    (O, L), (O2, L2) = call(K), call(K2)
    g = Hq // Hkv
    hit = torch.zeros(Q.shape[0], Hq, dtype=torch.bool)
    for h, node in enumerate(nodes):
        hit[:, h * g:(h + 1) * g] = _attends(cu, b, md, par, node)[:, None]
    hit = hit.to(DEV)
    assert torch.equal(torch.isnan(L2), hit)
    assert torch.equal(torch.isnan(O2).all(-1), hit) and torch.equal(torch.isnan(O2).any(-1), hit)
    assert torch.equal(O2[~hit], O[~hit]) and torch.equal(L2[~hit], L[~hit])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("N,Hq,Hkv,D", [
    (60, 16, 4, 128),   # one wave per query
    (60, 16, 4, 64),
    (600, 16, 4, 128),  # gather kernel
])
def test_nan_split_reaches_its_heads(N, Hq, Hkv, D, dtype):
    """NaN in every key of one of ten splits, in one key of another, or in a tree
    row: the kv head's queries (that attend it) become NaN, the others stay."""
    from qattention_amd import ragged_attn as ra
    b, md, L, ns = 3, 5, 640, 10
    Q, K, V, cu = make_inputs([N], Hq, D, 9200 + D + N, dtype=dtype, Hkv=Hkv)
    g = torch.Generator().manual_seed(9201)
    Kp, Vp = (torch.randn(1, L, Hkv, D, generator=g).to(dtype) for _ in range(2))
    call = lambda k, kp: ra.ragged_attention_prefix(  # noqa: E731
        *(x.to(DEV) for x in (Q, k, V, cu, kp, Vp)), b, md, max_seqlen=N, return_lse=True, num_splits=ns)
    say("nan split", N, Hq, Hkv, D, dtype)
    O, lse = call(K, Kp)
    K2, Kp2 = K.clone(), Kp.clone()
    Kp2[0, 64:128, 0, 1] = float("nan")
    Kp2[0, 600, 1, 1] = float("nan")
    K2[7, 2, 1] = float("nan")
    O2, lse2 = call(K2, Kp2)
    r = Hq // Hkv
    hit = torch.zeros(N, Hq, dtype=torch.bool)
    hit[:, :2 * r] = True
    hit[:, 2 * r:3 * r] = _attends(cu, b, md, None, 7)[:, None]
    hit = hit.to(DEV)
    assert torch.equal(torch.isnan(lse2), hit)
    assert torch.equal(torch.isnan(O2).all(-1), hit) and torch.equal(torch.isnan(O2).any(-1), hit)
    assert torch.equal(O2[~hit], O[~hit]) and torch.equal(lse2[~hit], lse[~hit])


@pytest.mark.parametrize("lens,Hq,Hkv,D,md,walk", [
    ([2048, 30], 32, 8, 128, 6, "heap"),   # group kernel, 4 heads per slot
    ([2048, 30], 32, 8, 128, 6, "parents"),
    ([2100, 30], 32, 8, 64, 6, "heap"),
    ([2100, 30], 32, 16, 64, 1, "parents"),  # 2 heads; a walk that ends before its chunk
    ([60], 16, 4, 128, 6, "prefix"),  # one wave per query: lane groups without a first or a second step
    ([60], 16, 4, 64, 3, "prefix"),
    ([60], 16, 4, 32, 3, "prefix"),
    ([300], 8, 2, 128, 40, "prefix"),
])
def test_infinite_value_of_an_attended_node(lens, Hq, Hkv, D, md, walk):
    """Where a wave holds walks of several lengths: an infinity in one element of
    a leaf's, an inner node's and a root's V row comes out as that infinity in that element of exactly the queries that attend
    the node (their weights are far above 0), and changes nothing else."""
    from qattention_amd import _lib, ragged_attn as ra
    b, L = 4, 300
    Q, K, V, cu = make_inputs(lens, Hq, D, 9300 + D + Hkv, Hkv=Hkv)
    par = np.concatenate([np.maximum(np.arange(n) - 1, 0) // b for n in lens]).astype(np.int32)
    g = torch.Generator().manual_seed(9301)
    Kp, Vp = (torch.randn(len(lens), L, Hkv, D, generator=g).half().to(DEV) for _ in range(2))
    V2 = V.clone()
    nodes = [lens[0] - 1, 6, 0][:Hkv]
    for h, node in enumerate(nodes):
        V2[node, h, 5 + h] = float("inf") if h != 1 else float("-inf")

    def call(v):
        q, k, v, pd = Q.to(DEV), K.to(DEV), v.to(DEV), torch.from_numpy(par).to(DEV)
        if walk == "heap":
            return ra._tree_forward(q, k, v, cu, b, md, max(lens), True, _lib.ALGO_GATHER)
        if walk == "parents":
            return ra.ragged_attention_with_parents(q, k, v, cu, pd, md, max(lens))
        return ra.ragged_attention_prefix(q, k, v, cu.to(DEV), Kp, Vp, b, md, max_seqlen=max(lens), return_lse=True,
                                          num_splits=3, parents=pd)

    say("inf value", walk, lens, Hq, Hkv, D, md)
    (O, lse), (O2, lse2) = call(V), call(V2)
    r = Hq // Hkv
    want = O.clone()
    for h, node in enumerate(nodes):
        hit = _attends(cu, b, md, None, node).to(DEV)
        want[hit, h * r:(h + 1) * r, 5 + h] = V2[node, h, 5 + h].to(DEV)
    assert torch.equal(O2, want) and torch.equal(lse2, lse)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("L,ns", [(65, 1), (127, 1), (129, 1), (200, 1), (255, 1), (193, 2), (255, 2), (500, 3)])
def test_infinite_prefix_value_near_the_end(L, ns, D, dtype):
    """The last key block of a prefix that is no multiple of 64 keys starts early;
    an infinite value among the keys it shares with the block before (L - 64 is
    always one) and of the last key comes out as that infinity, in its element
    alone.  Small queries: no weight is near 0.  128-row tiles, the last one with
    waves that hold no rows."""
    from qattention_amd import ragged_attn as ra
    B, N, b, md, Hq, Hkv = 8, 121, 3, 4, 32, 8
    Q, K, V, cu = make_inputs([N] * B, Hq, D, 9400 + D + L, dtype=dtype, Hkv=Hkv)
    Q = Q * 0.125
    g = torch.Generator().manual_seed(9401)
    Kp, Vp = (torch.randn(B, L, Hkv, D, generator=g).to(dtype) for _ in range(2))
    call = lambda vp: ra.ragged_attention_prefix(  # noqa: E731
        *(x.to(DEV) for x in (Q, K, V, cu, Kp, vp)), b, md, max_seqlen=N, return_lse=True, num_splits=ns)
    say("inf prefix value", L, ns, D, dtype)
    O, lse = call(Vp)
    Vp2 = Vp.clone()
    Vp2[:, L - 64, 0, 3] = float("inf")
    Vp2[:, L - 64, 1, 4] = float("-inf")
    Vp2[:, L - 1, 2, 5] = float("inf")
    O2, lse2 = call(Vp2)
    want = O.clone()
    r = Hq // Hkv
    want[:, :r, 3] = float("inf")
    want[:, r:2 * r, 4] = float("-inf")
    want[:, 2 * r:3 * r, 5] = float("inf")
    assert torch.equal(O2, want) and torch.equal(lse2, lse)
