"""Which kernel a call gets, at each limit of the dispatch rules and one past it.

The outputs of every case are checked against the fp64 oracle too (fp16 2e-3,
half an ulp of |o| in [4, 8); bf16 2^-7 max(1, |o|) + 1e-3, one rounding of O)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import make_inputs, oracle_tree

pytestmark = pytest.mark.gpu
DEV = "cuda"
GATHER, STREAM, MERGE = "tree_gather_kernel", "tree_stream_kernel", "tree_merge_kernel"
H2, H4 = "tree_group_kernel, 2 heads", "tree_group_kernel, 4 heads"
L8, L16 = "tree_group_kernel, 8 lanes", "tree_group_kernel, 16 lanes"


def _parents(lens, b):
    return np.concatenate([np.maximum(np.arange(n) - 1, 0) // b for n in lens]).astype(np.int32)


def _check(O, ref, dtype, what):
    bound = 2e-3 if dtype == torch.float16 else 2.0 ** -7 * np.maximum(1.0, np.abs(ref)) + 1e-3
    assert (np.abs(O.double().cpu().numpy() - ref) <= bound).all(), what


def _walk(walk, lens, b, md, Hq, Hkv, D, algo):
    from qattention_amd import _lib, ragged_attn as ra
    Q, K, V, cu = make_inputs(lens, Hq, D, 9500 + md + D, Hkv=Hkv)
    q, k, v = Q.to(DEV), K.to(DEV), V.to(DEV)
    print("walk", walk, lens, b, md, Hq, Hkv, D, flush=True)
    par = None
    if walk == "heap":
        O, _ = ra._tree_forward(q, k, v, cu, b, md, max(lens), False, algo)
    elif walk == "parents":
        par = _parents(lens, b)
        O, _ = ra.ragged_attention_with_parents(q, k, v, cu, torch.from_numpy(par).to(DEV), md, max(lens))
    else:
        Kc, Vc, pt = ra.build_paged_kv(list(k.split(lens)), list(v.split(lens)), 16)
        O, _ = ra._paged_forward(q, Kc, Vc, pt.to(DEV), cu, b, md, max(lens), False, algo)
    name = _lib.last_kernel()
    _check(O, oracle_tree(Q, K, V, cu, b, md, parents=par)[0], torch.float16, walk)
    return name


@pytest.mark.parametrize("lens,b,md,Hq,Hkv,D,want", [
    # 4 heads per slot from 2048 waves on (4 lanes per slot at D = 32, else 8), 2 from 4096
    ([2048], 4, 5, 32, 8, 128, H4),
    ([2047], 4, 5, 32, 8, 128, GATHER),
    ([4096], 4, 6, 32, 8, 32, H4),
    ([4095], 4, 6, 32, 8, 32, GATHER),
    ([4096], 4, 6, 16, 8, 64, H2),
    ([4095], 4, 6, 16, 8, 64, GATHER),
    # one head, 16 lanes at D = 128: 8192 queries
    ([256], 2, 8, 32, 8, 128, L16),
    ([257], 2, 8, 32, 8, 128, GATHER),
    # 8 lanes at D = 128: up to 65536 queries of at most 4 steps
    ([2048], 28, 3, 32, 32, 128, L8),
    ([2049], 28, 3, 32, 32, 128, GATHER),
    ([2048], 2, 4, 32, 32, 128, GATHER),
])
@pytest.mark.parametrize("walk", ["heap", "parents", "paged"])
def test_walk_kernel(lens, b, md, Hq, Hkv, D, want, walk):
    from qattention_amd import _lib
    assert _walk(walk, lens, b, md, Hq, Hkv, D, _lib.ALGO_GATHER) == want


@pytest.mark.parametrize("B,N,b,md,Hq,Hkv,D,want", [
    (1, 672, 28, 2, 32, 32, 128, L8),
    (4, 1365, 4, 5, 32, 32, 128, STREAM),
    (24, 341, 4, 4, 32, 8, 64, H4),
    (8, 1023, 2, 9, 32, 8, 128, STREAM),
])
def test_auto_choice(B, N, b, md, Hq, Hkv, D, want):
    from qattention_amd import _lib
    assert _walk("heap", [N] * B, b, md, Hq, Hkv, D, _lib.ALGO_AUTO) == want


@pytest.mark.parametrize("B,N,Hq,Hkv,D,dtype,want", [
    # one tree of up to 256 nodes: 8192 queries, else 6144 at D = 128 and 3072 at 64
    (1, 256, 32, 8, 128, torch.float16, MERGE),
    (1, 257, 32, 8, 128, torch.float16, GATHER),
    (2, 96, 32, 8, 128, torch.float16, MERGE),
    (2, 97, 32, 8, 128, torch.bfloat16, GATHER),
    (1, 256, 32, 8, 64, torch.bfloat16, MERGE),
    (2, 48, 32, 8, 64, torch.float16, MERGE),
    (2, 49, 32, 8, 64, torch.float16, GATHER),
    # D = 32: 1024 fp16, 3072 bf16
    (1, 32, 32, 8, 32, torch.float16, MERGE),
    (1, 33, 32, 8, 32, torch.float16, GATHER),
    (1, 96, 32, 8, 32, torch.bfloat16, MERGE),
    (1, 97, 32, 8, 32, torch.bfloat16, GATHER),
])
def test_split_merge_kernel(B, N, Hq, Hkv, D, dtype, want):
    from qattention_amd import _lib, ragged_attn as ra
    b, md, L = 3, 5, 300
    Q, K, V, cu = make_inputs([N] * B, Hq, D, 9600 + N + D, dtype=dtype, Hkv=Hkv)
    g = torch.Generator().manual_seed(9601)
    Kp, Vp = (torch.randn(B, L, Hkv, D, generator=g).to(dtype) for _ in range(2))
    print("merge", B, N, Hq, Hkv, D, dtype, flush=True)
    for par in (None, _parents([N] * B, b)):
        O = ra.ragged_attention_prefix(*(x.to(DEV) for x in (Q, K, V, cu, Kp, Vp)), b, md, max_seqlen=N, num_splits=3,
                                       parents=None if par is None else torch.from_numpy(par).to(DEV))
        assert _lib.last_kernel() == want
        _check(O, oracle_tree(Q, K, V, cu, b, md, parents=par, Kp=Kp, Vp=Vp)[0], dtype, (B, N, D))


@pytest.mark.parametrize("walk,lens,b,md,Hq,Hkv,want", [
    # 8 lanes at D = 64, up to 8192 queries, where 2 steps a round take less than
    # twice the rounds of 4 steps
    ("heap", [31], 2, 9, 32, 32, L8),      # 5 steps
    ("heap", [15, 15], 2, 3, 4, 4, GATHER),  # 4
    ("heap", [100], 28, 9, 32, 8, GATHER),  # 3
    ("heap", [200], 2, 9, 32, 8, GATHER),   # 8
    ("heap", [256], 2, 9, 32, 32, L8),     # 9
    ("heap", [257], 2, 9, 32, 32, GATHER),  # 8224 queries
    ("paged", [200], 4, 9, 32, 32, L8),    # 5
    ("paged", [80], 4, 9, 32, 32, GATHER),  # 4
    # explicit parents: more than 4 steps
    ("parents", [200], 4, 7, 32, 8, L8),
    ("parents", [200], 4, 3, 32, 8, GATHER),
])
def test_walk_kernel_d64(walk, lens, b, md, Hq, Hkv, want):
    from qattention_amd import _lib
    assert _walk(walk, lens, b, md, Hq, Hkv, 64, _lib.ALGO_GATHER) == want


@pytest.mark.parametrize("walk,N,want", [("heap", 384, L16), ("heap", 385, GATHER), ("parents", 384, L16),
                                         ("parents", 385, GATHER), ("paged", 256, L16), ("paged", 257, GATHER)])
def test_walk_kernel_ungrouped_heads(walk, N, want):
    """16 lanes at D = 128: 12288 queries of ungrouped heads, paged 8192."""
    from qattention_amd import _lib
    assert _walk(walk, [N], 2, 9, 32, 32, 128, _lib.ALGO_GATHER) == want


@pytest.mark.parametrize("N,md,want", [(2048, 31, H4), (2048, 32, GATHER), (8191, 40, GATHER), (8192, 40, H4)])
def test_deep_walk_kernel(N, md, want):
    """Walks of more than 32 steps at D = 128 need four times the waves."""
    from qattention_amd import _lib
    for walk in ("heap", "parents"):
        assert _walk(walk, [N], 1, md, 32, 8, 128, _lib.ALGO_GATHER) == want
