"""The one-wave-per-query merge and walk: split prefix states of few queries.

It serves split prefix calls of few (token, q head) pairs (the limits, by head
size and type, are in test_gpu_dispatch.py; the D = 32 case of 8160 pairs is the
gather kernel's).  Cases at the sizes where its sharing of states and steps between lane groups can go
wrong: fewer splits than groups, more than two per group, walks of one step,
of exactly and more than two rounds of steps, trees on both sides of the 256
parents kept in registers, empty sequences.  Checked against the fp64 oracle
(fp16: 2e-3 * max(1, |o|), half an ulp of an output of size |o| in [4, 8);
bf16: 2^-7 max(1, |o|) + 1e-3; LSE 1e-4 / 1e-3 as in the other GPU tests) and,
step by step, against the oracle's ancestor table."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import make_inputs, oracle_tree

pytestmark = pytest.mark.gpu
DEV = "cuda"


def say(*a):
    print(*a, flush=True)


def _parents(lens, seed, window):
    rng = np.random.default_rng(seed)
    out = []
    for n in lens:
        p = np.zeros(n, dtype=np.int32)
        for i in range(1, n):
            p[i] = rng.integers(max(0, i - window), i)
        out.append(p)
    return np.concatenate(out)


# lens, b (0: random parents), max_depth, Hq, Hkv, D, L, splits, dtype
CASES = [
    ([60], 0, 7, 32, 8, 128, 2048, 0, torch.float16),
    ([60], 0, 7, 32, 8, 128, 2048, 0, torch.bfloat16),
    ([60, 0, 1, 33], 4, 3, 8, 2, 128, 300, 2, torch.float16),
    ([85, 85], 4, 0, 8, 8, 128, 700, 11, torch.float16),
    ([85, 85], 2, 6, 8, 8, 64, 700, 11, torch.bfloat16),
    ([256], 0, 30, 8, 4, 128, 640, 9, torch.float16),
    ([257], 0, 30, 8, 4, 128, 640, 10, torch.float16),
    ([300, 10], 1, 40, 4, 2, 64, 1280, 17, torch.float16),
    ([200], 0, 70, 4, 1, 32, 2200, 34, torch.float16),
    ([255], 3, 8, 32, 8, 32, 130, 3, torch.bfloat16),
]


@pytest.mark.parametrize("lens,b,md,Hq,Hkv,D,L,ns,dtype", CASES)
def test_merge_walk(lens, b, md, Hq, Hkv, D, L, ns, dtype):
    from oracle import clib
    from qattention_amd import _lib, ragged_attn as ra
    say("merge", lens, b, md, Hq, Hkv, D, L, ns, dtype)
    assert len(lens) * max(lens) * Hq < 8192
    Q, K, V, cu = make_inputs(lens, Hq, D, 8000 + md + D, dtype=dtype, Hkv=Hkv)
    g = torch.Generator().manual_seed(8100 + L)
    Kp = torch.randn(len(lens), L, Hkv, D, generator=g).to(dtype)
    Vp = torch.randn(len(lens), L, Hkv, D, generator=g).to(dtype)
    par = None if b else _parents(lens, 8200 + md, 9 if md > 20 else 60)
    pd = None if b else torch.from_numpy(par).to(DEV)
    dev = [x.to(DEV) for x in (Q, K, V, cu, Kp, Vp)]

    def call():
        return ra.ragged_attention_prefix(*dev, b or 1, md, max_seqlen=max(lens), return_lse=True, num_splits=ns,
                                          parents=pd)

    O, lse = call()
    o_ref, lse_ref, _ = oracle_tree(Q, K, V, cu, b or 1, md, parents=par, Kp=Kp, Vp=Vp)
    o = O.double().cpu().numpy()
    one = np.maximum(1.0, np.abs(o_ref))
    bound = 2e-3 * one if dtype == torch.float16 else 2.0 ** -7 * one + 1e-3
    assert (np.abs(o - o_ref) <= bound).all(), np.abs(o - o_ref).max()
    assert np.abs(lse.double().cpu().numpy() - lse_ref).max() <= (1e-4 if dtype == torch.float16 else 1e-3)
    table = torch.full((Q.shape[0], Hq, md + 1), -9, dtype=torch.int32, device=DEV)
    with _lib.debug_walk(table):
        O2, _ = call()
    assert torch.equal(O, O2)
    ref = clib.ancestor_table_heap(cu.numpy(), b, md) if b else clib.ancestor_table_parents(cu.numpy(), par, md)
    assert (table.cpu().numpy() == ref[:, None, :]).all()
