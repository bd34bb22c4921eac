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
