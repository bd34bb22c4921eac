"""The group kernel: grouped q heads walked together (2 or 4 per loaded K/V row).

It serves packed calls without split states whose slots fill the GPU
(8192 / GS waves of 64 lanes, GS heads per slot), and with one head and more
lanes per slot those too small to fill it, through the heap walk, the
explicit-parents walk and paged K/V.  Each case is checked against the fp64
oracle, O and LSE, and its walk against the oracle's ancestor table; the cases
just below the threshold run the gather kernel on the same inputs.
Tolerances: fp16 max |o - o_ref| <= 2e-3 (half an ulp of |o| in [4, 8) is
1.95e-3; inputs N(0, 1)), bf16 2^-7 max(1, |o_ref|) + 1e-3 (one rounding of O),
LSE 1e-4 / 1e-3 (fp32 sums of rounded products), as in the other GPU tests."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import make_inputs, oracle_tree

pytestmark = pytest.mark.gpu
DEV = "cuda"


def say(*a):
    print(*a, flush=True)


def _ra():
    from qattention_amd import _lib, ragged_attn
    return ragged_attn, _lib


def _check(O, L, o_ref, lse_ref, dtype, what):
    o = O.double().cpu().numpy()
    bound = 2e-3 if dtype == torch.float16 else 2.0 ** -7 * np.maximum(1.0, np.abs(o_ref)) + 1e-3
    assert (np.abs(o - o_ref) <= bound).all(), f"{what}: {np.abs(o - o_ref).max():.3e}"
    if L is not None:
        err = np.abs(L.double().cpu().numpy() - lse_ref).max()
        assert err <= (1e-4 if dtype == torch.float16 else 1e-3), f"{what}: LSE {err:.3e}"


def _waves(lens, Hq, Hkv, D):
    gs = 4 if (Hq // Hkv) % 4 == 0 else 2
    return len(lens) * max(lens) * (Hq // gs) * (4 if D == 32 else 8) // 64, 8192 // gs


def _parents(lens, seed):
    rng = np.random.default_rng(seed)
    out = []
    for n in lens:
        p = np.zeros(n, dtype=np.int32)
        for i in range(1, n):
            p[i] = rng.integers(max(0, i - 40), i)
        out.append(p)
    return np.concatenate(out)


# lens, b, max_depth, Hq, Hkv, D, dtype: the threshold itself and one node below
# it, ragged with empty and one-token sequences, groups of 2, 4, 6 and 8 heads
CASES = [
    ([2048], 4, 5, 32, 8, 128, torch.float16),
    ([2047], 4, 5, 32, 8, 128, torch.float16),
    ([700, 0, 301, 1, 699], 3, 4, 32, 8, 64, torch.float16),
    ([700, 0, 301, 1, 699], 3, 4, 32, 8, 64, torch.bfloat16),
    ([1100, 1093], 28, 2, 32, 4, 128, torch.bfloat16),
    ([1365] * 2, 2, 10, 24, 4, 64, torch.float16),
    ([1025, 1024, 7], 2, 3, 16, 8, 128, torch.float16),
    ([2049, 2050], 5, 6, 32, 8, 32, torch.float16),
    ([2100], 1, 9, 32, 8, 64, torch.float16),
    # one head per slot (16 and 8 lanes) and the gather kernel beyond
    ([512], 2, 9, 32, 32, 128, torch.float16),
    ([513], 2, 9, 32, 32, 128, torch.bfloat16),
    ([256, 0], 4, 4, 16, 8, 128, torch.bfloat16),
    ([257], 4, 4, 32, 8, 64, torch.float16),
    ([15, 15], 2, 3, 4, 4, 64, torch.float16),
    ([2048], 28, 3, 32, 32, 128, torch.float16),
    ([2049], 28, 3, 32, 32, 128, torch.float16),
    ([1, 3, 0], 3, 2, 3, 1, 128, torch.float16),
]


@pytest.mark.parametrize("walk", ["heap", "parents"])
@pytest.mark.parametrize("lens,b,md,Hq,Hkv,D,dtype", CASES)
def test_group_walk(lens, b, md, Hq, Hkv, D, dtype, walk):
    ra, _lib = _ra()
    from oracle import clib
    say("group", walk, lens, b, md, Hq, Hkv, D, dtype, "waves", _waves(lens, Hq, Hkv, D))
    Q, K, V, cu = make_inputs(lens, Hq, D, 7000 + len(lens) * 10 + md, dtype=dtype, Hkv=Hkv)
    T = Q.shape[0]
    table = torch.full((T, Hq, md + 1), -9, dtype=torch.int32, device=DEV)
    q, k, v = Q.to(DEV), K.to(DEV), V.to(DEV)
    if walk == "heap":
        par = None
        call = lambda lse: ra._tree_forward(q, k, v, cu, b, md, max(lens), lse, _lib.ALGO_GATHER)  # noqa: E731
        ref = clib.ancestor_table_heap(cu.numpy(), b, md)
    else:
        par = _parents(lens, 7100 + md)
        pd = torch.from_numpy(par).to(DEV)
        call = lambda lse: ra.ragged_attention_with_parents(q, k, v, cu, pd, md, max(lens))  # noqa: E731
        ref = clib.ancestor_table_parents(cu.numpy(), par, md)
    o_ref, lse_ref, _ = oracle_tree(Q, K, V, cu, b, md, parents=par)
    O, L = call(True)
    _check(O, L, o_ref, lse_ref, dtype, walk)
    O2, _ = call(False)
    assert torch.equal(O, O2)
    with _lib.debug_walk(table):
        O3, _ = call(True)
    assert torch.equal(O, O3)
    got = table.cpu().numpy()
    assert (got == ref[:, None, :]).all(), "walk"


@pytest.mark.parametrize("D,dtype,Hkv", [(128, torch.float16, 8), (64, torch.bfloat16, 16)])
def test_group_paged(D, dtype, Hkv):
    """Paged K/V in shuffled pages, one page missing from the second sequence."""
    ra, _lib = _ra()
    lens, b, md, Hq, ps = [1500, 1365], 4, 5, 32, 16
    Q, K, V, cu = make_inputs(lens, Hq, D, 7300 + D, dtype=dtype, Hkv=Hkv)
    ks, vs = (list(x.to(DEV).split(lens)) for x in (K, V))
    Kc, Vc, pt = ra.build_paged_kv(ks, vs, ps)
    perm = torch.from_numpy(np.random.default_rng(3).permutation(Kc.shape[0]))
    K2, V2 = torch.empty_like(Kc), torch.empty_like(Vc)
    K2[perm.to(DEV)], V2[perm.to(DEV)] = Kc, Vc
    pt = perm.to(torch.int32)[pt.long()]
    say("group paged", D, dtype, Hkv)
    O, L = ra._paged_forward(Q.to(DEV), K2, V2, pt.to(DEV), cu, b, md, max(lens), True, _lib.ALGO_GATHER)
    o_ref, lse_ref, _ = oracle_tree(Q, K, V, cu, b, md)
    _check(O, L, o_ref, lse_ref, dtype, "paged")
    pt[1, 3] = -1
    G, GL = ra._paged_forward(Q.to(DEV), K2, V2, pt.to(DEV), cu, b, md, max(lens), True, _lib.ALGO_GATHER)
    S, SL = ra._paged_forward(Q.to(DEV), K2, V2, pt.to(DEV), cu, b, md, max(lens), True, _lib.ALGO_SUBTREE)
    bound = 2e-3 if dtype == torch.float16 else 2.0 ** -6 * max(1.0, float(S.abs().max()))
    assert float((G.float() - S.float()).abs().max()) <= bound
    fin = torch.isfinite(SL)
    assert torch.equal(fin, torch.isfinite(GL)) and float((GL - SL)[fin].abs().max()) <= 1e-3


def test_group_strided_and_captured():
    """Head-major storage (a permuted view) and a graph replayed over new inputs."""
    ra, _lib = _ra()
    lens, b, md, Hq, Hkv, D = [1365, 900], 4, 5, 32, 8, 128
    Q, K, V, cu = make_inputs(lens, Hq, D, 7400, Hkv=Hkv)
    hm = lambda x: x.to(DEV).permute(1, 0, 2).contiguous().permute(1, 0, 2)  # noqa: E731
    q, k, v = hm(Q), hm(K), hm(V)
    cud = cu.to(DEV)
    say("group strided")
    O, _ = ra._tree_forward(q, k, v, cud, b, md, max(lens), False, _lib.ALGO_GATHER)
    o_ref, lse_ref, _ = oracle_tree(Q, K, V, cu, b, md)
    _check(O, None, o_ref, lse_ref, torch.float16, "strided")
    side = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        R, _ = ra._tree_forward(q, k, v, cud, b, md, max(lens), False, _lib.ALGO_GATHER)
    for i in range(3):
        q.copy_(q.roll(1, 0))
        g.replay()
        E, _ = ra._tree_forward(q, k, v, cud, b, md, max(lens), False, _lib.ALGO_GATHER)
        torch.cuda.synchronize()
        assert torch.equal(R, E), i


@pytest.mark.parametrize("B,N,b,md,Hq,Hkv,D", [
    (1, 672, 28, 2, 32, 32, 128),   # auto: the walk, 8 lanes per query (one round of wide tiles costs more)
    (4, 1365, 4, 5, 32, 32, 128),   # auto: the subtree kernel
    (24, 341, 4, 4, 32, 8, 64),     # auto: the group kernel
    (8, 1023, 2, 9, 32, 8, 128),    # auto: the subtree kernel, deep trees
])
def test_auto_choice_agrees_with_every_kernel(B, N, b, md, Hq, Hkv, D):
    """The kernel that the estimates choose (test_gpu_dispatch.py asserts which)
    computes what the others do: two
    fp32 softmaxes over the same rounded rows differ by less than one fp16
    rounding of O (2^-10 of |O| <= 6)."""
    ra, _ = _ra()
    Q, K, V, cu = make_inputs([N] * B, Hq, D, 7500 + B, Hkv=Hkv)
    q, k, v = Q.to(DEV), K.to(DEV), V.to(DEV)
    say("auto", B, N, b, md, Hq, Hkv, D)
    o = [ra._tree_forward(q, k, v, cu, b, md, N, True, a) for a in (0, 1, 2)]
    assert any(torch.equal(o[0][0], x[0]) for x in o[1:])
    for x in o[1:]:
        assert float((x[0].float() - o[0][0].float()).abs().max()) <= 6 * 2.0 ** -10
        assert float((x[1] - o[0][1]).abs().max()) <= 1e-4
