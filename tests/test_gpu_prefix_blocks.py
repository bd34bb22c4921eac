"""The prefix kernel's key loop by number of 64-key blocks.

Its first block, its loop of two iterations, entered at either, its last block
(which starts early where the range is no multiple of 64) and the loads past
the end depend on the block count, its step placement on head_dim, and waves
without query rows run a loop of their own.  1 to 5 blocks per range, 1, 63 and
64 keys in the last, fused (one range) and split in two with at least 256 units
(128-row tiles), row counts that leave 1, 2 and 3 waves of the last tile idle.
Checked against the fp64 oracle (fp16: 2e-3, half an ulp of |o| in [4, 8);
bf16: 2^-7 max(1, |o|) + 1e-3, one rounding of O and of P; LSE 1e-4 / 1e-3, fp32
sums of rounded products)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import make_inputs, oracle_tree

pytestmark = pytest.mark.gpu
DEV = "cuda"
B, HQ, HKV, b, MD = 8, 32, 8, 3, 4


@pytest.mark.parametrize("splits", [1, 2])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("blocks", [1, 2, 3, 4, 5])
def test_blocks_per_range(blocks, D, dtype, splits):
    from qattention_amd import ragged_attn as ra
    for i, last in enumerate((1, 63, 64)):
        N = (33, 41, 49)[(i + blocks) % 3]  # 132, 164, 196 rows per kv head: 3, 2, 1 waves without rows
        assert B * HKV * -(-N * HQ // HKV // 128) * splits >= 256 or splits == 1
        L = 64 * (splits * blocks - 1) + last
        print("blocks", blocks, last, N, D, dtype, splits, flush=True)
        Q, K, V, cu = make_inputs([N] * B, HQ, D, 6000 + 100 * blocks + last, dtype=dtype, Hkv=HKV)
        g = torch.Generator().manual_seed(6001 + L)
        Kp, Vp = (torch.randn(B, L, HKV, D, generator=g).to(dtype) for _ in range(2))
        O, lse = ra.ragged_attention_prefix(*(x.to(DEV) for x in (Q, K, V, cu, Kp, Vp)), b, MD, max_seqlen=N,
                                            return_lse=True, num_splits=splits)
        o_ref, lse_ref, _ = oracle_tree(Q, K, V, cu, b, MD, Kp=Kp, Vp=Vp)
        o = O.double().cpu().numpy()
        bound = 2e-3 if dtype == torch.float16 else 2.0 ** -7 * np.maximum(1.0, np.abs(o_ref)) + 1e-3
        assert (np.abs(o - o_ref) <= bound).all(), (last, N, np.abs(o - o_ref).max())
        err = np.abs(lse.double().cpu().numpy() - lse_ref).max()
        assert err <= (1e-4 if dtype == torch.float16 else 1e-3), (last, N, err)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [32, 64, 128])
def test_small_weights_after_a_large_one(D, dtype):
    """One key of weight 1 and 2^17 of weight 2^-25: added one by one to a sum
    above 1 each would round away (a quarter of the 2^-8 in all, those of one
    lane's partial sum: 1e-3 of the LSE); added block by block 16 of them are 4
    ulps.  Both weights are within 1e-3 of those powers, so a block's 4 ulps
    round to 4 and at most 2^-10 of 2^-8 is lost: 4e-6, and 4e-6 for the fp32
    sums and the logarithm."""
    from qattention_amd import ragged_attn as ra
    L = 1 + 2 ** 17
    step = 2.0 ** (-10 if dtype == torch.float16 else -7)
    mant = 1.0 + step * np.arange(0, int(1 / step), max(1, int(1 / step) // 64))
    c = 1.0 + step * np.arange(int(1 / step))
    s = mant[:, None] * c[None, :] * 64 / np.sqrt(D) * np.log2(np.e)  # (both times 8)
    pow2 = 2.0 ** np.round(np.log2(25 / s))
    i, j = np.unravel_index(np.abs(s * pow2 - 25).argmin(), s.shape)
    Q = torch.zeros(1, 1, D)
    Q[0, 0, 0] = mant[i] * 8 * pow2[i, j]
    K = torch.zeros(L, 1, D)
    K[0, 0, 0] = c[j] * 8
    Q, K = Q.to(dtype).to(DEV), K.to(dtype).to(DEV)
    score = float(Q[0, 0, 0]) * float(K[0, 0, 0]) / np.sqrt(D)
    assert abs(score * np.log2(np.e) - 25) < 1e-3, score
    print("small weights", D, dtype, score, flush=True)
    _, lse = ra.prefix_attention(Q, K, torch.zeros_like(K), num_splits=1)
    want = score + np.log1p((L - 1) * np.exp(-score))
    assert abs(float(lse[0, 0]) - want) <= 8e-6, (float(lse[0, 0]), want)
