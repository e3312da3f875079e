"""prefill_split_kernel: row blocks of 64, 128 and 256 (token, head) rows with the
keys split over groups of waves, at head_dim 64 and 128, fp16 and FP8 caches, and the
256-row items of the one-wave kernels ordered in the call.
Query lengths at the edges of the blocks and of the key tiles, contexts shorter
than one tile (key groups without a key) and than a round of tiles; slots that no
row attends hold NaN (fp16 caches).  Reference: the oracle."""
import numpy as np
import pytest

from helpers import F16_ATOL, F16_RTOL, assert_close, to_dev, to_np
from test_gpu_prefill import _cache, _case, _threads

pytestmark = pytest.mark.gpu

# (H, Hkv, D, bs, query lengths, prior contexts).  The blocks are those with the least
# estimated time on 256 CUs; a name ends in its case's (d64-128 takes 64 with an FP8
# cache; 256w: contexts of at most 256 keys, one key group).
_EDGES = [2, 3, 9, 10, 31, 32, 33, 64, 65]
CASES = {
    "d64-64": (14, 2, 64, 16, _EDGES + [1], [0, 61, 0, 30, 1, 0, 31, 700, 64, 40]),
    "d64-64-mha": (6, 6, 64, 8, _EDGES + [129, 1], [0, 61, 0, 30, 1, 0, 31, 700, 64, 127, 9]),
    "d64-128": (14, 2, 64, 32, _EDGES + [1, 700, 601], [0, 61, 0, 30, 1, 0, 31, 70, 64, 40, 0, 129]),
    "d64-128-fp8": (14, 2, 64, 32, _EDGES + [1, 400, 401, 399, 410, 390], [0, 61, 0, 30, 1, 0, 31, 70, 64, 40, 0, 129, 64, 1, 31]),
    "d64-256w": (14, 2, 64, 16, _EDGES * 2 + [100] * 24 + [129, 255, 1],
                 [0, 61, 0, 30, 1, 0, 31, 70, 64] * 2 + [0, 7, 100] * 8 + [127, 0, 9]),
    "d64-256w-g16": (32, 2, 64, 16, _EDGES + [100] * 8 + [129, 255, 1],
                     [0, 61, 0, 30, 1, 0, 31, 70, 64] + [0, 7] * 4 + [127, 0, 9]),
    "d128-256": (28, 4, 128, 16, _EDGES + [100] * 14 + [1, 129], [0, 61, 0, 30, 1, 0, 31, 70, 64] + [0, 7] * 7 + [9, 40]),
    "d64-256": (32, 4, 64, 16, _EDGES + [1, 700, 601, 720], [0, 61, 0, 30, 1, 0, 31, 70, 64, 40, 0, 129, 64]),
    "d128-64": (28, 4, 128, 32, _EDGES + [1], [0, 61, 0, 30, 1, 0, 31, 700, 64, 40]),
    "d128-128": (32, 8, 128, 16, _EDGES + [1, 300, 301], [0, 61, 0, 30, 1, 0, 31, 70, 64, 40, 0, 129]),
    "d128-128-mqa": (40, 1, 128, 16, _EDGES + [1, 200, 101], [0, 61, 0, 30, 1, 0, 31, 70, 64, 40, 0, 129]),
}


@pytest.mark.parametrize("kvt", ["f16", "fp8"])
@pytest.mark.parametrize("case", list(CASES))
def test_prefill_split_vs_oracle(vkv, oracle, cuda, kvt, case):
    import torch
    H, Hkv, D, bs, q_lens, prior = CASES[case]
    lay, ctx, qsl, q, k, v, scale = _case(H, Hkv, D, bs, q_lens, prior, H + D)
    if case == "d64-64-mha":
        scale = -scale
    (kc, vc, ks, vs), (hk, hv, hks, hvs) = _cache(vkv, cuda, kvt, k, v)
    ref = oracle.paged_prefill(q.astype(np.float32), hk, hv, lay.block_tables, ctx, qsl, scale,
                               key_scales=hks, value_scales=hvs, nthreads=_threads())
    if kvt == "f16":
        used = np.zeros((lay.num_blocks, bs), bool)
        for s, n in enumerate(ctx):
            pos = np.arange(n)
            used[lay.block_tables[s, pos // bs], pos % bs] = True
        kc[to_dev(~used, cuda)] = float("nan")
        vc[to_dev(~used, cuda)] = float("nan")
    out = torch.full((q.shape[0], H, D), 7.0, dtype=torch.float16, device=cuda)
    vkv.paged_prefill(out, to_dev(q, cuda), kc, vc, to_dev(lay.block_tables, cuda), to_dev(ctx, cuda),
                      to_dev(qsl, cuda), int(max(q_lens)), scale, key_scales=ks, value_scales=vs)
    torch.cuda.synchronize()
    assert_close(to_np(out).astype(np.float32), ref, F16_ATOL, F16_RTOL, f"{case} ({kvt})")
