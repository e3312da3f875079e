"""decode_stream.hip: fp16 queries over fp16 caches at head_dim 64 to 128, as one
workgroup per (row, kv head) (short tables) and in equal slices (long tables).

Every unattended slot of the pool holds NaN, so a read of one that reaches the
result shows.  Reference: the oracle on the same pool (NaN replaced there: the
oracle reads attended slots only)."""
import numpy as np
import pytest

from helpers import F16_ATOL, F16_RTOL, assert_close, to_dev, to_np

pytestmark = pytest.mark.gpu

# (H, Hkv, D, block size): each head dimension, both head tiles, groups of one,
# block sizes that are no power of two or shorter than a step
SHAPES = [(14, 2, 64, 16), (2, 2, 64, 1), (34, 2, 64, 24), (4, 4, 80, 16), (32, 2, 80, 12), (33, 33, 80, 16),
          (3, 3, 96, 32), (16, 1, 96, 5), (16, 16, 112, 16), (34, 2, 112, 16), (32, 2, 128, 16), (32, 1, 128, 16),
          (8, 2, 128, 8), (8, 8, 128, 48)]
# contexts at the edges of a step (32 tokens), of a wave's share and of a slice
CONTEXTS = [1, 31, 0, 32, 33, 64, 65, 257, 0, 700]


def _case(rng, H, Hkv, D, bs, ctx, table_tokens):
    from vllm_kv_amd import workloads
    lay = workloads.make_layout(np.asarray(ctx, np.int32), bs, rng, max_blocks_per_seq=-(-table_tokens // bs))
    shape = (lay.num_blocks, bs, Hkv, D)
    pools = [(rng.standard_normal(shape, dtype=np.float32) * 0.7).astype(np.float16) for _ in range(2)]
    used = np.zeros((lay.num_blocks, bs), bool)
    for s, n in enumerate(ctx):
        pos = np.arange(n)
        used[lay.block_tables[s, pos // bs], pos % bs] = True
    for p in pools:
        p[~used] = np.nan
    q = (rng.standard_normal((len(ctx), H, D), dtype=np.float32) * 0.7).astype(np.float16)
    return lay, pools, q


@pytest.mark.parametrize("table", [1024, 6000], ids=["rows", "slices"])
@pytest.mark.parametrize("H,Hkv,D,bs", SHAPES)
def test_stream_edges_vs_oracle(vkv, oracle, cuda, H, Hkv, D, bs, table):
    import torch
    rng = np.random.default_rng(D * 100 + H + bs)
    lay, (k, v), q = _case(rng, H, Hkv, D, bs, CONTEXTS, table)
    scale = -float(D) ** -0.5 if bs == 24 else float(D) ** -0.5
    ref = oracle.paged_decode(q.astype(np.float32), np.nan_to_num(k).view(np.uint16), np.nan_to_num(v).view(np.uint16),
                              lay.block_tables, lay.context_lens, scale)
    args = (to_dev(q, cuda), to_dev(k, cuda), to_dev(v, cuda), to_dev(lay.block_tables, cuda),
            to_dev(lay.context_lens, cuda), scale)
    for size in (0, 64):  # the library's slices, and the caller's
        out = torch.full((len(CONTEXTS), H, D), 7.0, dtype=torch.float16, device=cuda)
        vkv.paged_decode(out, *args, partition_size=size)
        torch.cuda.synchronize()
        assert_close(to_np(out).astype(np.float32), ref, F16_ATOL, F16_RTOL, f"{H}/{Hkv}/{D}/bs{bs} size {size}")
    acc = torch.ones((len(CONTEXTS), H, D), dtype=torch.float16, device=cuda)
    vkv.paged_decode(acc, *args, accumulate=True)
    torch.cuda.synchronize()
    assert_close(to_np(acc).astype(np.float32), ref + 1.0, F16_ATOL, F16_RTOL, "accumulate")


@pytest.mark.parametrize("table", [1024, 6000], ids=["rows", "slices"])
@pytest.mark.parametrize("H,Hkv,D,bs", [(4, 4, 80, 16), (34, 2, 112, 24), (32, 2, 128, 16), (14, 2, 64, 8)])
def test_stream_fused_append(vkv, cuda, H, Hkv, D, bs, table):
    """The fused step against the append and the decode as two calls: same bits."""
    import torch
    rng = np.random.default_rng(D + bs)
    ctx = [1, 32, 33, 300, 31]
    lay, (k, v), q = _case(rng, H, Hkv, D, bs, ctx, table)
    new = [(rng.standard_normal((len(ctx), Hkv, D), dtype=np.float32) * 0.7).astype(np.float16) for _ in range(2)]
    slots = lay.slots(lay.context_lens - 1, np.arange(len(ctx)))
    slots[3] = -1  # skipped: the cache keeps its rows and the decode reads them
    got = []
    for fused in (True, False):
        kc, vc = to_dev(k, cuda), to_dev(v, cuda)
        out = torch.zeros((len(ctx), H, D), dtype=torch.float16, device=cuda)
        args = (out, to_dev(q, cuda), kc, vc, to_dev(lay.block_tables, cuda), to_dev(lay.context_lens, cuda), D ** -0.5)
        rows = (to_dev(new[0], cuda), to_dev(new[1], cuda))
        if fused:
            vkv.paged_decode_append(*args, *rows, to_dev(slots, cuda))
        else:
            vkv.reshape_and_cache(*rows, kc, vc, to_dev(slots, cuda))
            vkv.paged_decode(*args)
        torch.cuda.synchronize()
        got.append([to_np(x).view(np.uint16) for x in (out, kc, vc)])
    for a, b in zip(*got):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("S,table", [(520, 32), (520, 64), (520, 80), (520, 384), (520, 400), (1030, 128), (1030, 144),
                                     (2060, 528), (2060, 544)])
@pytest.mark.parametrize("H,Hkv,D,dtype", [(2, 2, 64, "f16"), (14, 2, 64, "f32"), (8, 2, 80, "f16"), (2, 2, 112, "f16"),
                                           (6, 2, 128, "f16"), (4, 2, 128, "fp8")])
def test_stream_many_short_rows(vkv, oracle, cuda, S, table, H, Hkv, D, dtype):
    """Over 4, 8 and 16 (row, kv head) pairs per CU at the edges of the tables that one
    wave and two attend: rows of every length against the oracle, and the fused append
    against the two calls bit for bit."""
    import torch
    from helpers import F32_ATOL, F32_RTOL
    bs = 16
    rng = np.random.default_rng(S + table + D)
    ctx = rng.integers(0, min(table, 400 if S < 2000 else 48) + 1, S)
    ctx[:9] = [table, 0, 1, 31, 32, table - 1, table // 2, table // 2 + 1, min(33, table)]
    lay, (k, v), q = _case(rng, H, Hkv, D, bs, ctx, table)
    rows = np.unique(np.concatenate([np.arange(9), np.linspace(9, S - 1, 24).astype(int)]))
    args = [to_dev(lay.block_tables, cuda), to_dev(lay.context_lens, cuda), D ** -0.5]
    if dtype == "fp8":
        hole = np.isnan(k)
        codes = [rng.integers(0, 0x70, k.shape).astype(np.uint8) for _ in range(2)]
        sc = [rng.uniform(0.005, 0.02, k.shape[:3]).astype(np.float32) for _ in range(2)]
        ref = oracle.paged_decode(q[rows].astype(np.float32), *codes, lay.block_tables[rows], lay.context_lens[rows], D ** -0.5,
                                  key_scales=sc[0], value_scales=sc[1])
        for c, x in zip(codes, sc):
            c[hole] = 0x7F
            x[hole[..., 0]] = np.nan
        out = torch.zeros((S, H, D), dtype=torch.float16, device=cuda)
        vkv.paged_decode(out, to_dev(q, cuda), *[to_dev(c, cuda) for c in codes], *args,
                         key_scales=to_dev(sc[0], cuda), value_scales=to_dev(sc[1], cuda))
        torch.cuda.synchronize()
        assert_close(to_np(out)[rows].astype(np.float32), ref, F16_ATOL, F16_RTOL, f"table {table}")
        return
    if dtype == "f32":
        k, v, q = (x.astype(np.float32) * np.float32(1.0001) for x in (k, v, q))
        pools = [np.nan_to_num(x) for x in (k, v)]
    else:
        pools = [np.nan_to_num(x).view(np.uint16) for x in (k, v)]
    ref = oracle.paged_decode(q[rows].astype(np.float32), *pools, lay.block_tables[rows], lay.context_lens[rows], D ** -0.5)
    out = torch.zeros(q.shape, dtype=torch.float32 if dtype == "f32" else torch.float16, device=cuda)
    vkv.paged_decode(out, to_dev(q, cuda), to_dev(k, cuda), to_dev(v, cuda), *args)
    torch.cuda.synchronize()
    tol = (F32_ATOL, F32_RTOL) if dtype == "f32" else (F16_ATOL, F16_RTOL)
    assert_close(to_np(out)[rows].astype(np.float32), ref, *tol, f"table {table}")
    new = [(rng.standard_normal((S, Hkv, D)) * 0.7).astype(q.dtype) for _ in range(2)]
    slots = lay.slots(np.maximum(lay.context_lens - 1, 0), np.arange(S))
    slots[lay.context_lens == 0] = -1
    got = []
    for fused in (True, False):
        kc, vc = to_dev(k, cuda), to_dev(v, cuda)
        out = torch.zeros_like(out)
        call, nw = (out, to_dev(q, cuda), kc, vc, *args), [to_dev(x, cuda) for x in new]
        if fused:
            vkv.paged_decode_append(*call, *nw, to_dev(slots, cuda))
        else:
            vkv.reshape_and_cache(*nw, kc, vc, to_dev(slots, cuda))
            vkv.paged_decode(*call)
        torch.cuda.synchronize()
        got.append([to_np(x).tobytes() for x in (out, kc, vc)])
    assert got[0] == got[1]


# (rows, contexts, caller's partition size): a call whose finer partials once did not
# fit the library's array, so that it ran unsplit; many rows of short contexts; and
# a caller's size whose slices, with one of each row more, do not fit (coarser ones do)
@pytest.mark.parametrize("S,Hkv,lo,hi,table,size", [(64, 1, 900, 1100, 32768, 0), (400, 2, 1, 40, 4096, 0),
                                                    (63, 2, 4096, 4096, 4096, 64)])
def test_stream_noalloc_fits_its_array(vkv, oracle, cuda, S, Hkv, lo, hi, table, size):
    """Accepted like the call with a workspace and as right, whatever the array holds."""
    import torch
    H, D, bs = 32, 128, 16
    rng = np.random.default_rng(3)
    ctx = rng.integers(lo, hi + 1, S)
    lay, (k, v), q = _case(rng, H, Hkv, D, bs, ctx, table)
    outs = [torch.zeros((S, H, D), dtype=torch.float16, device=cuda) for _ in range(2)]
    args = (to_dev(q, cuda), to_dev(k, cuda), to_dev(v, cuda), to_dev(lay.block_tables, cuda),
            to_dev(lay.context_lens, cuda), D ** -0.5)
    if size:
        assert vkv.decode_workspace_size(outs[0], *args, partition_size=size) > 64 << 20
    vkv.paged_decode_noalloc(outs[0], *args, partition_size=size)
    vkv.paged_decode(outs[1], *args, partition_size=size)
    torch.cuda.synchronize()
    if not size:  # the same slices
        assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))
    rows = np.unique(np.linspace(0, S - 1, 12).astype(int))
    ref = oracle.paged_decode(q[rows].astype(np.float32), np.nan_to_num(k).view(np.uint16),
                              np.nan_to_num(v).view(np.uint16), np.ascontiguousarray(lay.block_tables[rows]),
                              np.ascontiguousarray(lay.context_lens[rows]), D ** -0.5)
    for out in outs:
        assert_close(to_np(out)[rows].astype(np.float32), ref, F16_ATOL, F16_RTOL, "noalloc and workspace")


@pytest.mark.parametrize("S,H,Hkv,D,table", [(17000, 8, 2, 64, 6000), (9000, 4, 2, 96, 6000), (5000, 16, 1, 128, 6000),
                                             (300, 4, 4, 80, 6000)])
def test_stream_slices_of_many_rows(vkv, oracle, cuda, S, H, Hkv, D, table):
    """Equal slices over several launches (8 192 rows each) that share the partials and
    the rows' places, several rows to a thread of the scan, prefixes too long for two
    stages per wave, fewer slices than rows, rows without keys: every row against the
    oracle, and the same bits twice."""
    import torch
    rng = np.random.default_rng(S)
    ctx = rng.integers(0, 40, S)
    ctx[[0, S // 2, S - 1]] = [700, 1500, 333]
    lay, (k, v), q = _case(rng, H, Hkv, D, 16, ctx, table)
    outs = [torch.full((S, H, D), 7.0, dtype=torch.float16, device=cuda) for _ in range(2)]
    args = (to_dev(q, cuda), to_dev(k, cuda), to_dev(v, cuda), to_dev(lay.block_tables, cuda),
            to_dev(lay.context_lens, cuda), float(D) ** -0.5)
    for out in outs:
        vkv.paged_decode(out, *args)
    torch.cuda.synchronize()
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))
    ref = oracle.paged_decode(q.astype(np.float32), np.nan_to_num(k).view(np.uint16), np.nan_to_num(v).view(np.uint16),
                              lay.block_tables, lay.context_lens, float(D) ** -0.5, nthreads=8)
    assert_close(to_np(outs[0]).astype(np.float32), ref, F16_ATOL, F16_RTOL, f"{S} rows in slices")


@pytest.mark.parametrize("table", [1024, 6000], ids=["rows", "partitions"])
@pytest.mark.parametrize("H,Hkv,bs", [(28, 4, 32), (32, 8, 16), (8, 8, 16), (16, 2, 64)])
def test_stream_fp8_edges_vs_oracle(vkv, oracle, cuda, H, Hkv, bs, table):
    """FP8 caches at head_dim 128: unattended slots hold the NaN code and NaN scales."""
    import torch
    D = 128
    rng = np.random.default_rng(H + bs)
    lay, (k, v), q = _case(rng, H, Hkv, D, bs, CONTEXTS, table)
    used = ~np.isnan(k[:, :, 0, 0].astype(np.float32))
    N = lay.num_blocks
    codes = [np.zeros((N, bs, Hkv, D), np.uint8) for _ in range(2)]
    scales = [np.zeros((N, bs, Hkv), np.float32) for _ in range(2)]
    oracle.reshape_and_cache(np.nan_to_num(k).view(np.uint16).reshape(-1, Hkv, D),
                             np.nan_to_num(v).view(np.uint16).reshape(-1, Hkv, D), *codes,
                             np.arange(N * bs, dtype=np.int32), *scales)
    scale = float(D) ** -0.5
    ref = oracle.paged_decode(q.astype(np.float32), *codes, lay.block_tables, lay.context_lens, scale,
                              key_scales=scales[0], value_scales=scales[1])
    for c, s in zip(codes, scales):
        c[~used] = 0x7F
        s[~used] = np.nan
    out = torch.full((len(CONTEXTS), H, D), 7.0, dtype=torch.float16, device=cuda)
    vkv.paged_decode(out, to_dev(q, cuda), to_dev(codes[0], cuda), to_dev(codes[1], cuda), to_dev(lay.block_tables, cuda),
                     to_dev(lay.context_lens, cuda), scale, key_scales=to_dev(scales[0], cuda),
                     value_scales=to_dev(scales[1], cuda))
    torch.cuda.synchronize()
    assert_close(to_np(out).astype(np.float32), ref, F16_ATOL, F16_RTOL, f"FP8 {H}/{Hkv}/bs{bs}")


@pytest.mark.parametrize("table", [1024, 6000], ids=["rows", "slices"])
@pytest.mark.parametrize("H,Hkv,bs", [(14, 2, 16), (34, 2, 24), (4, 4, 1), (64, 2, 32)])
def test_stream_fp32_edges_vs_oracle(vkv, oracle, cuda, H, Hkv, bs, table):
    """All in fp32 at head_dim 64 (fp32 bounds: weights, sums and products stay fp32)."""
    import torch
    from helpers import F32_ATOL, F32_RTOL
    D = 64
    rng = np.random.default_rng(H + bs)
    lay, (k, v), q = _case(rng, H, Hkv, D, bs, CONTEXTS, table)
    # (full fp32 mantissas; the unattended slots stay NaN)
    k, v, q = ((x.astype(np.float32) * np.float32(1.0001)) for x in (k, v, q))
    scale = -float(D) ** -0.5 if bs == 24 else float(D) ** -0.5
    ref = oracle.paged_decode(q, np.nan_to_num(k), np.nan_to_num(v), lay.block_tables, lay.context_lens, scale)
    for size in (0, 64):
        out = torch.full((len(CONTEXTS), H, D), 7.0, dtype=torch.float32, device=cuda)
        vkv.paged_decode(out, to_dev(q, cuda), to_dev(k, cuda), to_dev(v, cuda), to_dev(lay.block_tables, cuda),
                         to_dev(lay.context_lens, cuda), scale, partition_size=size)
        torch.cuda.synchronize()
        assert_close(to_np(out), ref, F32_ATOL, F32_RTOL, f"fp32 {H}/{Hkv}/bs{bs} size {size}")


# All in fp32 at head_dim 64, groups of 1 to 5: by pairs, group and table the call
# runs on the VALU kernel, as one workgroup per (row, kv head) or in equal slices
@pytest.mark.parametrize("bs", [16, 24])  # (24: the generic kernel instead of the VALU one)
@pytest.mark.parametrize("table", [128, 256, 512, 1024, 2048, 6000])
@pytest.mark.parametrize("S,H,Hkv", [(12, 8, 8), (12, 4, 2), (12, 8, 2), (12, 10, 2), (70, 4, 4), (70, 16, 4), (300, 4, 4),
                                     (300, 8, 4)])
def test_fp32_small_groups_vs_oracle(vkv, oracle, cuda, S, H, Hkv, table, bs):
    """Against the oracle, and the fused append against the two calls bit for bit."""
    import torch
    from helpers import F32_ATOL, F32_RTOL
    D = 64
    rng = np.random.default_rng(S + H + table)
    ctx = rng.integers(1, min(table, 700 if S < 100 else 60) + 1, S)
    ctx[:2] = [min(table, 900), 1]
    lay, (k, v), q = _case(rng, H, Hkv, D, bs, ctx, table)
    k, v, q = ((x.astype(np.float32) * np.float32(1.0001)) for x in (k, v, q))
    ref = oracle.paged_decode(q, np.nan_to_num(k), np.nan_to_num(v), lay.block_tables, lay.context_lens, D ** -0.5)
    rest = (to_dev(lay.block_tables, cuda), to_dev(lay.context_lens, cuda), D ** -0.5)
    kc, vc = to_dev(k, cuda), to_dev(v, cuda)
    out = torch.full((S, H, D), 7.0, device=cuda)
    vkv.paged_decode(out, to_dev(q, cuda), kc, vc, *rest)
    torch.cuda.synchronize()
    assert_close(to_np(out), ref, F32_ATOL, F32_RTOL, f"fp32 {S} rows {H}/{Hkv}, table {table}")
    slots = lay.slots(lay.context_lens - 1, np.arange(S))
    new = [to_dev(rng.standard_normal((S, Hkv, D), dtype=np.float32), cuda) for _ in range(2)]
    two = [torch.empty_like(out), kc.clone(), vc.clone()]
    vkv.reshape_and_cache(*new, two[1], two[2], to_dev(slots, cuda))
    vkv.paged_decode(two[0], to_dev(q, cuda), two[1], two[2], *rest)
    vkv.paged_decode_append(out, to_dev(q, cuda), kc, vc, *rest, *new, to_dev(slots, cuda))
    torch.cuda.synchronize()
    for a, b in zip((out, kc, vc), two):
        assert torch.equal(a.view(torch.int32), b.view(torch.int32))


@pytest.mark.parametrize("dtype", ["f16", "f32"])
@pytest.mark.parametrize("D", [64, 80, 112, 128])
def test_stream_query_rows_of_any_alignment(vkv, cuda, D, dtype):
    """Queries at an odd element and with an odd row stride: bit for bit the
    result of the same queries in aligned rows."""
    import torch
    if dtype == "f32" and D != 64:
        pytest.skip("fp32 streams at head_dim 64 only")
    H, Hkv, bs = 6, 2, 16
    rng = np.random.default_rng(D)
    lay, (k, v), q = _case(rng, H, Hkv, D, bs, CONTEXTS, 1024)
    t = np.float16 if dtype == "f16" else np.float32
    q, n = to_dev(q.astype(t), cuda), len(CONTEXTS)
    odd = torch.empty(1 + n * (H * D + 3), dtype=q.dtype, device=cuda)
    odd = odd[1:].view(n, H * D + 3)[:, :H * D].unflatten(1, (H, D))
    odd.copy_(q)
    assert odd.data_ptr() % 16 != 0 and odd.stride(0) % 2 == 1
    rest = (to_dev(k.astype(t), cuda), to_dev(v.astype(t), cuda), to_dev(lay.block_tables, cuda),
            to_dev(lay.context_lens, cuda), float(D) ** -0.5)
    outs = [torch.zeros((n, H, D), dtype=q.dtype, device=cuda) for _ in range(2)]
    vkv.paged_decode(outs[0], q, *rest)
    vkv.paged_decode(outs[1], odd, *rest)
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1])
