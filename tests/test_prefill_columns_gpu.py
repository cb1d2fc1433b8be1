"""tb_paged_prefill_columns (prefill rows of any context, column tiles) against the oracle
through the C ABI: attention within 2e-2 at fp16 / bf16 against the oracle in the same
dtype, within 1e-5 at fp32.

Sizes where it can go wrong: contexts around its 64-position chunks and 128-column tiles
(one column past a tile, one position past a chunk), more chunks than one load of block
ids covers (64), 1 to 16 query heads per kv head, block sizes 16 to 64, cached prefixes,
stale NaN slots, steps with decode rows and short tails beside it, split rows merged by
this call or by the work items' one, RoPE, and the call without a workspace."""
import pytest
import torch

from oracle import reference_path as ref
from test_prefill_columns_work import both_routes
from test_prefill_stream_gpu import DEV, TOL, case
from tinybatch_amd import layer_ops, metadata as step_metadata, ops
from tinybatch_amd.kv_cache import PagedKVCache
from tinybatch_amd.metadata import TILE_PARTITION, build_step_metadata
from tinybatch_amd.model import rope_tables

pytestmark = pytest.mark.gpu


def metadata(c, rows=None):
    dt, Hq, Hkv, D = c["dtype"], c["Hq"], c["Hkv"], c["D"]
    route = ops.columns_route(dt, Hq, Hkv, D, c["BS"], DEV)
    return build_step_metadata(c["pos"], c["slices"], c["tables"], c["ctx"], block_size=c["BS"], num_blocks=c["NB"],
                               partition_tokens=ops.partition_tokens(dt, D),
                               rows_per_item=rows or ops.rows_per_item(dt, Hq, Hkv), tile_prefill=True,
                               columns_route=route).to(DEV)


def check(c, **kw):
    want = ref.attention(c["q"], c["pool"], c["slices"], c["tables"], c["ctx"], c["Hq"], c["Hkv"])
    meta = metadata(c)
    assert meta.num_columns_work and not meta.num_prefill_tiles
    out = ops.paged_attention(c["q"].to(DEV), c["pool"].to(DEV), meta, num_heads=c["Hq"], **kw)
    torch.cuda.synchronize()
    got = out.cpu()
    assert torch.isfinite(got).all()
    torch.testing.assert_close(got.float(), want.float(),
                               **(dict(atol=1e-5, rtol=0) if c["dtype"] == torch.float32 else TOL))
    return meta


@pytest.mark.parametrize("Hq,Hkv,D,dtype", [(14, 2, 64, torch.float16), (14, 2, 64, torch.bfloat16),
                                            (32, 8, 128, torch.bfloat16), (32, 8, 128, torch.float16),
                                            (4, 4, 64, torch.bfloat16), (16, 1, 128, torch.float16),
                                            (14, 2, 64, torch.float32), (32, 8, 128, torch.float32),
                                            (4, 4, 64, torch.float32)])
def test_edges_of_tiles_and_chunks(Hq, Hkv, D, dtype):
    qlens = [16, 18, 19, 63, 64, 65, 129]
    check(case(1, Hq, Hkv, D, 16, dtype, qlens, [0, 45, 46, 0, 1, 128, 300]))


@pytest.mark.parametrize("BS", [16, 32, 64])
def test_long_contexts_of_few_rows(BS):
    # 4097 .. 4300 positions: few rows, so that they are split
    meta = check(case(2, 14, 2, 64, BS, torch.bfloat16, [16, 40], [4081, 4260]))
    assert meta.num_split_rows == 56
    check(case(3, 2, 1, 64, BS, torch.float16, [4200], [0]))
    check(case(3, 2, 1, 64, BS, torch.float32, [30], [2100]))


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_rows_of_one_and_two_partitions_in_one_tile(dtype):
    """Rows that cross the first partition's end inside a tile of 18 rows: the second
    partition's workgroup leaves the earlier rows alone."""
    c = case(9, 14, 2, 64, 16, dtype, [2500], [0])
    meta = check(c)
    assert 0 < meta.num_split_rows < 2500


def test_whole_rows_when_the_step_fills_the_gpu():
    meta = check(case(4, 14, 2, 64, 16, torch.bfloat16, [700] * 8 + [900], [0] * 9))
    assert meta.num_split_rows == 0


@pytest.mark.parametrize("D,Hq,Hkv,dtype", [(64, 14, 2, torch.bfloat16), (128, 32, 8, torch.bfloat16),
                                            (64, 14, 2, torch.float32), (128, 32, 8, torch.float32)])
def test_beside_decode_rows_and_short_tails(D, Hq, Hkv, dtype):
    """Split rows of both kernels merged by the work items' call."""
    c = case(5, Hq, Hkv, D, 16, dtype, [90, 1, 5, 33, 1, 1], [1500, 700, 600, 0, 63, 1100])
    meta = check(c)
    assert meta.num_work_items and meta.num_split_rows > 90


def test_without_a_workspace_and_scratch_no_larger_than_the_tiles():
    c = case(6, 14, 2, 64, 16, torch.float16, [100, 20], [1900, 0])
    out = torch.empty(120, 14 * 64, dtype=torch.float16, device=DEV)
    check(c, noalloc=True, out=out)
    # a step whose finer split would outgrow the static scratch keeps the tiles' 1024 positions
    n = 2000
    c = case(7, 14, 2, 64, 16, torch.float16, [n], [6000])
    meta = metadata(c)
    scratch = meta.total_partitions * 14 * 66 * 4
    assert scratch <= 32 << 20 or meta.total_partitions <= sum(-(-(6000 + r + 1) // TILE_PARTITION) for r in range(n))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rope_equals_rotating_first(dtype):
    c = case(8, 14, 2, 64, 16, dtype, [50, 130], [700, 0])
    cos, sin = rope_tables(64, 1e6, 4096, DEV)
    meta = metadata(c)
    pool, q = c["pool"].to(DEV), c["q"].to(DEV)
    pos = torch.tensor(c["pos"], device=DEV)
    kv = torch.zeros(q.shape[0], 2, 64, dtype=q.dtype, device=DEV)
    qkv = torch.cat([q, kv], 1).reshape(q.shape[0], -1)
    rotated, _ = layer_ops.rope_qk(qkv, pos, cos, sin, 14, 2, 64)
    got = ops.paged_attention(q, pool, meta, num_heads=14, rope=ops.Rope(cos, sin))
    want = ops.paged_attention(rotated, pool, meta, num_heads=14)
    assert torch.equal(got, want)


def test_fused_append_refused_beside_column_rows():
    """tb_paged_prefill would append its own rows and the column tiles read unwritten ones."""
    meta = both_routes().to(DEV)
    pool = torch.zeros(70, 2, 2, 16, 64, dtype=torch.bfloat16, device=DEV)
    q = torch.zeros(1100, 14, 64, dtype=torch.bfloat16, device=DEV)
    kv = torch.ones(1100, 2, 64, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(ValueError, match="fused append"):
        ops.paged_attention(q, pool, meta, num_heads=14, k_new=kv, v_new=kv)
    assert not pool.any()


@pytest.mark.parametrize("Hq,Hkv", [(28, 2), (4, 4), (2, 1)])
def test_metadata_of_other_heads(Hq, Hkv, monkeypatch):
    """Metadata built for 14 / 2 heads serves a call with other heads: a list of its own,
    uploaded on the first call and not while a graph is captured."""
    c = case(10, Hq, Hkv, 64, 16, torch.bfloat16, [100, 20], [900, 0])
    want = ref.attention(c["q"], c["pool"], c["slices"], c["tables"], c["ctx"], Hq, Hkv)
    meta = metadata({**c, "Hq": 14, "Hkv": 2}, rows=1)
    q, pool = c["q"].to(DEV), c["pool"].to(DEV)
    out = torch.full((120, Hq * 64), float("nan"), dtype=torch.bfloat16, device=DEV)
    with monkeypatch.context() as m, pytest.raises(RuntimeError, match="call once"):
        m.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
        ops.paged_attention(q, pool, meta, num_heads=Hq, out=out)
    for _ in range(2):
        got = ops.paged_attention(q, pool, meta, num_heads=Hq, out=out).cpu()
        torch.testing.assert_close(got.float(), want.float(), **TOL)
    assert len(meta.columns_other) == 1


@pytest.mark.parametrize("Hq,Hkv,D,dtype", [(14, 2, 64, torch.bfloat16), (32, 8, 128, torch.float16),
                                            (14, 2, 64, torch.float32), (32, 8, 128, torch.float32)])
@pytest.mark.parametrize("sign", [-1, 0])
def test_negative_and_zero_scale(Hq, Hkv, D, dtype, sign):
    """The scores of -q at the scale's size, or uniform weights: masked positions stay masked."""
    c = case(11, Hq, Hkv, D, 16, dtype, [70, 20], [200, 0])
    want = ref.attention(sign * c["q"], c["pool"], c["slices"], c["tables"], c["ctx"], Hq, Hkv)
    got = ops.paged_attention(c["q"].to(DEV), c["pool"].to(DEV), metadata(c), num_heads=Hq, scale=sign * D ** -0.5)
    torch.testing.assert_close(got.cpu().float(), want.float(),
                               **(dict(atol=1e-5, rtol=0) if dtype == torch.float32 else TOL))


@pytest.mark.parametrize("dtype,qlens,cached,columns", [(torch.bfloat16, [40, 1, 1], [0, 300, 700], False),
                                                        (torch.bfloat16, [700, 3], [0, 50], False),
                                                        (torch.bfloat16, [1500] * 4 + [1], [0] * 4 + [200], True),
                                                        (torch.float32, [20, 1], [100, 300], False),
                                                        (torch.float32, [300] * 6, [0] * 6, True)])
def test_cache_takes_the_faster_route(dtype, qlens, cached, columns):
    """PagedKVCache.attention on both sides of the rule, against the oracle."""
    c = case(12, 14, 2, 64, 16, dtype, qlens, cached)
    want = ref.attention(c["q"], c["pool"], c["slices"], c["tables"], c["ctx"], 14, 2)
    cache = PagedKVCache(1, c["NB"], 16, 2, 64, DEV, dtype)
    cache.pools[0].copy_(c["pool"])
    pos = torch.tensor(c["pos"], device=DEV)
    got = cache.attention(0, c["q"].to(DEV), pos, c["slices"], c["tables"], c["ctx"])
    meta = cache.step_metadata(pos, c["slices"], c["tables"], c["ctx"], cache.rows_per_item(14), num_heads=14)
    assert bool(meta.num_columns_work) == columns
    torch.testing.assert_close(got.cpu().float(), want.float(),
                               **(dict(atol=1e-5, rtol=0) if dtype == torch.float32 else TOL))


@pytest.mark.parametrize("Hq,Hkv,D,dtype,qlens,cached,sets", [
    (14, 2, 64, torch.bfloat16, [16, 40], [4081, 8300], 2), (14, 2, 64, torch.float16, [16, 40], [4081, 8300], 2),
    (32, 8, 128, torch.float16, [33, 16], [8500, 4200], 2),
    (8, 8, 64, torch.bfloat16, [4250], [0], 1), (32, 8, 128, torch.bfloat16, [1100], [4300], 1),
    (14, 2, 64, torch.float32, [30, 18], [2100, 6300], 1), (32, 8, 128, torch.float32, [33], [4200], 1)])
def test_block_ids_of_a_part_past_the_first_64_chunks(Hq, Hkv, D, dtype, qlens, cached, sets, monkeypatch):
    """Rows kept whole, so that a workgroup walks more than 64 chunks (fp32: of 32 positions) and
    reads block ids again; with one set of waves, and with two (up to 256 entries)."""
    monkeypatch.setattr(step_metadata, "columns_partition", lambda *a: 1 << 20)
    c = case(15, Hq, Hkv, D, 16, dtype, qlens, cached)
    meta = check(c)
    longest = max(c["ctx"])
    assert meta.num_split_rows == 0 and -(-longest // (32 if dtype == torch.float32 else 64)) > 65
    assert dtype == torch.float32 or (meta.num_columns_work <= 256) == (sets == 2)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("cached,part", [(0, 1 << 20), (300, 512)])
def test_one_set_of_waves_at_head_dim_128(dtype, cached, part, monkeypatch):
    """More than 256 entries, rows whole and split, an odd last tile."""
    monkeypatch.setattr(step_metadata, "columns_partition", lambda *a: part)
    meta = check(case(16, 32, 8, 128, 16, dtype, [1237], [cached]))
    assert meta.num_columns_work > 256 and (meta.num_split_rows > 0) == (part == 512)


@pytest.mark.parametrize("Hq,Hkv,D", [(14, 2, 64), (32, 8, 128)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("log2_p,n,whole", [(14, 40, False), (16, 40, True), (16, 600, True), (18, 600, True),
                                            (22, 600, False)])
def test_one_dominant_key(Hq, Hkv, D, dtype, log2_p, n, whole, monkeypatch):
    """One key of weight 1 and 3999 of 2^-14 .. 2^-22, from 2^-15 on subnormal in fp16: the products
    with their values (ones beside a zero) and the row sum count them alike (a sum that dropped
    them would be 6% off at 2^-16). Bound: all weights are rounded the same way, by up to half a
    unit of 2^-24 in fp16, and the outputs by 2^-9 in bf16."""
    if whole:
        monkeypatch.setattr(step_metadata, "columns_partition", lambda *a: 1 << 20)
    bound = 2.0 ** (log2_p - 25) + 2.0 ** -8
    ctx = 4000
    k = torch.full((ctx, Hkv, D), 0.0)
    k[1:, :, 0] = -log2_p * 0.6931471805599453 / 8
    v = torch.ones(ctx, Hkv, D)
    v[0] = 0
    q = torch.zeros(n, Hq, D)
    q[:, :, 0] = 8 * D ** 0.5
    pool = torch.stack([k, v]).reshape(2, ctx // 16, 16, Hkv, D).permute(1, 0, 3, 2, 4).contiguous().to(dtype)
    route = ops.columns_route(dtype, Hq, Hkv, D, 16, DEV)
    meta = build_step_metadata(list(range(ctx - n, ctx)), [(0, n)], [list(range(ctx // 16))], [ctx], block_size=16,
                               num_blocks=ctx // 16, partition_tokens=256, columns_route=route).to(DEV)
    got = ops.paged_attention(q.to(DEV, dtype), pool.to(DEV), meta, num_heads=Hq).cpu().double().view(n, Hq, D)
    score = (k[:, 0, 0].to(dtype).double() * q[0, 0, 0].to(dtype).double() * D ** -0.5)
    weights = torch.exp(score - score[0])
    for row in (0, n // 2, n - 1):
        w = weights[1:ctx - n + row + 1].sum().item()
        assert ((got[row] * (1 + w) / w - 1).abs() <= bound).all(), (row, got[row, 0, 0], w / (1 + w))


@pytest.mark.parametrize("Hq,Hkv,D,dtype", [(14, 2, 64, torch.bfloat16), (32, 8, 128, torch.float16),
                                            (14, 2, 64, torch.float32), (32, 8, 128, torch.float32)])
def test_non_finite_keys_and_values_of_the_context(Hq, Hkv, D, dtype):
    """A NaN key reaches every row that sees it and no other; 64 positions of -inf scores weigh
    nothing; a NaN value of the cached context reaches every row, and no other sequence."""
    c = case(17, Hq, Hkv, D, 16, dtype, [60, 60, 60, 60], [300, 300, 300, 0])
    c["q"][:, :, 0] = 1.0
    at = lambda s, p: (c["tables"][s][p // 16], p % 16)
    b, o = at(0, 330)
    c["pool"][b, 0, :, o, 1] = float("nan")                 # rows 30 .. 59 of sequence 0 see it
    for p in range(64, 128):
        b, o = at(1, p)
        c["pool"][b, 0, :, o, 0] = float("-inf")
    b, o = at(2, 200)
    c["pool"][b, 1, :, o] = float("nan")
    want = ref.attention(c["q"], c["pool"], c["slices"], c["tables"], c["ctx"], Hq, Hkv)
    got = ops.paged_attention(c["q"].to(DEV), c["pool"].to(DEV), metadata(c), num_heads=Hq).cpu()
    assert got[:30].isfinite().all() and got[30:60].isnan().all() and got[120:180].isnan().all()
    tol = dict(atol=1e-5, rtol=0) if dtype == torch.float32 else TOL
    clean = {**c, "pool": c["pool"].clone()}
    b, o = at(0, 330)
    clean["pool"][b, 0, :, o, 1] = 0.0                      # rows that do not see it: any finite key there
    first = ref.attention(c["q"][:60], clean["pool"], [(0, 60)], c["tables"][:1], c["ctx"][:1], Hq, Hkv)
    torch.testing.assert_close(got[:30].float(), first[:30].float(), **tol)
    for rows in (slice(60, 120), slice(180, 240)):
        torch.testing.assert_close(got[rows].float(), want[rows].float(), **tol)
