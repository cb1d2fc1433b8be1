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
from tinybatch_amd import layer_ops, ops
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
def test_more_chunks_than_one_read_of_block_ids(BS):
    # 4097 .. 4300 positions: chunks 64 .. 67; few rows, so the rows are split as well
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
