"""Attention of long query windows (more than 64 rows per KV head): the kernel of
attn_prefill.hip against the fp64 oracle, at the edges of its row tiles (16 and 32 rows a
wave, four waves a workgroup), of its 64-key blocks, of its 64-entry table window and of the
block ranges a workgroup takes.  A chosen split always runs it; with the automatic one, calls
over few blocks stay with the verify or decode kernel (test_calls_over_few_blocks).

Bound: bf16 and fp16 inputs reach the matrix cores exactly, the weights as fp16 pairs (2^-22)
and the sums are binary32, so outputs of values of order 1 lie within 1e-4 of the oracle; 2e-3
is the bound of the repository's other attention tests."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import krill_amd  # noqa: E402
from oracle import oracle as O  # noqa: E402
from tests.kvutil import Filled, Rising, i32, oracle_attention, rand_bits, to_dev  # noqa: E402

pytestmark = pytest.mark.gpu
ATOL = 2e-3


def _run(mode, D, H, R, lens, Lq, dt="bf16", scale=None, split_blocks=1, out_dtype=torch.float32, q_mul=1.0, seed=0):
    rng = np.random.default_rng(seed)
    pool = krill_amd.KVPool(1, H, D, sum((n + 63) // 64 for n in lens) + 4, mode, dt, free_list_seed=7)
    if split_blocks:  # (one block a range, if not told otherwise)
        pool.set_option(krill_amd._lib.OPT_SPLIT_BLOCKS, split_blocks)
    f = Filled(pool, lens, rng, dt, max_chunk=500)
    tables, n, _ = f.tables()
    scale = 1.0 / np.sqrt(D) if scale is None else scale
    q = rand_bits(rng, (len(lens), H * R, Lq, D), dt, scale=q_mul)
    got = pool.attention(0, to_dev(q, dt), tables, n, max(lens), float(scale), out_dtype)
    torch.cuda.synchronize()
    ref = oracle_attention(pool, f, 0, q, dt, scale)
    pool.close()
    return got.double().cpu().numpy(), ref


@pytest.mark.parametrize("mode", ["affine_g64", "ref_row"])
@pytest.mark.parametrize("D,R,Lq", [(64, 5, 13), (64, 8, 17), (128, 5, 13), (128, 2, 64), (256, 2, 33), (256, 3, 43),
                                    (512, 8, 9), (512, 1, 65)])
def test_row_and_block_edges(mode, D, R, Lq):
    """65 (one row past four 16-row tiles) to 136 rows; sequences ending at, one before and one
    past a block edge, one holding only its new rows, one empty of older blocks."""
    print(f"\ncase long_window mode={mode} D={D} R={R} Lq={Lq}", flush=True)
    got, ref = _run(mode, D, 2, R, [Lq, 127, 128, 129, 300], Lq, dt="f16" if R == 8 else "bf16", seed=D + R)
    assert np.abs(got - ref).max() <= ATOL


@pytest.mark.parametrize("mode", ["affine_g64", "ref_row"])
@pytest.mark.parametrize("D,split", [(64, 0), (128, 64), (128, 3), (256, 2), (512, 2)])
def test_ranges_across_sequences(mode, D, split):
    """Ranges that begin and end inside sequences (partials merged), whole sequences inside one
    range, and (automatic split, one KV head) ranges over several sequences."""
    print(f"\ncase long_window_ranges mode={mode} D={D} split={split}", flush=True)
    got, ref = _run(mode, D, 1, 3, [40, 700, 65, 1300, 64, 90], 33, split_blocks=split, seed=D)
    assert np.abs(got - ref).max() <= ATOL


def _ranges(pool, B, Hq, Lq, mx, tile):
    """Block ranges per row group, from the workspace: a slot per (KV head, row group) and range
    or sequence, `tile` rows of D values and two more each."""
    groups = (Hq // pool.num_kv_heads * Lq + tile - 1) // tile
    slots = pool.workspace_size(B, Hq, Lq, mx) // (tile * (pool.head_dim + 2) * 4)
    return slots // (pool.num_kv_heads * groups) - B


def _rows_against_short_windows(pool, lens, Lq, R, seed, at, ranges, tile=32):
    """Rows `at` (offsets into the new rows) of a long window against the same rows as windows of
    two, which run on the decode kernel (two kernels, each within 1e-4 of fp64)."""
    rng = np.random.default_rng(seed)
    H, D, dt = pool.num_kv_heads, pool.head_dim, "bf16"
    f = Filled(pool, lens, rng, dt, max_chunk=4000)
    tables, n, _ = f.tables()
    assert _ranges(pool, len(lens), H * R, Lq, max(lens), tile) == ranges
    q = to_dev(rand_bits(rng, (len(lens), H * R, Lq, D), dt), dt)
    got = pool.attention(0, q, tables, n, max(lens), 1.0 / np.sqrt(D)).cpu()
    for j in at:
        m = i32([T - Lq + j for T in lens])
        want = pool.attention(0, q[:, :, j - 2:j].contiguous(), tables, m, max(lens), 1.0 / np.sqrt(D)).cpu()
        assert (got[:, :, j - 2:j] - want).abs().max() <= 2e-4
    pool.close()


@pytest.mark.parametrize("mode", ["affine_g64", "ref_row"])
@pytest.mark.parametrize("lens,Lq,R", [([72 * 64 - 5], 72 * 64 - 5, 3), ([50 * 64 - 9, 36 * 64], 2048, 4)])
def test_range_longer_than_the_table_window(mode, lens, Lq, R):
    """So many row-group workgroups that each takes its rows' whole range, past the 64 table
    entries a workgroup holds at once: a prompt of 72 blocks, and a second sequence whose blocks
    51 to 86 of the range cross the 64th."""
    print(f"\ncase long_window_table mode={mode} lens={lens}", flush=True)
    pool = krill_amd.KVPool(1, 8, 128, sum((T + 63) // 64 for T in lens) + 4, mode, "bf16", free_list_seed=9)
    _rows_against_short_windows(pool, lens, Lq, R, 3, (64, 1000, Lq), ranges=1)


@pytest.mark.parametrize("mode", ["affine_g64", "ref_row"])
@pytest.mark.parametrize("D,R,Lq,T,ranges,tile", [(128, 5, 1000, 5000, 3, 32), (256, 2, 700, 4700, 5, 16)])
def test_more_rounds_of_ranges(mode, D, R, Lq, T, ranges, tile):
    """Row groups that fill under three quarters of the chip over many blocks: two rounds of
    ranges (one round: 1 and 2)."""
    print(f"\ncase long_window_rounds mode={mode} D={D}", flush=True)
    pool = krill_amd.KVPool(1, 8, D, (T + 63) // 64 + 4, mode, "bf16", free_list_seed=9)
    _rows_against_short_windows(pool, [T], Lq, R, 5, (2, 500, Lq), ranges, tile)


@pytest.mark.parametrize("mode", ["affine_g64", "ref_row"])
@pytest.mark.parametrize("scale", [0.0, -0.05, 1.0])
def test_scales(mode, scale):
    print(f"\ncase long_window_scale mode={mode} scale={scale}", flush=True)
    got, ref = _run(mode, 128, 1, 4, [150, 400], 20, scale=scale, seed=11)
    assert np.abs(got - ref).max() <= ATOL


@pytest.mark.parametrize("mode", ["affine_g64", "ref_row"])
def test_queries_beyond_fp16(mode):
    """bf16 queries past fp16's range: scaled by 2^-k, their scores by 2^k."""
    print(f"\ncase long_window_qrange mode={mode}", flush=True)
    got, ref = _run(mode, 64, 1, 4, [130, 200], 18, scale=2.0 ** -18, q_mul=1e6, seed=13)
    assert np.abs(got - ref).max() <= ATOL


@pytest.mark.parametrize("D", [128, 512])
@pytest.mark.parametrize("out", [torch.bfloat16, torch.float16])
def test_low_precision_output(D, out):
    print(f"\ncase long_window_out D={D} {out}", flush=True)
    got, ref = _run("affine_g64", D, 1, 4, [40, 333], 19, out_dtype=out, split_blocks=2, seed=17)
    ulp = 2.0 ** -8 if out is torch.bfloat16 else 2.0 ** -11
    assert (np.abs(got - ref) - ulp * np.abs(ref)).max() <= ATOL


@pytest.mark.parametrize("mode,D,H,R,Lq,lens,ranges", [
    ("affine_g64", 256, 8, 2, 100, [400], 8),       # 7 blocks, at most 1.5 a range: verify kernel, one workgroup a CU
    ("affine_g64", 256, 8, 2, 200, [500] * 4, 9),   # 32 blocks: this kernel, two
    ("affine_g64", 256, 8, 2, 40, [40, 33 + 7], 32),  # one block each: this kernel
    ("ref_row", 256, 8, 2, 100, [190], None),
    ("ref_row", 256, 8, 2, 100, [420, 100, 333], None),
    ("affine_g64", 128, 8, 5, 48, [148], None),
    ("affine_g64", 128, 8, 5, 48, [48], None),
    ("affine_g64", 128, 8, 5, 60, [160, 60], None),  # more than 4096 rows
    ("ref_row", 128, 8, 5, 17, [117], None),
    ("ref_row", 128, 8, 5, 48, [900], None),
    ("affine_g64", 512, 2, 8, 30, [130, 30], None),  # decode kernel
    ("affine_g64", 512, 2, 8, 130, [130, 161], None),  # more than 4096 rows, over a quarter block a range
    ("ref_row", 512, 2, 8, 30, [1030, 700], None),
])
def test_calls_over_few_blocks(mode, D, H, R, Lq, lens, ranges):
    """Either side of each line between this kernel and the one that starts sooner."""
    print(f"\ncase long_window_few mode={mode} D={D} R={R} Lq={Lq} lens={lens}", flush=True)
    if ranges is not None:
        pool = krill_amd.KVPool(1, H, D, 4, mode, "bf16")
        assert _ranges(pool, len(lens), H * R, Lq, max(lens), 16) == ranges
        pool.close()
    got, ref = _run(mode, D, H, R, lens, Lq, split_blocks=0, seed=D + Lq)
    assert np.abs(got - ref).max() <= ATOL


def test_many_query_heads_per_kv_head():
    """One new row, 70 query heads per KV head: the same kernel, decode's plan."""
    print("\ncase long_window_mqa", flush=True)
    got, ref = _run("affine_g64", 64, 1, 70, [1, 64, 500], 1, seed=19)
    assert np.abs(got - ref).max() <= ATOL


@pytest.mark.parametrize("mode", ["affine_g64", "ref_row"])
def test_batch_past_one_wave_of_lengths(mode):
    """70 sequences: lengths past the 64 a wave holds in one register."""
    print(f"\ncase long_window_batch mode={mode}", flush=True)
    rng = np.random.default_rng(23)
    lens = [int(x) for x in rng.integers(33, 200, size=70)]
    got, ref = _run(mode, 64, 1, 2, lens, 33, seed=29)
    assert np.abs(got - ref).max() <= ATOL


def test_blocks_at_the_pools_end():
    """head_dim 64, affine: 128 metadata words a block for 256 threads, in a pool whose last
    layer's last block is attended (that no load leaves a block's region is asserted where the
    kernel is compiled)."""
    print("\ncase long_window_pool_end", flush=True)
    rng = np.random.default_rng(31)
    lens, H, R, D, Lq = [128, 200, 64], 2, 4, 64, 20
    pool = krill_amd.KVPool(2, H, D, sum((n + 63) // 64 for n in lens), "affine_g64", "bf16", free_list_seed=1)
    f = Filled(pool, lens, rng, "bf16", layers=(1,))
    tables, n, _ = f.tables()
    assert int(tables.max()) == pool.num_blocks - 1
    q = rand_bits(rng, (len(lens), H * R, Lq, D), "bf16")
    got = pool.attention(1, to_dev(q, "bf16"), tables, n, max(lens), 0.125)
    torch.cuda.synchronize()
    ref = oracle_attention(pool, f, 1, q, "bf16", 0.125)
    pool.close()
    assert np.abs(got.double().cpu().numpy() - ref).max() <= ATOL


@pytest.mark.parametrize("mode", ["affine_g64", "ref_row"])
@pytest.mark.parametrize("D,split", [(64, 64), (128, 64), (128, 3), (256, 64), (512, 64), (512, 2)])
@pytest.mark.parametrize("rise,s_v", [(2.1, 0), (2.5, 0), (2.9, 0), (7.5, 0), (0.0, 3000.0), (2.9, 60000.0)])
def test_large_value_scales(mode, D, split, rise, s_v):
    """Weights p s_v stay finite in fp16 for every fp16 V scale, also while the running reference
    is not raised (whole sequences in one range, and ranges of 2 or 3 blocks).

    Bound: scores of up to 7.5 * 9 = 68 in binary32 err by a few 2^-18, so weights by a few 2^-18
    of themselves, outputs by that of the largest |V|: 2^-14 of it."""
    if s_v and mode == "ref_row":
        pytest.skip("row mode holds dequantized V values in fp16")
    print(f"\ncase long_window_large_v mode={mode} D={D} split={split} rise={rise} s_v={s_v}", flush=True)
    rng = np.random.default_rng(37)
    R, Lq, lens = 5, 20, [600, 40, 64 * 4]
    pool = krill_amd.KVPool(1, 1, D, 24, mode, "f16", free_list_seed=5)
    pool.set_option(krill_amd._lib.OPT_SPLIT_BLOCKS, split)
    f = Rising(pool, lens, rng, rise, s_v)
    tables, n, _ = f.tables()
    q = rng.standard_normal((len(lens), R, Lq, D)).astype(np.float32) * 0.01
    q[..., 0] = 1.0
    q = O.f32_to_f16_bits(q)
    got = pool.attention(0, to_dev(q, "f16"), tables, n, max(lens), float(np.log(2.0)), torch.float32)
    got = got.double().cpu().numpy()
    ref = oracle_attention(pool, f, 0, q, "f16", float(np.log(2.0)))
    pool.close()
    top = max(255 * s_v, 65504.0)
    assert np.isfinite(got).all()
    assert np.abs(got - ref).max() <= 2.0 ** -14 * top


@pytest.mark.parametrize("mode", ["affine_g64", "ref_row"])
@pytest.mark.parametrize("D,H,R,Lq", [(64, 2, 4, 342), (128, 2, 5, 280), (256, 2, 2, 690), (512, 1, 8, 350)])
def test_merge_by_row_groups(mode, D, H, R, Lq):
    """From 8192 rows the partials are merged by row group: 72 partials of a sequence (more than
    a wave reads at once), few, and a sequence with no blocks, whose rows are zero.  Against the
    same sequences one by one, below 8192 rows each, merged by row: the same partials, at most 72
    binary32 terms under 4 summed in another order."""
    print(f"\ncase long_window_merge mode={mode} D={D}", flush=True)
    rng = np.random.default_rng(41)
    lens = [72 * 64 - 5, Lq + 3, 0, Lq]
    assert 4 * H * R * Lq >= 8192 > H * R * Lq
    pool = krill_amd.KVPool(1, H, D, sum((T + 63) // 64 for T in lens) + 4, mode, "bf16", free_list_seed=9)
    pool.set_option(krill_amd._lib.OPT_SPLIT_BLOCKS, 1)
    f = Filled(pool, lens, rng, "bf16", max_chunk=4000)
    tables, n, _ = f.tables()
    q = to_dev(rand_bits(rng, (len(lens), H * R, Lq, D), "bf16"), "bf16")
    got = pool.attention(0, q, tables, n, max(lens), 1.0 / np.sqrt(D))
    for b in range(len(lens)):
        one = pool.attention(0, q[b:b + 1], tables[b:b + 1], n[b:b + 1], max(lens), 1.0 / np.sqrt(D))
        assert (got[b] - one[0]).abs().max() <= 72 * 2.0 ** -24 * 4
    assert not got[2].any()
    # and rows of the first against the decode kernel (two kernels, each within 1e-4 of fp64)
    want = pool.attention(0, q[:1, :, Lq - 1:].contiguous(), tables[:1], n[:1], max(lens), 1.0 / np.sqrt(D))
    assert (got[:1, :, Lq - 1:] - want).abs().max() <= 2e-4
    pool.close()


@pytest.mark.parametrize("mode", ["affine_g64", "ref_row"])
@pytest.mark.parametrize("D,H,R,lens,split", [(64, 2, 70, [70, 1, 200, 64], 2), (128, 2, 70, [70, 1, 200, 64], 2),
                                              (256, 2, 72, [517, 63], 3), (64, 8, 1024, [1000] * 8, 0),
                                              (128, 8, 1024, [1000] * 8, 0)])
def test_rope_step_of_many_query_heads(mode, D, H, R, lens, split):
    """The fused decode step with RoPE of 65 and more query heads per KV head (16-row waves, and
    32-row ones): the RoPE append, then attention of queries rotated by the oracle, bit for bit."""
    print(f"\ncase long_window_rope mode={mode} D={D} R={R}", flush=True)
    B, dt, scale = len(lens), "bf16", 1.0 / np.sqrt(D)
    rng = np.random.default_rng(D + R)
    kn, vn = rand_bits(rng, (B, H, 1, D), dt), rand_bits(rng, (B, H, 1, D), dt)
    q = rand_bits(rng, (B, H * R, 1, D), dt)
    pos = np.array(lens, np.int32)
    full, mx = [T + 1 for T in lens], max(lens) + 1
    cs = krill_amd.pool.rope_table(mx, D)
    csd = torch.from_numpy(cs).cuda()
    outs, snaps = [], []
    for fused in (False, True):
        pool = krill_amd.KVPool(1, H, D, sum((T + 63) // 64 for T in full) + 4, mode, dt, free_list_seed=3)
        pool.set_option(krill_amd._lib.OPT_SPLIT_BLOCKS, split)
        f = Filled(pool, lens, np.random.default_rng(7), dt, max_chunk=300)
        slots = np.stack([pool.reserve_append(s, 1).copy() for s in f.seqs])
        tables, n = (i32(a) for a in pool.batch_tables(f.seqs, (mx + 63) // 64))
        if fused:
            outs.append(pool.decode_append_attention_rope(0, to_dev(q, dt), to_dev(kn, dt), to_dev(vn, dt), tables, n,
                                                          mx, scale, csd))
        else:
            pool.quantize_append_rope(0, to_dev(kn, dt), to_dev(vn, dt), i32(slots), i32(pos.reshape(B, 1)), csd)
            q_rot = O.rope_rows(q, O.DT_BF16, np.broadcast_to(pos[:, None, None], (B, H * R, 1)), cs)
            outs.append(pool.attention(0, to_dev(q_rot, dt), tables, n, mx, scale))
        snaps.append({k: v.cpu() for k, v in pool.gather(0, tables, n, mx).items()})
        pool.close()
    assert torch.equal(outs[0], outs[1])
    for k in snaps[0]:
        assert torch.equal(snaps[0][k].view(torch.uint8), snaps[1][k].view(torch.uint8)), k
