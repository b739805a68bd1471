"""Decode over short sequences: a workgroup per (sequence, KV head), against the fp64 oracle
and the flat split, at the lengths where the choice between them turns (blocks per wave, one
workgroup per compute unit).  That form leaves the workspace as it was, the flat split writes
the partials of sequences of several blocks into it: so each case states which one runs."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import krill_amd  # noqa: E402
from tests.kvutil import Filled, i32, oracle_attention, rand_bits, to_dev  # noqa: E402

pytestmark = pytest.mark.gpu
SPLIT = krill_amd._lib.OPT_SPLIT_BLOCKS


def _workspace(pool, B, Hq, Lq, mx):
    return torch.full((pool.workspace_size(B, Hq, Lq, mx),), 0xA5, dtype=torch.uint8, device="cuda")


def _left_alone(ws):
    return bool((ws == 0xA5).all())


def _check(mode, D, H, R, Lq, lens, per_seq, seed):
    rng = np.random.default_rng(seed)
    pool = krill_amd.KVPool(1, H, D, sum((n + 63) // 64 for n in lens) + 4, mode, "bf16", free_list_seed=3)
    f = Filled(pool, lens, rng, "bf16", max_chunk=300)
    tables, n, _ = f.tables()
    q = rand_bits(rng, (len(lens), H * R, Lq, D), "bf16")
    scale = 1.0 / np.sqrt(D)
    ws = _workspace(pool, len(lens), H * R, Lq, max(lens))
    got = pool.attention(0, to_dev(q, "bf16"), tables, n, max(lens), scale, ws=ws).cpu()
    assert _left_alone(ws) == per_seq
    pool.set_option(SPLIT, 1)  # a chosen split: always the flat one
    ws = _workspace(pool, len(lens), H * R, Lq, max(lens))
    flat = pool.attention(0, to_dev(q, "bf16"), tables, n, max(lens), scale, ws=ws).cpu()
    assert not _left_alone(ws)
    ref = oracle_attention(pool, f, 0, q, "bf16", scale)
    pool.close()
    assert np.abs(got.double().numpy() - ref).max() <= 2e-3  # the decode tests' bound
    # the same products in another order: binary32 sums of at most 768 values of order 1
    assert (got - flat).abs().max() <= 768 * 2.0 ** -24 * 4


@pytest.mark.parametrize("mode,D,R,Lq,lens,per_seq", [
    *((m, *c) for m in ("affine_g64", "ref_row") for c in [
        (64, 4, 1, [1, 64, 65, 512, 576], True),    # 9 blocks, six waves
        (64, 4, 1, [1, 577, 64], False),            # one block more
        (64, 2, 4, [500, 4, 130], True),            # a few new rows
        (128, 5, 1, [0, 1, 63, 700, 768], True),    # an empty sequence; 12 blocks, eight waves
        (128, 5, 1, [769, 5], False),
    ]),
    ("affine_g64", 128, 8, 1, [384, 5, 128], True),  # four waves: the LDS
    ("affine_g64", 128, 8, 1, [385, 5, 128], False),
    ("affine_g64", 128, 2, 4, [384, 4, 130], True),
    ("affine_g64", 256, 2, 1, [768, 1, 64], True),
    ("affine_g64", 256, 2, 2, [384, 2, 64], True),
    ("affine_g64", 256, 8, 1, [100, 192, 31], True),  # two waves
    ("affine_g64", 256, 8, 1, [193, 31], False),
    ("ref_row", 128, 8, 1, [512, 5, 128], True),     # row mode, many rows or 256 dims: a block a wave
    ("ref_row", 128, 8, 1, [513, 5], False),
    ("ref_row", 128, 2, 4, [512, 4, 130], True),
    ("ref_row", 256, 2, 1, [512, 1, 64], True),
    ("ref_row", 256, 2, 1, [513, 1], False),
    ("ref_row", 256, 2, 2, [500, 2, 64], True),
    ("ref_row", 256, 2, 2, [600, 2, 64], False),
    ("ref_row", 256, 8, 1, [256, 31], True),
    ("ref_row", 256, 8, 1, [257, 31], False),
])
def test_short_sequences(mode, D, R, Lq, lens, per_seq):
    print(f"\ncase short_decode mode={mode} D={D} R={R} Lq={Lq} lens={lens}", flush=True)
    _check(mode, D, 2, R, Lq, lens, per_seq, seed=D + R)


@pytest.mark.parametrize("more", [0, 1])
def test_one_workgroup_per_compute_unit(more):
    """Up to one round of workgroups; one sequence more takes the flat split."""
    print(f"\ncase short_decode_round more={more}", flush=True)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    _check("affine_g64", 64, 2, 2, 1, [70] * (cus // 2 + more), more == 0, seed=5)


@pytest.mark.parametrize("mode", ["affine_g64", "ref_row"])
@pytest.mark.parametrize("D,R,lens", [(64, 4, [0, 63, 64, 500]), (128, 5, [5, 128, 640]), (128, 8, [1, 100, 300]),
                                      (256, 2, [64, 450]), (256, 8, [1, 64, 150])])
@pytest.mark.parametrize("rope", [False, True])
def test_fused_step(mode, D, R, lens, rope):
    """The decode step with the append (and RoPE) fused, both ways on twin pools: outputs as
    above, the pools' bytes the same."""
    print(f"\ncase short_decode_fused mode={mode} D={D} R={R} rope={rope}", flush=True)
    H, B, scale = 2, len(lens), 1.0 / np.sqrt(D)
    rng = np.random.default_rng(D + R)
    new = [to_dev(rand_bits(rng, (B, H, 1, D), "bf16"), "bf16") for _ in range(2)]
    q = to_dev(rand_bits(rng, (B, H * R, 1, D), "bf16"), "bf16")
    full = [T + 1 for T in lens]
    outs, snaps = [], []
    for split in (0, 1):
        pool = krill_amd.KVPool(1, H, D, sum((n + 63) // 64 for n in full) + 4, mode, "bf16", free_list_seed=3)
        pool.set_option(SPLIT, split)
        f = Filled(pool, lens, np.random.default_rng(7), "bf16", max_chunk=300)
        for s in f.seqs:
            pool.reserve_append(s, 1)
        tables, n = (i32(a) for a in pool.batch_tables(f.seqs, (max(full) + 63) // 64))
        ws = _workspace(pool, B, H * R, 1, max(full))
        args = (0, q, *new, tables, n, max(full), scale)
        if rope:
            cs = torch.from_numpy(krill_amd.pool.rope_table(max(full), D)).cuda()
            outs.append(pool.decode_append_attention_rope(*args, cs, ws=ws).cpu())
        else:
            outs.append(pool.decode_append_attention(*args, ws=ws).cpu())
        assert _left_alone(ws) == (split == 0)
        snaps.append({k: v.cpu() for k, v in pool.gather(0, tables, n, max(full)).items()})
        pool.close()
    assert (outs[0] - outs[1]).abs().max() <= 768 * 2.0 ** -24 * 4
    for k in snaps[0]:
        assert torch.equal(snaps[0][k].view(torch.uint8), snaps[1][k].view(torch.uint8)), k
