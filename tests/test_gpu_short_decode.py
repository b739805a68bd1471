"""Decode over short sequences: a workgroup per (sequence, KV head), against the fp64 oracle
and the flat split, at the lengths where the choice between them turns (1.5 blocks per wave,
one workgroup per compute unit)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import krill_amd  # noqa: E402
from tests.kvutil import Filled, oracle_attention, rand_bits, to_dev  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["affine_g64", "ref_row"])
@pytest.mark.parametrize("D,R,Lq,lens", [
    (64, 4, 1, [1, 64, 65, 512, 576]),          # 9 blocks, six waves: the last length that takes it
    (64, 4, 1, [1, 577, 64]),                   # one block more: the flat split
    (128, 5, 1, [0, 1, 63, 700, 768]),          # an empty sequence
    (128, 8, 1, [384, 5, 128]),
    (128, 2, 4, [768, 4, 130]),                 # a few new rows
    (256, 2, 1, [768, 1, 64]),
    (256, 8, 1, [100, 256, 31]),
])
def test_short_sequences(mode, D, R, Lq, lens):
    print(f"\ncase short_decode mode={mode} D={D} R={R} Lq={Lq} lens={lens}", flush=True)
    rng = np.random.default_rng(D + R)
    H = 2
    pool = krill_amd.KVPool(1, H, D, sum((n + 63) // 64 for n in lens) + 4, mode, "bf16", free_list_seed=3)
    f = Filled(pool, lens, rng, "bf16", max_chunk=300)
    tables, n, _ = f.tables()
    q = rand_bits(rng, (len(lens), H * R, Lq, D), "bf16")
    scale = 1.0 / np.sqrt(D)
    got = pool.attention(0, to_dev(q, "bf16"), tables, n, max(lens), scale).cpu()
    pool.set_option(krill_amd._lib.OPT_SPLIT_BLOCKS, 2)  # a chosen split: always the flat one
    flat = pool.attention(0, to_dev(q, "bf16"), tables, n, max(lens), scale).cpu()
    ref = oracle_attention(pool, f, 0, q, "bf16", scale)
    pool.close()
    assert np.abs(got.double().numpy() - ref).max() <= 2e-3  # the decode tests' bound
    # the same products in another order: binary32 sums of at most 768 values of order 1
    assert (got - flat).abs().max() <= 768 * 2.0 ** -24 * 4
