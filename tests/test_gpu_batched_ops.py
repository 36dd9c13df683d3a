"""Batched limb-wise sums: homo_add_many / homo_sub_many give, word for
word, what homo_add / homo_sub give pair by pair, past one launch's 64
pairs, and refuse pairs of different shapes."""

from __future__ import annotations

import numpy as np
import pytest

from conftest import device_context

pytestmark = pytest.mark.gpu


def test_add_many_matches_pairwise_adds():
    from easyfhe import fhe

    client, ctx = device_context("small")
    rng = np.random.default_rng(5)
    n = 70  # two launches
    a = [client.encrypt(rng.uniform(-1, 1, ctx.max_slots), enc_id=3000 + i) for i in range(n)]
    b = [client.encrypt(rng.uniform(-1, 1, ctx.max_slots), enc_id=4000 + i) for i in range(n)]
    for op_many, op in ((fhe.homo_add_many, fhe.homo_add), (fhe.homo_sub_many, fhe.homo_sub)):
        got = op_many(a, b, ctx)
        for x, y, g in zip(a, b, got):
            want = op(x, y, ctx)
            assert np.array_equal(g.download(), want.download())
            want.release()
        for g in got:
            g.release()
    # one operand a level lower: refused before any output exists
    low = fhe.align_to(b[1], b[1].state.replace(cur_limbs=ctx.L - 1, scaling_factor=None), ctx)
    with pytest.raises(ValueError, match="limb count"):
        fhe.homo_add_many(a[:2], [b[0], low], ctx)
    for c in a + b + [low]:
        c.release()
    ctx.close()


@pytest.mark.parametrize("params,expected", [
    # whole-ring kernels: parts of 8
    (dict(log_n=10, depth=9, dnum=2, dcrt_bits=40, first_mod=60, special_bits=60),
     {(5, 9): 1, (10, 12): 1, (10, 16): 2}),
    # 64-bit special primes from N = 2^15 on: by the words of the batch
    (dict(log_n=15, depth=3, dnum=4, dcrt_bits=40, first_mod=40, special_bits=60),
     {(2, 12): 1, (4, 8): 1, (4, 9): 2, (4, 16): 2, (2, 16): 2}),
    (dict(log_n=16, depth=9, dnum=2, dcrt_bits=59, first_mod=60, special_bits=60),
     {(2, 6): 1, (10, 5): 1, (10, 6): 2, (10, 9): 3}),
    # fp64 special primes: parts of 8
    (dict(log_n=16, depth=3, dnum=2, dcrt_bits=40, first_mod=40, special_bits=44),
     {(4, 12): 1, (4, 16): 2}),
], ids=["ring", "2^15", "wide", "fp64"])
def test_batched_rotations_run_in_as_many_parts_as_pay(params, expected):
    """A batched key switch repeats its launches in every part, so short
    batches stay whole (one key product a part); the words are the single
    rotations' however it is split."""
    from easyfhe import fhe

    client, ctx = device_context(params, rotations=(3,))
    rng = np.random.default_rng(8)
    for (limbs, n), parts in expected.items():
        cts = [client.encrypt(rng.uniform(-1, 1, 16), slots=16, cur_limbs=limbs, enc_id=i)
               for i in range(n)]
        want = [fhe.homo_rotate(c, 3, ctx).download() for c in cts]
        for split, runs in ((0, parts), (1, 1)):
            ctx.set_split_parts(split)
            ctx.profile(True)
            ctx.profile_read()
            got = fhe.homo_rotate_many(cts, 3, ctx)
            launched = ctx.profile_read()
            ctx.profile(False)
            assert sum(launched[k]["launches"] for k in ("key_inner", "ntt_low_key")
                       if k in launched) == runs, (limbs, n, split)
            for g, w in zip(got, want):
                assert np.array_equal(g.download(), w), (limbs, n, split)
        ctx.set_split_parts(0)
    ctx.close()


def test_split_batches_keep_the_fused_combine():
    """Limbs move out of the fused key product + combine only where a batch
    runs alone: of 24 rotations at 12 limbs (three parts) the separate combine
    takes q_0 alone, of one at 36 limbs a last round's limbs too."""
    from easyfhe import fhe

    client, ctx = device_context("keyswitch", rotations=(3,), relin=False)
    rng = np.random.default_rng(9)
    for limbs, n, runs in ((12, 24, 1), (36, 1, 4)):
        cts = [client.encrypt(rng.uniform(-1, 1, 16), slots=16, cur_limbs=limbs, enc_id=i)
               for i in range(n)]
        want = [fhe.homo_rotate(c, 3, ctx).download() for c in cts]
        ctx.profile(True)
        ctx.profile_read()
        got = fhe.homo_rotate_many(cts, 3, ctx)
        # accumulators, converted words and outputs of two components, one addend
        words = ctx.profile_read()["ntt_fwd_moddown"]["bytes"] / (8.0 * (1 << 16) * 7 * n)
        ctx.profile(False)
        assert round(words, 3) == runs, (limbs, n)
        for g, w in zip(got, want):
            assert np.array_equal(g.download(), w), (limbs, n)
    ctx.close()
