"""The measured cases: calls of the public entry points over the sizes, chains
and options that an encrypted prefill, a bootstrap and the key-switch
benchmark use.

Chains (every name is a parameter set of this repository's own programs):

* ``matvec``     N = 2^12 .. 2^14, 4 x 40-bit limbs, one 60-bit special prime:
                 the small-ring BSGS matrix-vector product;
* ``deep40``     N = 2^16, 60 + 35 x 40 bits, dnum 3, 12 x 44-bit special
                 primes: the key-switch benchmark and the standalone bootstrap;
* ``reference``  N = 2^16, 60 + 37 x 59 bits, dnum 5, 8 x 60-bit special
                 primes: the 32-layer prefill.

A context (keys, tables) is made once per chain and kept, as a program keeps
it; inputs are encrypted vectors of the case's seed.  Results are ciphertexts:
they stay on the device, and their limbs are downloaded when they are read.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch  # before the library: the two then share one HIP runtime

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "easyfhe-llama3-8b_amd"))

from easyfhe import fhe  # noqa: E402
from easyfhe.bs import openfhe as bs  # noqa: E402
from easyfhe.chebyshev import eval_chebyshev_series_many  # noqa: E402
from feature_major import (LinearOperator, LinearOperatorConfig, LinearWeight,  # noqa: E402
                           linear_rotations)
from feature_major.approx import silu_entry  # noqa: E402

CHAINS = {
    "deep40": dict(log_n=16, depth=35, dnum=3, dcrt_bits=40, first_mod=60, special_bits=44),
    "reference": dict(log_n=16, depth=37, dnum=5, dcrt_bits=59, first_mod=60, special_bits=60),
}
BUDGET = (3, 3)  # CoeffToSlot / SlotToCoeff levels of the bootstrap


def listed():
    return [
        # a 128 x 128 matrix-vector product on a small ring: latency and launches count
        dict(name="matvec", kind="matvec", log_n=13, limbs=4, dimension=128, baby=16),
        # the product of one slim (row-sum) ciphertext near the bottom of the chain
        dict(name="multiply_low", kind="multiply", chain="deep40", n=1, limbs=3, primes=1,
             square=False),
        # one rotation of one fresh ciphertext: a conjugation, an interactive call
        dict(name="rotate_one", kind="rotate", chain="deep40", n=1, limbs=36, rotation=1),
        # a level of the key-switch benchmark with an odd batch and level
        dict(name="multiply_mid", kind="multiply", chain="deep40", n=19, limbs=21, primes=1,
             square=False),
        # one rotation step of the key-switch benchmark
        dict(name="rotate_batch", kind="rotate", chain="deep40", n=64, limbs=36, rotation=2048),
        # a paired refresh of the residual stream: full-slot bootstraps
        dict(name="bootstrap", kind="bootstrap", log_slots=15, n=8),
        # the prefill's giant steps and head-sum rotations
        dict(name="rotate_ref", kind="rotate", chain="reference", n=16, limbs=13, rotation=512),
        # the prefill's products after a refresh
        dict(name="multiply_ref", kind="multiply", chain="reference", n=16, limbs=26, primes=1,
             square=False),
        # attention: masked sums of 8 rotations of every query-key product
        dict(name="head_sums_ref", kind="head_sums", chain="reference", n=16, limbs=17, babies=8),
        # SiLU of the gate projection's ciphertexts
        dict(name="silu_ref", kind="silu", chain="reference", n=6, limbs=14, degree=63),
        # the square projection of a decoder layer over 128 tokens
        dict(name="linear_ref", kind="linear", chain="reference", n=16, limbs=13, dimension=4096,
             fp32=False),
        # the client: masks encoded, vectors encrypted, results decrypted
        dict(name="client", kind="client", chain="deep40", n=3, limbs=36, slots=32768),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    """An integer of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(["matvec", "multiply", "multiply", "rotate", "rotate", "bootstrap",
                       "head_sums", "silu", "linear", "client"])
    chain = rng.choice(["deep40", "reference"])
    top = 36 if chain == "deep40" else 38
    if kind == "matvec":
        return dict(kind=kind, log_n=rng.choice([12, 13, 14]), limbs=rng.randint(2, 4),
                    dimension=1 << rng.randint(4, 7), baby=1 << rng.randint(2, 4))
    if kind == "multiply":
        limbs = rng.randint(3, top)
        return dict(kind=kind, chain=chain, n=_log_int(rng, 1, 48), limbs=limbs,
                    primes=1 if limbs < 5 else rng.choice([1, 1, 2]), square=rng.random() < 0.3)
    if kind == "rotate":
        return dict(kind=kind, chain=chain, n=_log_int(rng, 1, 48), limbs=rng.randint(2, top),
                    rotation=1 << rng.randint(0, 14))
    if kind == "bootstrap":
        return dict(kind=kind, log_slots=rng.choice([7, 15]), n=_log_int(rng, 1, 8))
    if kind == "head_sums":
        return dict(kind=kind, chain=chain, n=_log_int(rng, 1, 24), limbs=rng.randint(8, 24),
                    babies=rng.choice([2, 3, 4, 8]))
    if kind == "silu":
        degree = rng.choice([15, 31, 59, 63])
        return dict(kind=kind, chain=chain, n=_log_int(rng, 1, 12), limbs=rng.randint(10, 20),
                    degree=degree)
    if kind == "linear":
        return dict(kind=kind, chain=chain, n=_log_int(rng, 1, 12), limbs=rng.randint(5, 13),
                    dimension=rng.choice([512, 1024, 2048, 4096]), fp32=rng.random() < 0.5)
    return dict(kind="client", chain=chain, n=_log_int(rng, 1, 5), limbs=rng.randint(1, top),
                slots=1 << rng.choice([7, 12, 15]))


# ---------------------------------------------------------------------------
# contexts, programs
# ---------------------------------------------------------------------------

_contexts: dict = {}
_programs: dict = {}


def _context(chain: str, **params):
    """(client, context) of a chain, with its relinearisation key."""
    key = (chain, tuple(sorted(params.items())))
    if key not in _contexts:
        spec = fhe.CKKSContextSpec(**(params or CHAINS[chain]), seed=0)
        _contexts[key] = fhe.generate_client_context(spec, device="cuda:0")
    return _contexts[key]


def _matvec_context(log_n: int):
    return _context("matvec", log_n=log_n, depth=3, dnum=4, dcrt_bits=40, first_mod=40,
                    special_bits=60)


def _bootstrap_program(ctx, log_slots: int):
    if log_slots not in _programs:
        depth = bs.generate(ctx, bs.BootstrapSpec(log_slots=log_slots, level_budget=BUDGET,
                                                  output_levels=0)).depth_limbs
        _programs[log_slots] = bs.generate(
            ctx, bs.BootstrapSpec(log_slots=log_slots, level_budget=BUDGET,
                                  output_levels=ctx.L - depth - 1))
    return _programs[log_slots]


def _vectors(seed: int, n: int, slots: int):
    return np.random.default_rng(seed).uniform(-1.0, 1.0, (n, slots))


def _encrypt(client, rows, seed: int, limbs: int, first: int = 0):
    return [client.encrypt(z, slots=len(z), cur_limbs=limbs,
                           enc_id=(seed * 1000003 + first + i) & 0xFFFFFFFF)
            for i, z in enumerate(rows)]


class Limbs(tuple):
    """Ciphertexts (or plaintexts) of one shape; read, they are one array of
    their limbs."""

    def __iter__(self):
        words = np.stack([c.download() for c in super().__iter__()])
        yield torch.from_numpy(words.view(np.int64))


# ---------------------------------------------------------------------------
# what a program has in hand
# ---------------------------------------------------------------------------


def prepare(case, seed):
    kind, n = case["kind"], case.get("n", 1)
    if kind == "matvec":
        client, ctx = _matvec_context(case["log_n"])
        D, B, limbs, slots = case["dimension"], case["baby"], case["limbs"], ctx.max_slots
        lanes, G = slots // D, D // B
        ctx.generate_rotation_keys([lanes * b for b in range(1, B)] + ([B * lanes] if G > 1 else []))
        rng = np.random.default_rng(seed)
        W = rng.uniform(-1, 1, (D, D))
        feat = np.arange(slots) // lanes
        rows = np.stack([W[(feat - g * B) % D, (feat + b) % D]
                         for g in range(G) for b in range(B)])
        pts = fhe.encode_rows(ctx, rows, limbs=limbs, scale=ctx.scale_at(limbs), slots=slots)
        x = np.repeat(rng.uniform(-1, 1, D), lanes)
        return dict(kind=kind, ctx=ctx, ct=_encrypt(client, [x], seed, limbs)[0], pts=pts,
                    offsets=[lanes * b for b in range(B)], giant=B * lanes, giants=G)
    if kind == "bootstrap":
        client, ctx = _context("deep40")
        prog = _bootstrap_program(ctx, case["log_slots"])
        cts = _encrypt(client, _vectors(seed, n, 1 << case["log_slots"]), seed, 1)
        return dict(kind=kind, ctx=ctx, cts=cts, program=prog)

    client, ctx = _context(case["chain"])
    limbs = case["limbs"]
    if kind == "client":
        slots = case["slots"]
        z = np.random.default_rng(seed).uniform(-1, 1, (n, slots, 2)) @ [1.0, 1.0j]
        return dict(kind=kind, ctx=ctx, client=client, values=z, seed=seed, limbs=limbs,
                    slots=slots, cts=_encrypt(client, z, seed, limbs, first=500000))
    if kind == "silu":
        entry = silu_entry(-12.0, 12.0, case["degree"])
        x = np.clip(np.random.default_rng(seed).normal(0.0, 2.0, (n, ctx.max_slots)), -12, 12)
        return dict(kind=kind, ctx=ctx, cts=_encrypt(client, x, seed, limbs), entry=entry)

    cts = _encrypt(client, _vectors(seed, n, ctx.max_slots), seed, limbs)
    if kind == "rotate":
        ctx.generate_rotation_keys([case["rotation"]])
        return dict(kind=kind, ctx=ctx, cts=cts, rotation=case["rotation"])
    if kind == "multiply":
        other = cts if case["square"] else _encrypt(
            client, _vectors(seed + 7919, n, ctx.max_slots), seed, limbs, first=900000)
        return dict(kind=kind, ctx=ctx, cts=cts, other=other, primes=case["primes"])
    if kind == "head_sums":
        lanes, babies = 8, case["babies"]
        offsets = [(e - 1) * lanes for e in range(babies)]
        ctx.generate_rotation_keys([o for o in offsets if o])
        mask = np.zeros(ctx.max_slots)
        mask.reshape(-1, lanes)[1::babies] = 1.0
        pts = fhe.encode_rows(ctx, mask, limbs=limbs, scale=ctx.scale_at(limbs),
                              slots=ctx.max_slots, is_ext=True)
        return dict(kind=kind, ctx=ctx, cts=cts, offsets=offsets, pts=pts * babies)
    # kind == "linear"
    D = case["dimension"]
    lanes = ctx.max_slots // D
    cfg = LinearOperatorConfig(reuse_baby_rotations=False, timed_stages=False)
    ctx.generate_rotation_keys(linear_rotations(dimension=D, token_lanes=lanes,
                                                operator_config=cfg))
    W = np.random.default_rng(seed).normal(0.0, 0.02, (D, D))
    weight = LinearWeight(W, dtype=np.float32 if case["fp32"] else np.float64, context=ctx)
    return dict(kind=kind, ctx=ctx, cts=cts, weight=weight,
                op=LinearOperator(context=ctx, token_lanes=lanes, config=cfg))


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------


def run(s):
    kind, ctx = s["kind"], s["ctx"]
    if kind == "matvec":
        acc = fhe.hoisted_mac_sum(s["ct"], s["offsets"], s["pts"], s["giant"], s["giants"], ctx)
        out = fhe.rescale(acc, ctx)
        acc.release()
        return Limbs([out])
    if kind == "rotate":
        if len(s["cts"]) == 1:
            return Limbs([fhe.homo_rotate(s["cts"][0], s["rotation"], ctx)])
        return Limbs(fhe.homo_rotate_many(s["cts"], s["rotation"], ctx))
    if kind == "multiply":
        return Limbs(fhe.homo_mul_relin_rescale_many(s["cts"], s["other"], ctx,
                                                     primes=s["primes"]))
    if kind == "bootstrap":
        return Limbs(bs.bootstrap_many(s["cts"], ctx, s["program"]))
    if kind == "head_sums":
        acc = fhe.hoisted_mac_sum_ext_many(s["cts"], s["offsets"], s["pts"], 0, 1, ctx)
        outs = fhe.rescale_many(acc, ctx)
        for a in acc:
            a.release()
        return Limbs(outs)
    if kind == "silu":
        lo, hi = s["entry"]["fit_interval"]
        return Limbs(eval_chebyshev_series_many(s["cts"], s["entry"]["coefficients"],
                                                lower_bound=lo, upper_bound=hi,
                                                crypto_context=ctx))
    if kind == "linear":
        outs, _ = s["op"].apply(s["cts"], s["weight"])
        return Limbs(outs)
    client, limbs = s["client"], s["limbs"]
    pts = fhe.encode_rows(ctx, s["values"], limbs=limbs, scale=ctx.scale_at(limbs),
                          slots=s["slots"])
    cts = _encrypt(client, s["values"], s["seed"], limbs)
    return dict(plaintexts=Limbs(pts), ciphertexts=Limbs(cts),
                values=np.stack([client.decrypt_complex(c) for c in s["cts"]]))


def exact(case, seed):
    """The decrypted values are the encrypted ones; limbs have no value of
    their own (keys and noise are the context's)."""
    if case["kind"] != "client":
        return None
    z = np.random.default_rng(seed).uniform(-1, 1, (case["n"], case["slots"], 2)) @ [1.0, 1.0j]
    return dict(plaintexts=None, ciphertexts=None, values=z)


def tolerance(case):
    """Limbs are integers and stay the same.  Decrypted values: the words are
    the same, what may differ is the order of the fp64 transform's sums (on
    the 59-bit chain the decrypted values are 2e-15 off the encrypted ones)."""
    return {"rel": 1e-14, "max": 1e-12} if case["kind"] == "client" else "exact"


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------


def _keyswitch_ops(N: int, limbs: int, alpha: int, digits: int) -> float:
    """Modular products of one key switch: the inverse NTTs of the input and
    of the two special parts, the forward ones of the extended digits and of
    the two converted parts, the base conversions and the key product."""
    bfly = N / 2 * math.log2(N)
    E = limbs + alpha
    ntts = limbs + 2 * alpha + digits * E - limbs + 2 * limbs
    conv = N * (limbs * E + 2 * alpha * limbs)
    return ntts * bfly + conv + 2.0 * digits * E * N


def work(case):
    kind, n = case["kind"], case.get("n", 1)
    if kind == "matvec":
        N, alpha, size, limbs = 1 << case["log_n"], 1, 1, case["limbs"]
    else:
        chain = case.get("chain", "deep40")
        N, limbs = 1 << 16, case.get("limbs", 36)
        alpha, size = (12, 12) if chain == "deep40" else (8, 8)
    lp = 8.0 * N  # bytes of a limb-polynomial
    digits = -(-limbs // size)
    E = limbs + alpha
    key = 2.0 * digits * E * lp
    ks = _keyswitch_ops(N, limbs, alpha, digits)
    ct = 2.0 * limbs * lp
    if kind == "matvec":
        D, B = case["dimension"], case["baby"]
        switches = B - 1 + D // B - 1
        return {"bytes": ct + B * key + D * limbs * lp + 2.0 * (limbs - 1) * lp,
                "flops": 2.0 * (switches * ks + 2.0 * D * limbs * N)}
    if kind == "rotate":
        return {"bytes": 2.0 * n * ct + key, "flops": 2.0 * n * ks}
    if kind == "multiply":
        ins = 1 if case["square"] else 2
        out = 2.0 * (limbs - case["primes"]) * lp
        return {"bytes": n * (ins * ct + out) + key, "flops": 2.0 * n * (ks + 4.0 * limbs * N)}
    if kind == "head_sums":
        B = case["babies"]
        return {"bytes": n * (2.0 * ct - 2.0 * lp) + (B - 1) * key + E * lp,
                "flops": 2.0 * n * (B - 1) * (ks + 2.0 * E * N)}
    if kind == "silu":
        products = 2.0 * math.sqrt(2.0 * case["degree"])
        return {"bytes": n * 2.0 * ct + key, "flops": 2.0 * n * products * ks}
    if kind == "bootstrap":
        # 60 products of EvalMod on two halves and 40 rotations at the mean level
        return {"bytes": n * 2.0 * 20 * lp + 40 * key,
                "flops": 2.0 * n * 160 * _keyswitch_ops(N, 24, 12, 2)}
    if kind == "linear":
        D, B = case["dimension"], 64
        switches = B - 1 + D // B - 1
        return {"bytes": n * 2.0 * ct + (B + 8) * key + D * D * (4.0 if case["fp32"] else 8.0),
                "flops": 2.0 * (n * (switches * ks + 2.0 * D * limbs * N)
                                + D * limbs * N / 2 * 16)}
    z = 16.0 * case["slots"]
    return {"bytes": n * (limbs * lp + z + ct + z + ct + z),
            "flops": 2.0 * n * 6 * limbs * N / 2 * 16}
