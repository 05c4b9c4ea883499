"""Timed cases of the CKKS engine on one GPU.

Each case is one call (or the few calls that belong together) a program makes
through the public entry points, at a parameter set the package ships.
``listed`` names the cases, ``draw`` samples more from the same ranges,
``prepare`` makes what a program holds before the call, ``run`` makes the call
and ``work`` counts what it cannot do without.

One engine per parameter set is built once per process (its tables depend on
the parameter set alone); keys and operands belong to the state, and ``run``
installs the state's keys first, as a server does that evaluates for several
clients on one engine.
"""

from __future__ import annotations

import functools
import math

import numpy as np
import torch

from fhelium_amd.config import CkksConfig, Preset
from fhelium_amd.core import Ciphertext
from fhelium_amd.csprng import Csprng
from fhelium_amd.engine import CkksEngine
from fhelium_amd.linear import diagonal_matvec, prepare_diagonals
from fhelium_amd.rns import RnsLayout

N14_S30 = "slots8192-scale30-levels9-int64"
N14_S40 = "slots8192-scale40-levels7-int64"
N15_S30 = "slots16384-scale30-levels21-int64"
N16_S40 = "slots32768-scale40-levels34-int64"
N16_S50 = "slots32768-scale50-levels27-int64"
PRESETS = [p.value for p in Preset]
KINDS = ["rotate", "hmult", "chain", "rotate_steps", "ntt", "matvec", "encode", "decrypt"]


def listed():
    return [
        # one ciphertext, smallest ring: an interactive client waiting for one rotation (latency)
        {"name": "rotate_one_n14", "kind": "rotate", "preset": N14_S40, "level": 0, "batch": 1},
        # one product at full depth on the headline parameter set
        {"name": "hmult_one_n16", "kind": "hmult", "preset": N16_S40, "level": 0, "batch": 1},
        # the same product as the four public methods, half way down the chain
        # (what code written against the engine's method surface calls)
        {"name": "chain_one_n16", "kind": "chain", "preset": N16_S40, "level": 17, "batch": 1},
        # one level group of the batched benchmark: every entry rotated by its own step
        {"name": "rotate_steps_n16", "kind": "rotate_steps", "preset": N16_S40, "level": 6, "batch": 7},
        # one level group of the batched benchmark, products, a large group
        {"name": "hmult_batch_n16", "kind": "hmult", "preset": N16_S40, "level": 2, "batch": 16},
        # a small batch near the end of the chain, where few limbs are left
        {"name": "rotate_late_n16", "kind": "rotate", "preset": N16_S40, "level": 29, "batch": 5},
        # the high-precision parameter set (50-bit scale primes)
        {"name": "chain_s50_n16", "kind": "chain", "preset": N16_S50, "level": 3, "batch": 3},
        # the middle ring with 30-bit scale primes
        {"name": "hmult_s30_n15", "kind": "hmult", "preset": N15_S30, "level": 4, "batch": 6},
        # ring kernel: a batch of level-0 ciphertexts to the NTT domain and back
        {"name": "ntt_n16", "kind": "ntt", "preset": N16_S40, "level": 0, "batch": 24},
        # plaintext matrix times encrypted vector, diagonal method
        {"name": "matvec_n16", "kind": "matvec", "preset": N16_S40, "level": 8, "batch": 32},
        # encoding a weight matrix's diagonals for that product, and decoding
        # results, both next to the data
        {"name": "encode_n16", "kind": "encode", "preset": N16_S40, "level": 8, "batch": 12},
        {"name": "decrypt_n16", "kind": "decrypt", "preset": N16_S40, "level": 19, "batch": 9},
    ]


@functools.lru_cache(maxsize=None)
def _config(preset: str) -> CkksConfig:
    return CkksConfig.from_preset(preset)


@functools.lru_cache(maxsize=None)
def _layout(preset: str) -> RnsLayout:
    return RnsLayout(_config(preset))


@functools.lru_cache(maxsize=None)
def _engine(preset: str) -> CkksEngine:
    return CkksEngine(preset, rng_seed=0)


def _top_level(kind: str, cfg: CkksConfig) -> int:
    """Last level the call accepts: a product or a matrix-vector product also rescales."""

    return cfg.public_level_count - (2 if kind in ("hmult", "chain", "matvec") else 1)


def draw(rng):
    """A case of the listed kinds at any parameter set, level and batch, costing
    no more than the largest listed one."""

    ceiling = max(_cost(c) for c in listed())
    kind = rng.choice(KINDS)
    preset = rng.choice(PRESETS)
    cfg = _config(preset)
    if kind == "hmult" and cfg.scale_bits == 50:
        kind = "chain"  # products at the high-precision sets go through the method chain
    case = {"kind": kind, "preset": preset, "level": rng.randint(0, _top_level(kind, cfg)), "batch": 1}
    low, high = (2, 48) if kind == "matvec" else (1, 24)
    case["batch"] = round(math.exp(rng.uniform(math.log(low), math.log(high))))
    while case["batch"] > low and _cost(case) > ceiling:
        case["batch"] = max(low, case["batch"] * 2 // 3)
    return case


# ---------------------------------------------------------------------------
# States
# ---------------------------------------------------------------------------
def _uniform(eng, rng, components, batch, level):
    """Ciphertext payload: RLWE ciphertexts are uniform residues to every
    evaluation call (no key or noise is looked at)."""

    cfg = eng.config
    q = torch.tensor(cfg.moduli[level: cfg.num_q_primes], dtype=torch.int64, device=eng.device)
    shape = (components,) if batch == 1 else (components, batch)
    return rng.uniform_mod(q, shape, cfg.N)


def _ciphertext(eng, rng, batch, level):
    return Ciphertext(_uniform(eng, rng, 2, batch, level), level, eng.config.default_scale)


def _steps(seed, count, slots):
    """Distinct rotation steps in 1..1024, as the batched benchmark draws them."""

    gen = np.random.default_rng(seed)
    return [int(s) for s in 1 + gen.permutation(min(1024, slots - 1))[:count]]


def _slots(case, seed):
    cfg = _config(case["preset"])
    gen = np.random.default_rng(seed)
    shape = (case["batch"], cfg.slots)
    return gen.uniform(-1, 1, shape) + 1j * gen.uniform(-1, 1, shape)


def prepare(case, seed):
    kind, level, batch = case["kind"], case["level"], case["batch"]
    eng = _engine(case["preset"])
    cfg = eng.config
    rng = Csprng(seed, eng.device)
    eng.rng = rng
    st = {"eng": eng, "kind": kind, "level": level}
    if kind in ("rotate", "hmult", "chain", "rotate_steps", "matvec", "decrypt"):
        eng.rotation_keys = {}
        st["secret"] = eng.generate_secret_key()
    if kind in ("hmult", "chain"):
        st["relin"] = eng.generate_relinearization_key()
        st["a"], st["b"] = (_ciphertext(eng, rng, batch, level) for _ in range(2))
    elif kind == "rotate":
        st["steps"] = _steps(seed, 1, cfg.slots)
        st["a"] = _ciphertext(eng, rng, batch, level)
    elif kind == "rotate_steps":
        st["steps"] = _steps(seed, batch, cfg.slots)
        st["a"] = Ciphertext(_uniform(eng, rng, 2, batch, level).view(2, batch, -1, cfg.N), level, cfg.default_scale)
    elif kind == "ntt":
        st["a"] = _ciphertext(eng, rng, batch, level)
    elif kind == "matvec":
        st["steps"] = list(range(1, batch))
        st["a"] = _ciphertext(eng, rng, 1, level)
        gen = np.random.default_rng(seed)
        st["diagonals"] = prepare_diagonals(eng, gen.uniform(-1, 1, (batch, cfg.slots)), level)
    elif kind == "encode":
        st["values"] = torch.from_numpy(_slots(case, seed)).to(eng.device)
    elif kind == "decrypt":
        st["a"] = eng.encrypt(_slots(case, seed), level=level)
    if kind in ("rotate", "rotate_steps", "matvec"):
        for step in st["steps"]:
            eng.generate_rotation_key(step)
        st["rotation"] = dict(eng.rotation_keys)
    return st


def run(st):
    eng, kind = st["eng"], st["kind"]
    # the caller's keys
    if "secret" in st:
        eng.secret_key = st["secret"]
    if "relin" in st:
        eng.relinearization_key = st["relin"]
    if "rotation" in st:
        eng.rotation_keys = st["rotation"]

    if kind == "rotate":
        return eng.rotate_by_step(st["a"], st["steps"][0]).data
    if kind == "hmult":
        return eng.hmult(st["a"], st["b"]).data
    if kind == "chain":
        a = eng.coefficient_domain_to_ntt_domain(st["a"])
        b = eng.coefficient_domain_to_ntt_domain(st["b"])
        return eng.rescale_to_next_level(eng.relinearize(eng.multiply(a, b))).data
    if kind == "rotate_steps":
        return eng.rotate_by_steps(st["a"], st["steps"]).data
    if kind == "ntt":
        there = eng.coefficient_domain_to_ntt_domain(st["a"])
        return there.data, eng.ntt_domain_to_coefficient_domain(there).data
    if kind == "matvec":
        return diagonal_matvec(eng, st["a"], st["diagonals"]).data
    if kind == "encode":
        return eng.encode_on_device(st["values"], level=st["level"], polynomial_domain="ntt").data
    if kind == "decrypt":
        return eng.decrypt_on_device(st["a"])
    raise ValueError(kind)


def exact(case, seed):
    """Decoded slots against the values that were encrypted (the rest is the
    encryption's own noise).  Every other output is integer residues."""

    if case["kind"] == "decrypt":
        return torch.from_numpy(_slots(case, seed))
    return None


# ---------------------------------------------------------------------------
# Compulsory work
# ---------------------------------------------------------------------------
_MULMOD = 6     # binary64 operations of one exact modular product
_BUTTERFLY = 8  # one product, one sum, one difference


def work(case):
    """Bytes of the operands, keys and results (each once), and arithmetic in
    binary64 operations, modular products and butterflies counted once each."""

    kind, level, batch = case["kind"], case["level"], case["batch"]
    cfg = _config(case["preset"])
    n, p = cfg.N, cfg.num_p_primes
    lq = cfg.num_q_primes - level
    lqp = lq + p
    limb = 8 * n
    row_ntt = n // 2 * cfg.logN * _BUTTERFLY
    digits = [len(s.prime_ids) for s in _layout(case["preset"]).digit_specs(level)]
    key = len(digits) * 2 * lqp * limb
    mul = _MULMOD * n
    up = sum(lqp * (d * mul + row_ntt) for d in digits)  # digits onto the rows, transformed
    down = len(digits) * 2 * lqp * mul + 2 * lqp * row_ntt + 2 * lq * (p + 1) * mul  # products, back, divided
    if kind in ("rotate", "rotate_steps"):
        keys = batch if kind == "rotate_steps" else 1
        return {"bytes": batch * 4 * lq * limb + keys * key, "flops": batch * (up + down)}
    if kind in ("hmult", "chain"):
        front = 7 * lq * row_ntt + 4 * lq * mul
        return {"bytes": batch * (4 * lq + 2 * (lq - 1)) * limb + key, "flops": batch * (front + up + down)}
    if kind == "ntt":
        return {"bytes": 3 * batch * 2 * lq * limb, "flops": 2 * batch * 2 * lq * row_ntt}
    if kind == "matvec":
        return {"bytes": (2 * lq + 2 * (lq - 1) + batch * lq) * limb + (batch - 1) * key,
                "flops": up + (batch - 1) * (down + 2 * lq * row_ntt) + batch * 2 * lq * mul + 2 * lq * row_ntt}
    if kind == "encode":
        return {"bytes": batch * (16 * cfg.slots + lq * limb),
                "flops": batch * (n // 2 * cfg.logN * 10 + lq * (mul + row_ntt))}
    if kind == "decrypt":
        # two residues of each coefficient determine it
        rows = min(2, lq)
        return {"bytes": batch * (2 * rows * limb + 16 * cfg.slots),
                "flops": batch * (rows * (2 * row_ntt + mul) + n // 2 * cfg.logN * 10)}
    raise ValueError(kind)


def _cost(case) -> float:
    """Relative cost of a case (what draw compares)."""

    w = work(case)
    return w["bytes"] / 5e12 + w["flops"] / 3e13
