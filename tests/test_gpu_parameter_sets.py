"""The fused key switch against the per-digit op sequence it replaces
(hybrid_keyswitch.py:321-371), bit for bit, over every shipped parameter set
and a longer chain on a small ring, in both arithmetic modes: digit widths 1
to 6 (a level that cuts into the leading digit narrows it), one to six P
primes, 30-, 40- and 50-bit scale primes, and residues at both ends of their
range, where the sums of products are largest."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from fhelium_amd import kernels as K
from fhelium_amd.config import CkksConfig, Preset
from fhelium_amd.core import Ciphertext
from fhelium_amd.csprng import Csprng
from fhelium_amd.engine import CkksEngine

pytestmark = pytest.mark.gpu


CHAINS = {p.value: CkksConfig.from_preset(p).with_ring_log(12) for p in Preset}
# the last five scale primes lie above and below 2^50 + 2^30 in turn: integer
# rows beside binary64 ones, an integer row the first to be dropped at level 71
CHAINS["scale50-levels76-p6"] = CkksConfig(12, 50, 76, 6, 1 << 16)


@pytest.fixture(scope="module", params=[(c, m) for c in CHAINS for m in ("fast", "exact")], ids="-".join)
def eng(request):
    chain, mode = request.param
    return CkksEngine(CHAINS[chain], ntt_mode=mode, rng_seed=17)


def components(eng, level):
    """[3, rows, N]: uniform residues, all q - 1, and q - 1 next to 0."""

    q = torch.tensor(eng.config.moduli[level: eng.config.num_q_primes], dtype=torch.int64, device=eng.device)
    uniform = Csprng(level, eng.device).uniform_mod(q, (), eng.config.N)
    top = (q - 1).unsqueeze(1).expand_as(uniform)
    mixed = top * (torch.arange(eng.config.N, device=eng.device) % 2)
    return torch.stack([uniform, top, mixed])


@pytest.mark.parametrize("offset", [0, 1, 2, 3, -2, -5])
def test_key_switch_matches_per_digit_sequence(eng, offset):
    level = offset if offset >= 0 else eng.config.public_level_count + offset
    if not 0 <= level < eng.config.public_level_count - 1:
        pytest.skip("this chain is shorter")
    key = eng.generate_relinearization_key()
    x = components(eng, level)
    base = x.flip(0).contiguous()
    ks = eng.key_switcher
    params = eng.runtime.params(level)
    corr0, corr1 = ks.apply_key_switch(x, key, level)
    want = torch.stack([K.add_canonical(base, corr0, params), corr1])
    assert torch.equal(ks.key_switch_fused(x, key, level, base0=base), want)
    rescaled = ks.key_switch_fused(x, key, level, base0=base, rescale=True)
    assert torch.equal(rescaled, eng.rescale_to_next_level(Ciphertext(want, level, 1.0)).data)


@pytest.mark.parametrize("offset", [0, -2, -5])
def test_product_and_hoisted_rotation_match_composition(eng, offset):
    level = offset if offset >= 0 else eng.config.public_level_count + offset
    eng.generate_relinearization_key()
    x = components(eng, level)
    a = Ciphertext(torch.stack([x, x.flip(0)]), level, eng.config.default_scale)
    b = Ciphertext(torch.stack([x.flip(0), x.roll(1, 0)]), level, eng.config.default_scale)
    fused = eng.hmult(a, b).data
    one = Ciphertext(a.data[:, 1].contiguous(), level, a.scale)
    hoisted = eng.rotate_hoisted(one, [1, 5]).data
    eng.fused_keyswitch = False
    try:
        assert torch.equal(fused, eng.hmult(a, b).data)
        assert torch.equal(hoisted, eng.rotate_hoisted(one, [1, 5]).data)
    finally:
        eng.fused_keyswitch = True


@pytest.mark.parametrize("offset", [0, -2])
def test_rotations_take_residues_below_twice_the_prime(eng, offset):
    """Words in [q, 2q) stand for their residues, also where a rotation negates them."""

    level = offset if offset >= 0 else eng.config.public_level_count + offset
    q = torch.tensor(eng.config.moduli[level: eng.config.num_q_primes], dtype=torch.int64, device=eng.device)
    x = components(eng, level)
    a = Ciphertext(torch.stack([x, x.flip(0)]), level, eng.config.default_scale)
    above = torch.arange(eng.config.N, device=eng.device) % 3 > 0
    lazy = Ciphertext(a.data + q.unsqueeze(1) * above, level, a.scale)
    assert torch.equal(eng.rotate_by_step(lazy, 1).data, eng.rotate_by_step(a, 1).data)
    assert torch.equal(eng.rotate_by_steps(lazy, [1, 5, 1]).data, eng.rotate_by_steps(a, [1, 5, 1]).data)
    one, lazy_one = (Ciphertext(c.data[:, 0].contiguous(), level, c.scale) for c in (a, lazy))
    assert torch.equal(eng.rotate_hoisted(lazy_one, [1, 5]).data, eng.rotate_hoisted(one, [1, 5]).data)


@pytest.mark.parametrize("offset", [0, -2])
def test_device_decryption_matches_the_host_codec(eng, offset):
    """On the two rows it decodes: a 60-bit one and the last scale prime's, of every kind."""

    level = offset if offset >= 0 else eng.config.public_level_count + offset
    ct = eng.encrypt(np.random.default_rng(level).uniform(-1, 1, (2, eng.config.slots)), level=level)
    got, want = eng.decrypt_on_device(ct).cpu().numpy(), eng.decrypt(ct, crt_primes=2)
    assert np.abs(got - want).max() < 1e-9 * 2.0 ** max(0, 40 - eng.config.scale_bits)


@pytest.mark.parametrize("log_n,chain", [(12, "slots8192-scale50-levels5-int64"),
                                         (13, "slots8192-scale30-levels9-int64"),
                                         (14, "slots8192-scale50-levels5-int64"),
                                         (15, "slots16384-scale50-levels12-int64"),
                                         (16, "slots32768-scale40-levels34-int64"),
                                         (16, "slots32768-scale50-levels27-int64")])
def test_fast_transforms_match_exact_on_extreme_residues(log_n, chain):
    """Both arithmetic modes of the NTT over every QP row (in fast mode the
    60-bit primes take the 2^60 - delta folds and the 50-bit primes binary64,
    in exact mode both take Shoup products), on residues at the ends of their
    range."""

    cfg = CkksConfig.from_preset(chain).with_ring_log(log_n)
    fast, exact = CkksEngine(cfg, ntt_mode="fast", rng_seed=1), CkksEngine(cfg, ntt_mode="exact", rng_seed=1)
    q = torch.tensor(cfg.moduli, dtype=torch.int64, device=fast.device)
    uniform = Csprng(log_n, fast.device).uniform_mod(q, (), cfg.N)
    top = (q - 1).unsqueeze(1).expand_as(uniform)
    x = torch.stack([uniform, top, top * (torch.arange(cfg.N, device=q.device) % 2),
                     top * (torch.arange(cfg.N, device=q.device) == 0)])
    for name in ("forward_to_montgomery_", "forward_montgomery_"):
        a, b = x.clone(), x.clone()
        getattr(fast.runtime.ntt, name)(a, 0)
        getattr(exact.runtime.ntt, name)(b, 0)
        assert torch.equal(a, torch.remainder(b, q.unsqueeze(1)))
    for name in ("inverse_montgomery_", "inverse_to_standard_", "inverse_to_centered_"):
        a, b = x.clone(), x.clone()
        getattr(fast.runtime.ntt, name)(a, 0)
        getattr(exact.runtime.ntt, name)(b, 0)
        assert torch.equal(a, b)


@pytest.mark.parametrize("preset,level,batch,limit", [("slots32768-scale40-levels34-int64", 0, 10, 2816),
                                                      ("slots32768-scale50-levels27-int64", 0, 12, 2816),
                                                      ("slots8192-scale30-levels9-int64", 0, 36, 2816),
                                                      # three digits of 50-bit rows, all rows in one tile pass
                                                      ("slots8192-scale50-levels5-int64", 3, 48, 1500)])
def test_small_calls_match_large_ones(preset, level, batch, limit):
    """A batch large enough for the launch per arithmetic path, entry by
    entry against single-entry calls, whose digits are dealt over the waves
    of a block (shared and per-entry keys, bases, seeds, fused rescale)."""

    eng = CkksEngine(CkksConfig.from_preset(preset).with_ring_log(12), rng_seed=23)
    eng.generate_relinearization_key()
    rows = eng.config.total_num_primes - level
    assert rows * 8 * batch > limit >= rows * 8
    q = torch.tensor(eng.config.moduli[level: eng.config.num_q_primes], dtype=torch.int64, device=eng.device)
    data = Csprng(5, eng.device).uniform_mod(q, (4, batch), eng.config.N)
    a = Ciphertext(data[:2].contiguous(), level, eng.config.default_scale)
    b = Ciphertext(data[2:].contiguous(), level, eng.config.default_scale)
    steps = [1 + e % 3 for e in range(batch)]
    product, rotated = eng.hmult(a, b).data, eng.rotate_by_steps(a, steps).data
    for e in (0, 1, batch - 1):
        one_a = Ciphertext(data[:2, e: e + 1].contiguous(), level, a.scale)
        one_b = Ciphertext(data[2:, e: e + 1].contiguous(), level, a.scale)
        assert torch.equal(eng.hmult(one_a, one_b).data[:, 0], product[:, e])
        assert torch.equal(eng.rotate_by_steps(one_a, [steps[e]]).data[:, 0], rotated[:, e])


def test_small_call_sums_extreme_shares():
    """Eight digits dealt to eight waves, on a prime above 2^50: key words that
    bring every wave's share of one accumulator near (q - 1) / 2 and of its
    neighbour near -(q - 1) / 2, whose difference no binary64 integer holds."""

    eng = CkksEngine(CkksConfig(12, 50, 7, 1, 1 << 16), rng_seed=3)
    cfg, row = eng.config, 1
    q = cfg.moduli[row]
    assert q > 1 << 50 and len(eng.layout.digit_specs(0)) == 8
    # every digit is the constant 1: its transform is R mod q everywhere
    x = torch.zeros((1, cfg.num_q_primes, cfg.N), dtype=torch.int64, device=eng.device)
    x[..., 0] = 1
    key = eng.generate_relinearization_key()
    key.data.zero_()
    r_inverse = pow(1 << 62, -1, q)
    half = (q - 1) // 2 - 1000
    for digit in range(8):
        key.data[digit, :, row, 0::2] = (half - (digit == 0)) * r_inverse % q
        key.data[digit, :, row, 1::2] = -half * r_inverse % q
    assert 2 * 8 * half - 1 > 1 << 53
    want = torch.stack(eng.key_switcher.apply_key_switch(x, key, 0))
    assert torch.equal(eng.key_switcher.key_switch_fused(x, key, 0), want)
