"""The fused key switch against the per-digit op sequence it replaces
(hybrid_keyswitch.py:321-371), bit for bit, over every shipped parameter set
on a small ring: digit widths 1 to 4 (a level that cuts into the leading
digit narrows it), one to four P primes, 30-, 40- and 50-bit scale primes,
and residues at both ends of their range, where the sums of products are
largest."""

from __future__ import annotations

import pytest
import torch

from fhelium_amd import kernels as K
from fhelium_amd.config import CkksConfig, Preset
from fhelium_amd.core import Ciphertext
from fhelium_amd.csprng import Csprng
from fhelium_amd.engine import CkksEngine

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=[p.value for p in Preset])
def eng(request):
    return CkksEngine(CkksConfig.from_preset(request.param).with_ring_log(12), rng_seed=17)


def components(eng, level):
    """[3, rows, N]: uniform residues, all q - 1, and q - 1 next to 0."""

    q = torch.tensor(eng.config.moduli[level: eng.config.num_q_primes], dtype=torch.int64, device=eng.device)
    uniform = Csprng(level, eng.device).uniform_mod(q, (), eng.config.N)
    top = (q - 1).unsqueeze(1).expand_as(uniform)
    mixed = top * (torch.arange(eng.config.N, device=eng.device) % 2)
    return torch.stack([uniform, top, mixed])


@pytest.mark.parametrize("offset", [0, 1, 2, 3, -2])
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


@pytest.mark.parametrize("offset", [0, -2])
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
