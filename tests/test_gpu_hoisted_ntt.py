"""Hoisted rotations left in the NTT domain (fh_keyswitch_hoisted_ntt) against
the hoisted rotations in the coefficient domain followed by the forward
transform: the same canonical residues, bit for bit, over every shipped
parameter set (digit widths, one to four P primes; chains whose rows do not
allow it take the general path), ring sizes, levels and residues at both ends
of their range."""

from __future__ import annotations

import pytest
import torch

from fhelium_amd.config import CkksConfig, Preset
from fhelium_amd.core import Ciphertext, CkksStateError, ScaleMismatchError
from fhelium_amd.csprng import Csprng
from fhelium_amd.engine import CkksEngine

pytestmark = pytest.mark.gpu

LARGE = max(Preset, key=lambda p: CkksConfig.from_preset(p).catalog_ring_dimension).value
CASES = [(p.value, 12) for p in Preset] + [(LARGE, n) for n in (13, 14, 15, 16)]


@pytest.mark.parametrize("preset,log_n", CASES)
def test_equals_transform_of_coefficient_domain_rotations(preset, log_n):
    eng = CkksEngine(CkksConfig.from_preset(preset).with_ring_log(log_n), rng_seed=23)
    cfg = eng.config
    steps = [1, 5, cfg.slots - 3]
    for level in sorted({0, 1, cfg.public_level_count // 2, cfg.public_level_count - 2}):
        q = torch.tensor(cfg.moduli[eng.runtime.row_start(level): cfg.num_q_primes], dtype=torch.int64,
                         device=eng.device)
        uniform = Csprng(level, eng.device).uniform_mod(q, (), cfg.N)
        top = (q - 1).unsqueeze(1).expand_as(uniform)
        mixed = top * (torch.arange(cfg.N, device=eng.device) % 2)
        for c0, c1 in ((uniform, uniform.flip(1)), (top, top), (mixed, uniform), (top - mixed, mixed)):
            ct = Ciphertext(torch.stack([c0, c1]), level, cfg.default_scale)
            want = eng.coefficient_domain_to_ntt_domain(eng.rotate_hoisted(ct, steps)).data % q.unsqueeze(1)
            got = eng.rotate_hoisted_ntt(ct, steps)
            assert (got.polynomial_domain, got.residue_representation) == ("ntt", "montgomery")
            assert torch.equal(got.data % q.unsqueeze(1), want)
            if eng.key_switcher.hoisted_ntt_ready(level):
                assert torch.equal(got.data, want)
        given = eng.rotate_hoisted_ntt(ct, steps[:1], eng.coefficient_domain_to_ntt_domain(ct))
        assert torch.equal(given.data % q.unsqueeze(1), want[:, :1])


def test_general_path_keeps_every_step_and_error():
    eng = CkksEngine(CkksConfig.from_preset(list(Preset)[0]).with_ring_log(12), rng_seed=24)
    ct = eng.encrypt([0.5, -0.25], level=1)
    q = torch.tensor(eng.config.moduli[eng.runtime.row_start(1): eng.config.num_q_primes], device=eng.device)
    got = eng.rotate_hoisted_ntt(ct, [0, 2]).data % q.unsqueeze(1)  # step 0: the ciphertext itself
    want = eng.coefficient_domain_to_ntt_domain(eng.rotate_hoisted(ct, [0, 2])).data % q.unsqueeze(1)
    assert torch.equal(got, want)
    batched = eng.encrypt([[0.5], [0.25]], level=1)
    with pytest.raises(ValueError, match="unbatched"):
        eng.rotate_hoisted_ntt(batched, [1])


@pytest.mark.parametrize("preset", ["slots8192-scale40-levels7-int64", "slots8192-scale50-levels5-int64"])
def test_given_transform_must_be_the_ciphertexts(preset):
    """On the NTT-domain path and on the general one."""

    eng = CkksEngine(CkksConfig.from_preset(preset).with_ring_log(12), rng_seed=25)
    ct = eng.encrypt([0.5, -0.25], level=1)
    ntt = eng.coefficient_domain_to_ntt_domain(ct)
    with pytest.raises(CkksStateError, match="ntt-domain"):
        eng.rotate_hoisted_ntt(ct, [1, 2], ct)
    with pytest.raises(ScaleMismatchError):
        eng.rotate_hoisted_ntt(ct, [1, 2], Ciphertext(ntt.data, 1, 2 * ct.scale, "ntt", "montgomery"))
    with pytest.raises(ValueError, match="level"):
        eng.rotate_hoisted_ntt(ct, [1, 2], Ciphertext(ntt.data, 2, ct.scale, "ntt", "montgomery"))
    with pytest.raises(ValueError, match="shape"):
        eng.rotate_hoisted_ntt(ct, [1, 2], Ciphertext(ntt.data[:, 1:], 1, ct.scale, "ntt", "montgomery"))
