"""The two-pass codec (fh_ckks_encode_coefficients, fh_ntt_forward_lifted,
fh_ckks_lift_montgomery, fh_ckks_decode_rows, fh_ckks_decrypt_decode) on every
ring it takes: encoded residues equal the one-launch-per-stage encoder's bit
for bit (same butterflies, same rounding), whatever the coefficients' size;
decoded slots equal the host codec's of the same residues."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from fhelium_amd import _native as nat
from fhelium_amd import codec
from fhelium_amd import kernels as K
from fhelium_amd.config import CkksConfig
from fhelium_amd.core import Ciphertext, SecretKey
from fhelium_amd.engine import CkksEngine

pytestmark = pytest.mark.gpu

PRESETS = {12: "slots8192-scale50-levels5-int64", 13: "slots8192-scale30-levels9-int64",
           14: "slots8192-scale40-levels7-int64", 15: "slots16384-scale50-levels12-int64",
           16: "slots32768-scale40-levels34-int64"}


@pytest.fixture(scope="module", params=sorted(PRESETS))
def eng(request):
    e = CkksEngine(CkksConfig.from_preset(PRESETS[request.param]).with_ring_log(request.param), rng_seed=31)
    e.generate_secret_key()
    return e


def slots(eng, batch, seed):
    rng = np.random.default_rng(seed)
    shape = (batch, eng.config.slots)
    return rng.uniform(-1, 1, shape) + 1j * rng.uniform(-1, 1, shape)


# 2^40 and 2^52 bracket the lift's short form (|c| < 2^50), 2^61 its widest input
@pytest.mark.parametrize("scale_bits,batch", [(40, 3), (52, 1), (61, 2)])
def test_encode_equals_the_stage_encoder(eng, scale_bits, batch):
    cfg = eng.config
    z = torch.from_numpy(slots(eng, batch, scale_bits)).to(eng.device)
    level, scale = 1, float(1 << scale_bits)
    rows = eng.layout.prime_ids(level)
    moduli = torch.tensor([cfg.moduli[i] for i in rows], dtype=torch.int64, device=eng.device)
    ws = torch.empty((batch, cfg.N, 2), dtype=torch.float64, device=eng.device)
    want = torch.empty((batch, len(rows), cfg.N), dtype=torch.int64, device=eng.device)
    nat.call("fh_ckks_encode", torch.view_as_real(z).data_ptr(), batch, cfg.logN, eng._slot_positions().data_ptr(),
             scale, moduli.data_ptr(), len(rows), ws.data_ptr(), want.data_ptr(), nat.stream_ptr(eng.device))
    ntt = want.clone()
    eng.runtime.ntt.forward_to_montgomery_(ntt, level)
    K.to_montgomery_(want, eng.runtime.params(level))
    assert torch.equal(eng.encode_on_device(z, level=level, scale=scale).data, want)
    assert torch.equal(eng.encode_on_device(z, level=level, scale=scale, polynomial_domain="ntt").data, ntt)
    # fewer slots, real values and a strided input take the padded copy
    short = z[:, ::2].real
    padded = torch.zeros_like(z)
    padded[:, : short.size(1)] = short
    assert torch.equal(eng.encode_on_device(short, level=level, scale=scale).data,
                       eng.encode_on_device(padded, level=level, scale=scale).data)
    # conjugate and negative views are read as the values they stand for
    for lazy, plain in ((z.conj(), z.conj_physical()), (torch._neg_view(z), -z)):
        assert torch.equal(eng.encode_on_device(lazy, level=level, scale=scale).data,
                           eng.encode_on_device(plain, level=level, scale=scale).data)


@pytest.mark.parametrize("batch", [1, 5])
def test_decrypt_equals_the_host_codec(eng, batch):
    level = eng.config.public_level_count - 2
    x = slots(eng, batch, batch)
    ct = eng.encrypt(x, level=level)
    want = eng.decrypt(ct, crt_primes=2)
    tol = 1e-9 * 2.0 ** max(0, 40 - eng.config.scale_bits)
    assert np.abs(eng.decrypt_on_device(ct).cpu().numpy() - want).max() < tol
    # NTT-domain and three-component values, a view of more rows, a strided batch
    ntt = eng.coefficient_domain_to_ntt_domain(ct)
    assert np.abs(eng.decrypt_on_device(ntt).cpu().numpy() - want).max() < tol
    square = eng.multiply(ntt, ntt)
    dec = eng.decrypt_on_device(square).cpu().numpy()
    assert np.abs(dec - eng.decrypt(square, crt_primes=2)).max() < tol
    viewed = eng.mod_switch_to_level_(eng.encrypt(x, level=0), level)
    assert np.abs(eng.decrypt_on_device(viewed).cpu().numpy() - eng.decrypt(viewed, crt_primes=2)).max() < tol
    wide = torch.empty((*ct.data.shape[:-1], 2 * eng.config.N), dtype=torch.int64, device=eng.device)[..., ::2]
    wide.copy_(ct.data)
    strided = Ciphertext(wide, level, ct.scale)
    assert torch.equal(eng.decrypt_on_device(strided), eng.decrypt_on_device(ct))


def test_decode_of_extreme_residues(eng):
    """Residues at the ends of their range, near both halves of q_a q_b."""

    cfg = eng.config
    level = cfg.public_level_count - 1
    start = cfg.num_q_primes - 2
    qb, qa = cfg.moduli[start], cfg.moduli[start + 1]
    big = [0, 1, qa - 1, qa, qa * qb // 2, qa * qb // 2 + 1, qa * qb - 1, 3 * qa + 5, qa * qb - 3 * qa]
    x = [big[i % len(big)] for i in range(cfg.N)]
    res = torch.tensor([[v % qb for v in x], [v % qa for v in x]], dtype=torch.int64, device=eng.device)
    zero = torch.zeros_like(res)
    got = eng.decrypt_on_device(Ciphertext(torch.stack([res, zero]), level, 1.0)).cpu().numpy()
    centred = np.array([float(v - qa * qb if v > qa * qb // 2 else v) for v in x])
    want = codec.embed(centred)
    assert np.abs(got - want).max() < 1e-12 * np.abs(want).max()


def test_decrypt_with_other_secret_keys(eng):
    """A strided secret key decrypts; one of another ring, row count or type is refused."""

    ct = eng.encrypt(slots(eng, 2, 9), level=1)
    want = eng.decrypt_on_device(ct)
    secret = eng.secret_key
    data = torch.empty((*secret.data.shape[:-1], 2 * eng.config.N), dtype=torch.int64, device=eng.device)[..., ::2]
    data.copy_(secret.data)
    rows = eng.config.num_q_primes
    try:
        eng.secret_key = SecretKey(data, secret.coefficients)
        assert torch.equal(eng.decrypt_on_device(ct), want)
        for bad in (secret.data[:, ::2].contiguous(), secret.data[: rows - 1].contiguous(), secret.data[1:, :1],
                    secret.data.to(torch.int32)):
            eng.secret_key = SecretKey(bad, secret.coefficients)
            with pytest.raises((RuntimeError, TypeError)):
                eng.decrypt_on_device(ct)
    finally:
        eng.secret_key = secret
