"""The encoder's two-launch FFT at every ring size: both parts take 4 to 8 stages (N = 2^10 .. 2^17), and a
round of three stages is followed by a last one of 1, 2 or 3.

The oracle is numpy's FFT of the same twisted vector.  Both transforms are sums of M terms in log2(M) rounded
stages, so a value is off by at most about log2(M) 2^-52 times the sum of the terms' magnitudes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _slot_index(n):
    t, p = np.empty(n // 2, dtype=np.int64), 1
    for j in range(n // 2):
        t[j], p = (p - 1) // 4, p * 5 % (2 * n)
    return t


@pytest.mark.parametrize("logn", range(10, 18))
@pytest.mark.parametrize("fill", ["full", "one", "odd"])
def test_encode_decode_against_numpy(logn, fill):
    import pyPhantom as ph

    n = 1 << logn
    m = n // 2
    p = ph.params(ph.scheme_type.ckks)
    p.set_poly_modulus_degree(n)
    p.set_coeff_modulus(ph.create_coeff_modulus(n, [60, 40, 50, 60]))
    p.set_special_modulus_size(1)
    ctx = ph.context(p)
    enc = ph.ckks_encoder(ctx)
    rng = np.random.default_rng(logn)
    count = {"full": m, "one": 1, "odd": m // 2 + 1}[fill]
    v = rng.uniform(-1, 1, count) + 1j * rng.uniform(-1, 1, count)
    scale = 2.0 ** 40
    pt = enc.encode_complex_vector(ctx, v, scale, 1)

    t = _slot_index(n)
    w = np.zeros(m, dtype=np.complex128)
    w[t[:count]] = v
    twist = np.exp(1j * np.pi * np.arange(m) / n)
    z = np.fft.fft(w) / m / twist * scale
    want = np.concatenate([z.real, z.imag])
    bound = 0.5 + 2 * (logn + 2) * 2.0 ** -52 * scale * np.abs(v).sum() / m

    coef = pt.data.clone()
    ph.ntt_inverse(ctx, coef, coef.shape[0], 0, 1)
    coef = coef.cpu().numpy()
    got = None
    for l in range(coef.shape[0]):
        q = ctx.moduli[l]
        c = coef[l].astype(np.int64)
        c = np.where(c > q // 2, c - q, c)
        assert got is None or np.array_equal(c, got), l  # every prime holds the same integers (|m_k| < q / 2)
        got = c
        if np.abs(want).max() + 1 >= min(ctx.moduli[:3]) / 2:
            break
    assert np.abs(got - want).max() <= bound

    # a 40-bit prime cannot tell coefficients of more bits apart: decode composes all limbs
    back = np.array(enc.decode_complex_vector(ctx, pt))
    zi = (got[:m] + 1j * got[m:]) / scale
    exact = (np.fft.ifft(zi * twist) * m)[t]
    assert np.abs(back - exact).max() <= 2 * (logn + 2) * 2.0 ** -52 * np.abs(zi).sum()


def test_encode_refuses_what_does_not_fit():
    """The size check's verdict comes from the device; the next call on the same stream starts it anew."""
    import pyPhantom as ph

    n = 1 << 12
    p = ph.params(ph.scheme_type.ckks)
    p.set_poly_modulus_degree(n)
    p.set_coeff_modulus(ph.create_coeff_modulus(n, [50, 40, 50]))
    p.set_special_modulus_size(1)
    ctx = ph.context(p)
    enc = ph.ckks_encoder(ctx)
    v = np.ones(n // 2)
    for bad in (2.0 ** 60, np.inf, np.nan):
        with pytest.raises(Exception, match="too large"):
            enc.encode_double_vector(ctx, v * bad, 2.0 ** 40, 1)
        pt = enc.encode_double_vector(ctx, v, 2.0 ** 40, 1)
        assert np.abs(np.array(enc.decode_double_vector(ctx, pt)) - 1).max() < 1e-9


@pytest.mark.parametrize("form", ["list", "reversed", "readonly", "strided", "float32", "2d"])
def test_real_vectors_as_complex_ones(form):
    """encode_double_vector gives encode_complex_vector's plaintext for any array or list of reals, and
    decode_double_vector the real parts of decode_complex_vector."""
    import pyPhantom as ph
    import torch

    n = 1 << 11
    p = ph.params(ph.scheme_type.ckks)
    p.set_poly_modulus_degree(n)
    p.set_coeff_modulus(ph.create_coeff_modulus(n, [60, 40, 50, 60]))
    p.set_special_modulus_size(1)
    ctx = ph.context(p)
    enc = ph.ckks_encoder(ctx)
    v = np.random.default_rng(5).uniform(-1, 1, 600)
    if form == "readonly":
        v.flags.writeable = False
    x = {"list": v.tolist(), "reversed": v[::-1], "readonly": v, "strided": v[::3], "float32": v.astype(np.float32),
         "2d": v.reshape(20, 30).T}[form]
    a = enc.encode_double_vector(ctx, x, 2.0 ** 40)
    b = enc.encode_complex_vector(ctx, np.array(x, dtype=np.complex128), 2.0 ** 40)
    assert torch.equal(a.data.view(torch.int64), b.data.view(torch.int64))
    got = enc.decode_double_vector(ctx, a)
    assert isinstance(got, list) and got == [z.real for z in enc.decode_complex_vector(ctx, b)]
