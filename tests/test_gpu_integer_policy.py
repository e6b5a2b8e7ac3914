"""The integer arithmetic policy (primes from 2^50 to 2^61) at the edges of its
ranges, bit for bit against the oracle: primes just above 2^50, just below and
above 2^60 (values hold 8 q below, 4 q above) and near 2^61, with residues that
drive the lazy bounds (all 0, all q - 1, the two alternating) as well as random
ones; and base conversions on both sides of the rules that pick how they sum
(one input, up to seven inputs by 30-bit limbs, more inputs or primes of 2^60
and above by wider sums), with narrow and wide primes mixed.
"""
import numpy as np
import pytest

import py_oracle as O
from gpu_util import _is_prime64, empty, first_mismatch, to_dev, to_host, uniform_limbs

pytestmark = pytest.mark.gpu


def _primes(N, near, count, down):
    """`count` primes q = 1 mod 2N next to `near`, below or above it."""
    step = 2 * N
    q = (near - 1) // step * step + 1
    if not down:
        q += step
    out = []
    while len(out) < count:
        if _is_prime64(q) and (q < near) == down:
            out.append(q)
        q += -step if down else step
    return out


def _edge_primes(N):
    return (_primes(N, 1 << 50, 1, True) + _primes(N, 1 << 50, 1, False) + _primes(N, 1 << 55, 1, True)
            + _primes(N, 1 << 60, 2, True) + _primes(N, 1 << 60, 1, False) + _primes(N, 1 << 61, 1, True))


def _extremes(rng, moduli, N):
    """[4][L][N]: random residues, zeros, q - 1 everywhere, 0 and q - 1 in turn."""
    q1 = np.array(moduli, dtype=np.uint64)[:, None] - np.uint64(1)
    x = np.zeros((4, len(moduli), N), dtype=np.uint64)
    x[0] = uniform_limbs(rng, (len(moduli), N), moduli)
    x[2] = q1
    x[3, :, 1::2] = q1
    return x


@pytest.mark.parametrize("logN", [10, 11, 13, 14, 16, 17])
def test_ntt_edge_primes(dev, logN):
    import pfa_native as P

    N = 1 << logN
    mods = _edge_primes(N)
    ctx, orc = P.NativeContext(N, mods, 1), O.Oracle(N, mods, 1)
    x = _extremes(np.random.default_rng(logN), mods, N)
    for repeat in (1, 12):  # 28 limbs, and enough for the large-batch inverse rows pass
        d = to_dev(np.concatenate([x] * repeat), dev)
        ctx.ntt_forward(d, 4 * repeat, len(mods), 0)
        want = orc.ntt_fwd(x)
        got = to_host(d).reshape(repeat, *x.shape)
        assert all(np.array_equal(g, want) for g in got), first_mismatch(got[0], want)
        d = to_dev(np.concatenate([x] * repeat), dev)
        ctx.ntt_inverse(d, 4 * repeat, len(mods), 0)
        want = orc.ntt_inv(x)
        got = to_host(d).reshape(repeat, *x.shape)
        assert all(np.array_equal(g, want) for g in got), first_mismatch(got[0], want)


@pytest.mark.parametrize("logN", [13, 14])
@pytest.mark.parametrize("kind", ["narrow", "wide", "mixed"])
def test_rows_passes_with_and_without_stage(dev, logN, kind):
    """N = 2^13 and 2^14: the forward rows pass with integer twiddles in LDS up to three tiles a CU, without beyond and
    for 50-bit primes alone; the inverse one with them for any integer prime from 48 limbs on."""
    import pfa_native as P
    import torch

    N = 1 << logN
    narrow, wide = _primes(N, 1 << 50, 3, True), _primes(N, 1 << 60, 3, True)
    mods = {"narrow": narrow, "wide": wide, "mixed": narrow[:2] + wide[:1]}[kind]
    ctx, orc = P.NativeContext(N, mods, 1), O.Oracle(N, mods, 1)
    x = _extremes(np.random.default_rng(logN), mods, N)
    tiles = N // 128 // 32  # of a limb: rows of 128, 32 a tile
    most = torch.cuda.get_device_properties(dev).multi_processor_count * 3 // tiles // len(mods)  # polys
    for batch in (4, 16, most, most + 1):
        y = np.concatenate([x] * (batch // 4 + 1))[:batch]
        for transform, check in ((ctx.ntt_forward, orc.ntt_fwd), (ctx.ntt_inverse, orc.ntt_inv)):
            d = to_dev(y, dev)
            transform(d, batch, len(mods), 0)
            want, got = check(x), to_host(d)
            for k in range(batch):
                assert np.array_equal(got[k], want[k % 4]), (batch, k, first_mismatch(got[k], want[k % 4]))


def _chain(N, kind, nq, alpha):
    """Data primes then special primes of a kind."""
    if kind == "wide":  # all just below 2^60
        return _primes(N, 1 << 60, nq + alpha, True)
    if kind == "small":  # all just below 2^50
        return _primes(N, 1 << 50, nq + alpha, True)
    if kind == "mixed":  # narrow and wide data primes in turn, wide special ones
        w, n = _primes(N, 1 << 60, nq + alpha, True), _primes(N, 1 << 50, nq, True)
        return [(w if i % 3 == 0 else n)[i] for i in range(nq)] + w[nq:]
    if kind == "narrow":  # narrow data primes, wide special ones
        return _primes(N, 1 << 50, nq, True) + _primes(N, 1 << 59, alpha, True)
    return _primes(N, 1 << 61, nq + alpha, True)  # "tight": above 2^60


_SHAPES = [(logN, nq, alpha, kind) for logN in (10, 13) for nq, alpha in ((3, 1), (4, 2), (12, 6), (14, 7), (8, 8))
           for kind in ("wide", "mixed", "narrow", "small", "tight")]
# rounds of 16 and 32 elements, and the inner product without staged twiddles (N = 2^17)
_SHAPES += [(logN, nq, alpha, kind) for logN in (14, 16, 17) for nq, alpha in ((4, 2), (8, 8))
            for kind in ("mixed", "tight")]


@pytest.mark.parametrize("logN,nq,alpha,kind", _SHAPES)
def test_conversions_edge(dev, logN, nq, alpha, kind):
    """multiply, relinearize and rescale (the fused conversion of alpha + 1
    inputs), then relinearize alone (ModUp and ModDown of alpha inputs), at the
    top and at a level with a short last digit."""
    import pfa_native as P

    N = 1 << logN
    mods = _chain(N, kind, nq, alpha)
    ctx, orc = P.NativeContext(N, mods, alpha), O.Oracle(N, mods, alpha)
    rng = np.random.default_rng(nq * alpha + logN)
    key = uniform_limbs(rng, (orc.dnum, 2, nq + alpha, N), mods)
    dkey = to_dev(key, dev)
    for chain in (1, 2):
        L = orc.size_Ql(chain)
        x = _extremes(rng, mods[:L], N)
        for a, b in ((x[[0, 0]], x[[0, 2]]), (x[[2, 2]], x[[2, 2]]), (x[[3, 2]], x[[1, 3]])):
            want = orc.multiply_and_relin(chain, a, b, key)
            da, db = to_dev(a, dev), to_dev(b, dev)
            out, res = empty((2, L, N), dev), empty((2, L - 1, N), dev)
            ctx.multiply_and_relin(chain, da, db, dkey, out)
            got = to_host(out)
            assert np.array_equal(got, want), first_mismatch(got, want)
            ctx.multiply_relin_rescale(chain, da, db, dkey, res)
            got, want = to_host(res), orc.rescale(chain, want)
            assert np.array_equal(got, want), first_mismatch(got, want)
