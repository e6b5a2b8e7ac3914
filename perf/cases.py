"""The workloads this framework is measured on, through pyPhantom, its public API.

A case is a dict of plain values; its "op" says which call it is:

  ntt        ntt_forward / ntt_inverse of a batch of residue polynomials
  hmult      multiply_and_relin_rescale of two ciphertexts
  mulrelin   multiply_and_relin, then rescale_to_next, the reference's two calls
  rotate     one rotation with its own Galois key
  hoist      several rotations of one ciphertext, sharing the ModUp
  bsgs       an encrypted matrix-vector product with pre-encoded diagonals
  bootstrap  a whole bootstrap
  encode     host values into a plaintext
  decode     a plaintext back into host values

"bits" of a chain: q0, then nq - 1 primes of mid bits, then alpha special
primes of special bits.  Contexts, keys, encoded matrices and bootstrap keys
are made once per parameter set and kept, as a program keeps them; what a
seed draws anew are the ciphertexts, residues and slot values.
"""
import collections
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "phantom-fhe_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import pyPhantom as ph  # noqa: E402

SCALE = 2.0 ** 40


def _case(name, op, logn, q0, mid, nq, special, alpha, **more):
    return {"name": name, "op": op, "logn": logn, "q0": q0, "mid": mid, "nq": nq, "special": special, "alpha": alpha,
            **more}


def listed():
    return [
        # the smallest call: 4 primes of 50-60 bits at N = 2^13, one polynomial each way
        _case("ntt_n13_4", "ntt", 13, 60, 50, 4, 60, 1, limbs=4, batch=1, way="both"),
        # the headline batch: both polynomials of a ciphertext, 35 primes of 50 bits, N = 2^16
        _case("ntt_n16_2x35", "ntt", 16, 50, 50, 35, 60, 1, limbs=35, batch=2, way="forward"),
        # one product of a shallow circuit at the smallest ring in common use
        _case("hmult_n13_q3", "hmult", 13, 60, 40, 3, 60, 1, chain=1),
        # the reference's two calls at a lower, odd level of a mid-size chain (11 limbs, a short last digit)
        _case("mulrelin_n15_q12", "mulrelin", 15, 60, 50, 12, 60, 3, chain=2),
        # product, relinearization and rescale of a deep circuit: 24 primes, 4 special, 6 digits
        _case("hmult_n16_q24", "hmult", 16, 60, 50, 24, 60, 4, chain=1),
        # the same with one special prime: 35 digits, the key is 1.3 GB
        _case("hmult_n16_q35", "hmult", 16, 60, 50, 35, 60, 1, chain=1),
        # a rotation, the step of every slot sum and matrix product
        _case("rotate_n16_q20", "rotate", 16, 60, 40, 20, 60, 4, chain=1, step=64),
        # the baby steps of a linear transform: 7 rotations of one ciphertext, wide primes, 6 special
        _case("hoist_n16_q30", "hoist", 16, 60, 60, 30, 60, 6, chain=3, steps=7),
        # a 4096 x 4096 matrix times an encrypted vector: 64 babies, 64 giants
        _case("bsgs_n16_4096", "bsgs", 16, 60, 40, 20, 60, 4, chain=1, d_pad=4096, baby=64),
        # a bootstrap of 2^15 slots on the reference engine's chain (30 primes, 6 special)
        _case("bootstrap_n16", "bootstrap", 16, 58, 0, 30, 58, 6, evalmod="k28_r3"),
        # a full vector of slots into a plaintext of a mid-size chain
        _case("encode_n15_q12", "encode", 15, 60, 50, 12, 60, 3, chain=1),
        # the result of a computation: few limbs are left when it is decoded
        _case("decode_n15_q3", "decode", 15, 60, 50, 12, 60, 3, chain=10),
    ]


def draw(rng):
    op = rng.choice(["ntt", "ntt", "hmult", "hmult", "mulrelin", "rotate", "rotate", "hoist", "bsgs", "bootstrap",
                     "encode", "decode"])
    logn = rng.randint(12, 16)
    if op == "bootstrap":
        return _drawn(op, logn, 58, 0, 30, 58, 6, evalmod=rng.choice(["k28_r3", "cheb63"]))
    q0 = rng.choice([50, 58, 60])
    mid = rng.choice([36, 40, 45, 50, 50, 55, 60])
    if op == "ntt":
        limbs, batch = round(2 ** rng.uniform(0, 5.1)), rng.randint(1, 5)
        return _drawn(op, logn, q0, mid, limbs, 60, 1, limbs=limbs, batch=batch,
                      way=rng.choice(["forward", "inverse", "both"]))
    alpha = rng.randint(1, 6)
    nq = max(2, alpha * max(1, round(2 ** rng.uniform(1, 5) / alpha)))
    special = max(q0, mid)
    chain = rng.randint(1, max(1, nq - 1)) if rng.random() < 0.5 else 1
    if op == "rotate":
        return _drawn(op, logn, q0, mid, nq, special, alpha, chain=chain, step=rng.randint(1, (1 << logn) // 2 - 1))
    if op == "hoist":
        return _drawn(op, logn, q0, mid, nq, special, alpha, chain=chain, steps=rng.randint(2, 4 + 2 * alpha))
    if op == "bsgs":
        d = 1 << rng.randint(4, 9)
        return _drawn(op, logn, q0, mid, nq, special, alpha, chain=min(chain, nq - 1), d_pad=d,
                      baby=1 << rng.randint(1, d.bit_length() - 1))
    return _drawn(op, logn, q0, mid, nq, special, alpha, chain=chain)


def _drawn(op, *a, **more):
    c = _case("", op, *a, **more)
    del c["name"]
    return c


# ------------------------------------------------------------- what a program keeps
_kept = collections.OrderedDict()


def _keep(key, make, most=24):
    if key not in _kept:
        _kept[key] = make()
        while len(_kept) > most:
            _kept.popitem(last=False)
    _kept.move_to_end(key)
    return _kept[key]


def _chain_bits(case):
    if case["op"] == "bootstrap":
        return ph.ckks_engine_coeff_bits() if case["evalmod"] == "k28_r3" else ph.bootstrap_coeff_bits()
    return [case["q0"]] + [case["mid"]] * (case["nq"] - 1) + [case["special"]] * case["alpha"]


def _steps(case):
    op = case["op"]
    if op == "rotate":
        return [case["step"]]
    if op == "hoist":
        return [(k + 1) * ((1 << case["logn"]) // 64) for k in range(case["steps"])]
    if op == "bsgs":
        return ph.bsgs_required_steps(case["baby"])
    return []


def _stages(case):
    """The log2(slots) butterfly stages of a bootstrap's transform, in three layers."""
    k = case["logn"] - 1
    return [k // 3 + (1 if i < k % 3 else 0) for i in range(3)]


def _context(case):
    """Context, encoder and secret key of the case's parameters."""
    n, bits, steps = 1 << case["logn"], _chain_bits(case), _steps(case)

    def make():
        p = ph.params(ph.scheme_type.ckks)
        p.set_poly_modulus_degree(n)
        p.set_coeff_modulus(ph.create_coeff_modulus(n, bits))
        p.set_special_modulus_size(case["alpha"])
        if case["op"] == "bootstrap":
            p.set_galois_elts(ph.bootstrap_required_galois_elts(case["logn"], _stages(case)))
        else:
            p.set_galois_elts(ph.get_elts_from_steps(steps, n))
        ctx = ph.context(p)
        ph.set_seed(1)
        return ctx, ph.ckks_encoder(ctx), ph.secret_key(ctx).generate_sparse(ctx, 192)

    return _keep(("context", n, tuple(bits), case["alpha"], tuple(steps)), make)


def _key_id(case):
    return tuple(sorted((k, v) for k, v in case.items() if k != "name"))


def _keys(case):
    """The relinearization key, the Galois keys, the matrix's diagonals or the bootstrap key the case uses."""
    ctx, enc, sk = _context(case)
    op = case["op"]

    def make():
        ph.set_seed(2)
        if op in ("hmult", "mulrelin"):
            return {"rlk": sk.gen_relinkey(ctx)}
        if op in ("rotate", "hoist"):
            return {"glk": sk.create_galois_keys(ctx)}
        if op == "bsgs":
            # coefficients of encoded diagonals are near normal, with this deviation for entries uniform in +-1/64
            gen = torch.Generator(device=ctx.dev)
            gen.manual_seed(3)
            dev = SCALE / 64 / 3 ** 0.5 * (2 / ctx.N) ** 0.5
            co = torch.empty((case["d_pad"], ctx.N), dtype=torch.int64, device=ctx.dev)
            for d in range(0, case["d_pad"], 256):
                part = co[d:d + 256]
                part.copy_((torch.randn(part.shape, dtype=torch.float64, device=ctx.dev, generator=gen) * dev).round())
            diags = ph.bsgs_diagonals(co, SCALE, case["d_pad"], case["baby"])
            diags.expanded(ctx, case["chain"])
            return {"glk": sk.create_galois_keys(ctx), "diags": diags}
        if op == "bootstrap":
            more = {"eval_mod_levels": 9, "user_scale": SCALE} if case["evalmod"] == "k28_r3" else {}
            return {"bk": ph.create_bootstrap_key(ctx, enc, sk, sparse_hamming_weight=192, evalmod=case["evalmod"],
                                                  stages_per_layer=_stages(case), **more)}
        return {}

    return _keep(("keys",) + _key_id(case), make)


def _residues(ctx, batch, limbs, gen):
    t = torch.empty((batch, limbs, ctx.N), dtype=torch.int64, device=ctx.dev)
    for l in range(limbs):
        t[:, l] = torch.randint(0, ctx.moduli[l], (batch, ctx.N), dtype=torch.int64, device=ctx.dev, generator=gen)
    return t.view(torch.uint64)


# ------------------------------------------------------------- the cases
def prepare(case, seed):
    ctx, enc, sk = _context(case)
    op = case["op"]
    rng = np.random.default_rng([seed, case["logn"]])
    s = {"op": op, "ctx": ctx, "enc": enc, **_keys(case)}
    if op == "ntt":
        gen = torch.Generator(device=ctx.dev)
        gen.manual_seed(seed)
        s.update(way=case["way"], limbs=case["limbs"], batch=case["batch"])
        s["x"] = _residues(ctx, case["batch"], case["limbs"], gen)
        if case["way"] == "both":
            s["y"] = _residues(ctx, case["batch"], case["limbs"], gen)
        return s
    n_slots = enc.slot_count()
    if op in ("encode", "decode"):
        v = rng.uniform(-1, 1, n_slots)
        s["chain"] = case["chain"]
        if op == "encode":
            s["values"] = v
        else:
            s["pt"] = enc.encode_double_vector(ctx, v, SCALE, case["chain"])
        return s

    def fresh(chain, period=None):
        v = rng.uniform(-1, 1, period or n_slots)
        v = np.tile(v, n_slots // v.size)
        return sk.encrypt_symmetric(ctx, enc.encode_double_vector(ctx, v, SCALE, chain), seed=rng)

    if op == "bootstrap":
        s["a"] = fresh(ctx.size_Q - (1 if case["evalmod"] == "k28_r3" else 0))
        return s
    s["a"] = fresh(case["chain"], case.get("d_pad"))
    if op in ("hmult", "mulrelin"):
        s["b"] = fresh(case["chain"])
    s["steps"] = _steps(case)
    return s


def run(s):
    r = _run(s)
    # residues as int64: torch has few operations on uint64
    return r if isinstance(r, np.ndarray) else [t.view(torch.int64) for t in r]


def _run(s):
    op, ctx = s["op"], s["ctx"]
    if op == "ntt":
        if s["way"] != "inverse":
            ph.ntt_forward(ctx, s["x"], s["limbs"], 0, s["batch"])
        if s["way"] != "forward":
            ph.ntt_inverse(ctx, s["y"] if s["way"] == "both" else s["x"], s["limbs"], 0, s["batch"])
        return [s["x"], s["y"]] if s["way"] == "both" else [s["x"]]
    if op == "hmult":
        return [ph.multiply_and_relin_rescale(ctx, s["a"], s["b"], s["rlk"]).data]
    if op == "mulrelin":
        return [ph.rescale_to_next(ctx, ph.multiply_and_relin(ctx, s["a"], s["b"], s["rlk"])).data]
    if op == "rotate":
        return [ph.rotate(ctx, s["a"], s["steps"][0], s["glk"]).data]
    if op == "hoist":
        return [c.data for c in ph.hoist_rotations(ctx, s["a"], s["glk"], s["steps"])]
    if op == "bsgs":
        return [ph.bsgs_matmul_preencoded(ctx, s["glk"], s["a"], s["diags"]).data]
    if op == "bootstrap":
        return [ph.bootstrap(ctx, s["enc"], s["a"], s["bk"], SCALE).data]
    if op == "encode":
        return [s["enc"].encode_double_vector(ctx, s["values"], SCALE, s["chain"]).data]
    return np.array(s["enc"].decode_double_vector(ctx, s["pt"]))


def work(case):
    """Bytes: every operand, key limb and plaintext the level reads, once, and the result, once.  Operations: a
    butterfly is a modular product and two sums (3); a base conversion or key product is 2 per term."""
    n, log, a, op = 1 << case["logn"], case["logn"], case["alpha"], case["op"]
    limb, ntt = 8 * n, 1.5 * n * log
    if op == "ntt":
        k = case["limbs"] * case["batch"] * (2 if case["way"] == "both" else 1)
        return {"bytes": 2 * k * limb, "flops": k * ntt}
    if op in ("encode", "decode"):
        L = case["nq"] - case["chain"] + 1
        fft = 2.5 * n * log  # a complex transform of n / 2 points
        return {"bytes": (L + 0.5) * limb, "flops": L * (ntt + 4 * n) + fft}

    def switch(L, rotations=1):
        """One ModUp, then `rotations` key products and ModDowns over L primes: (key limbs, operations)."""
        beta = -(-L // a)
        return (2 * beta * (L + a) * rotations,
                (L + beta * (L + a) + 2 * rotations * (a + L)) * ntt + 2 * n * L * (L + a) +
                rotations * (4 * n * beta * (L + a) + 4 * n * a * L))

    if op == "bootstrap":
        # 6 transform layers of 2^(s+1) - 1 diagonals in about 2^((s+3)/2) - 2 rotations each, some 40 key switches between
        rot = sum(2 * (2 ** ((s + 3) / 2) - 2) for s in _stages(case))
        diag = sum(2 * (2 ** (s + 1) - 1) for s in _stages(case))
        k, f = switch(20)
        return {"bytes": (0.5 * rot * 2 * 5 * 36 + diag * 20 + 2 * (30 + 11)) * limb, "flops": (rot + 40) * f}
    L = case["nq"] - case["chain"] + 1
    if op in ("hmult", "mulrelin"):
        k, f = switch(L)
        return {"bytes": (4 * L + k + 2 * (L - 1)) * limb, "flops": f + 7 * n * L + 2 * L * ntt}
    if op == "rotate":
        k, f = switch(L)
        return {"bytes": (4 * L + k) * limb, "flops": f}
    if op == "hoist":
        k, f = switch(L, case["steps"])
        return {"bytes": (2 * L + 2 * L * case["steps"] + k) * limb, "flops": f}
    d, baby = case["d_pad"], case["baby"]
    k, f = switch(L)
    packed = [(5 if b <= 40 else 8) / 8 for b in _chain_bits(case)[:L]]
    return {"bytes": (d * sum(packed) + len(_steps(case)) * k + 4 * L) * limb,
            "flops": (baby + d // baby - 2) * f + 4 * d * L * n}


def tolerance(case):
    """Residues are whole numbers and come out the same; decoded slots are a double-precision transform of the same
    integers (numpy's, with its sums in another order, is 3e-16 of their norm away)."""
    return {"rel": 1.5e-15, "max": 1.5e-14} if case["op"] == "decode" else "exact"


def exact(case, seed):
    """The slots a decode case returns: the encoded values' integer coefficients, read back in double precision."""
    if case["op"] != "decode":
        return None
    n = 1 << case["logn"]
    v = np.random.default_rng([seed, case["logn"]]).uniform(-1, 1, n // 2)
    # slot j is m(zeta^(5^j)), zeta = exp(i pi / n): index t_j = (5^j mod 2n - 1) / 4 of a twisted DFT of n / 2 points
    t, p = np.empty(n // 2, dtype=np.int64), 1
    for j in range(n // 2):
        t[j], p = (p - 1) // 4, p * 5 % (2 * n)
    w = np.empty(n // 2, dtype=np.complex128)
    w[t] = v
    twist = np.exp(1j * np.pi * np.arange(n // 2) / n)
    z = np.fft.fft(w) / (n // 2) / twist * SCALE
    z = (np.rint(z.real) + 1j * np.rint(z.imag)) / SCALE
    return (np.fft.ifft(z * twist) * (n // 2))[t].real
