"""The work a user of this package has a GPU do, as cases for timing: sizes, inputs, and one pass through the entry points.

Two layers are called, as programs call them: `Context` (the kernel-level interface: device tensors of residues
[polys][limbs][N] in, device tensors out) and `hellm.HEMMer` (encrypted matrices: handles in and out, numpy matrices at
either end, so a pass ends where the program gets its matrix back).  N = 2^log_n is the ring degree; a HEMMer of
ring degree N works on n x n tiles, 2 n^2 = N / 2.  The common parameter set is the package's preset: N = 2^16, a 60-bit prime
and twelve 42-bit ones in the chain, four 60-bit special primes, three key-switching digits.
"""
import importlib
import math

import numpy as np
import torch

PKG = "encryption-friendly_llm_architecture_amd"
CHAIN, SPECIAL, DNUM, LOG_SCALE = 13, 4, 3, 42   # the preset's shape
_kept = {}                                      # contexts and evaluators: made once, as a program does


def _package():
    return importlib.import_module(PKG), importlib.import_module(PKG + ".hellm")


def _moduli(log_n, chain, special, bits):
    """(chain primes, special primes): `bits` 60: all of 60 bits; 42: one of 60 bits, then primes below 2^42."""
    pkg, _ = _package()
    if bits == 60:
        p = pkg.primes_below(60, log_n, chain + special)
        return p[:chain], p[chain:]
    big = pkg.primes_below(60, log_n, 1 + special)
    return big[:1] + (pkg.primes_below(42, log_n, chain - 1) if chain > 1 else []), big[1:]


def _context(log_n, chain, special, dnum, bits):
    key = ("context", log_n, chain, special, dnum, bits)
    if key not in _kept:
        q, p = _moduli(log_n, chain, special, bits)
        _kept[key] = _package()[0].Context(log_n, q, p, dnum)
    return _kept[key]


def _hemmer(log_n, lowest=3):
    """The evaluator with its keys.  lowest: the level the preset's products refuse to go below."""
    key = ("hemmer", log_n, lowest)
    if key not in _kept:
        hellm = _package()[1]
        if log_n == 16:
            preset = hellm.HEMMer(preset=True, seed=3)
            _kept["hemmer", 16, 3] = preset
            if lowest != 3:
                _kept[key] = hellm.HEMMer(16, preset.q, preset.p, dnum=preset.dnum, min_bootstrap_level=lowest, seed=3)
        else:
            q, p = _moduli(log_n, CHAIN, SPECIAL, 42)
            _kept[key] = hellm.HEMMer(log_n, q, p, dnum=DNUM, log_scale=LOG_SCALE, min_bootstrap_level=lowest, seed=3)
    return _kept[key]


def listed():
    return [
        # A batch of transforms as a bootstrapping-sized or multi-input step issues them: 32 polynomials of 24 limbs.
        {"name": "ntt_32x24_60bit", "kind": "ntt", "log_n": 16, "polys": 32, "limbs": 24, "bits": 60, "inverse": False},
        # A few polynomials on a smaller ring, back to coefficients.
        {"name": "intt_ring14_5x7", "kind": "ntt", "log_n": 14, "polys": 5, "limbs": 7, "bits": 42, "inverse": True},
        # The smallest call: one slot rotation of one ciphertext on a small ring.
        {"name": "rotate_ring13_level5", "kind": "rotate", "log_n": 13, "chain": 6, "special": 2, "dnum": 3, "bits": 42, "level": 5, "step": 1},
        # One slot rotation on a long chain: level 20 of 24 primes of 60 bits.
        {"name": "rotate_60bit_level20", "kind": "rotate", "log_n": 16, "chain": 24, "special": 4, "dnum": 3, "bits": 60, "level": 20, "step": 64},
        # A slot-wise product of two ciphertexts in the middle of a computation: tensor, relinearise, rescale.
        {"name": "mult_level9", "kind": "mult", "log_n": 16, "chain": CHAIN, "special": SPECIAL, "dnum": DNUM, "bits": 42, "level": 9},
        # The client's side: a matrix encrypted, a matrix decrypted, from and to host memory.
        {"name": "client_128", "kind": "client", "log_n": 16, "rows": 128, "cols": 128, "pair": False},
        # The weights of a layer encoded as plaintexts of the level they are used at: 9 groups of four 128 x 128 tiles.
        {"name": "encode_9_weights", "kind": "encode", "log_n": 16, "messages": 9, "level": 5},
        # A product of two encrypted 32 x 32 tiles on a small ring: launches count.
        {"name": "ccmm_32", "kind": "ccmm", "log_n": 12, "pair": False, "level": 12, "target": 4},
        # The product of two encrypted 128 x 128 matrices, fresh from encryption.
        {"name": "ccmm_128", "kind": "ccmm", "log_n": 16, "pair": False, "level": 12, "target": 4},
        # Encrypted activations times plaintext weights, two 128 x 128 products in one ciphertext.
        {"name": "pcmm_128_pair", "kind": "pcmm", "log_n": 16, "pair": True, "level": 12, "target": 4},
        # The frozen projection of a 768-wide layer: 6 activation tiles against 36 weight tiles, hoisted.
        {"name": "projection_768", "kind": "projection", "log_n": 16, "tiles_in": 6, "tiles_out": 6, "level": 12, "target": 4},
        # Attention scores times values for four heads with the Gaussian-kernel score: masks, squares, rotate-and-sum,
        # transposes, four encrypted products and two degree-15 polynomials.
        {"name": "attention_4_heads", "kind": "attention", "log_n": 16, "degree": 15},
    ]


def _spread(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))


def draw(rng):
    kind = rng.choice(("ntt", "ntt", "rotate", "rotate", "mult", "client", "encode", "ccmm", "pcmm", "projection", "attention"))
    even = rng.choice((12, 14, 16, 16))   # rings that hold square tiles
    if kind == "ntt":
        return {"kind": kind, "log_n": rng.randint(11, 16), "polys": _spread(rng, 1, 32), "limbs": _spread(rng, 1, 24),
                "bits": rng.choice((42, 60)), "inverse": rng.random() < 0.5}
    if kind in ("rotate", "mult"):
        log_n, bits = rng.choice((12, 13, 14, 15, 16, 16)), rng.choice((42, 60))
        chain, dnum = _spread(rng, 3, 24), rng.choice((2, 3, 3, 4))
        dnum = min(dnum, chain)
        alpha = -(-chain // dnum)
        case = {"kind": kind, "log_n": log_n, "chain": chain, "special": max(1, -(-alpha * bits // 60)), "dnum": dnum, "bits": bits,
                "level": rng.randint(1, chain - 1)}
        return case if kind == "mult" else dict(case, step=_spread(rng, 1, (1 << log_n) // 2 - 1))
    if kind == "client":
        n = 1 << (even - 2) // 2
        return {"kind": kind, "log_n": even, "rows": rng.randint(1, n), "cols": rng.randint(1, n), "pair": rng.random() < 0.5}
    if kind == "encode":
        return {"kind": kind, "log_n": rng.choice((12, 13, 14, 15, 16, 16)), "messages": _spread(rng, 1, 36), "level": rng.randint(1, 12)}
    if kind in ("ccmm", "pcmm"):
        target = rng.randint(3, 5)
        return {"kind": kind, "log_n": even, "pair": rng.random() < 0.5, "level": rng.randint(target + 3, 12), "target": target}
    if kind == "projection":
        target = rng.randint(3, 5)
        return {"kind": kind, "log_n": even, "tiles_in": rng.choice((2, 4, 6)), "tiles_out": rng.choice((2, 4, 6)),
                "level": rng.randint(target + 3, 11), "target": target}
    return {"kind": "attention", "log_n": even, "degree": rng.randint(4, 14)}


# ---- inputs ------------------------------------------------------------------------------------------------------------

def _residues(gen, primes, lead):
    """Uniform residues [lead..][len(primes)][N]: what NTT-form polynomials, ciphertexts and keys hold."""
    n = lead[-1]
    q = torch.tensor(primes, dtype=torch.int64, device="cuda").view(-1, 1)
    return torch.randint(0, 1 << 62, tuple(lead[:-1]) + (len(primes), n), dtype=torch.int64, device="cuda", generator=gen).remainder_(q)


def prepare(case, seed):
    kind, log_n = case["kind"], case["log_n"]
    n_ring = 1 << log_n
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    s = {"kind": kind}
    if kind == "ntt":
        ctx = _context(log_n, case["limbs"], 0, 1, case["bits"])
        s.update(ctx=ctx, data=_residues(gen, ctx.q, (case["polys"], n_ring)), index=list(range(case["limbs"])), inverse=case["inverse"])
    elif kind in ("rotate", "mult"):
        ctx = _context(log_n, case["chain"], case["special"], case["dnum"], case["bits"])
        nq = case["level"] + 1
        s.update(ctx=ctx, nq=nq, key=_residues(gen, ctx.q + ctx.p, (case["dnum"], 2, n_ring)), a=_residues(gen, ctx.q[:nq], (2, n_ring)))
        if kind == "rotate":
            s["galois"] = pow(5, case["step"], 2 * n_ring)
        else:
            s["b"] = _residues(gen, ctx.q[:nq], (2, n_ring))
    elif kind == "encode":
        ctx = _context(log_n, CHAIN, SPECIAL, DNUM, 42)
        z = torch.randn((case["messages"], n_ring // 2, 2), dtype=torch.float64, device="cuda", generator=gen).mul_(0.02)
        s.update(ctx=ctx, slots=torch.view_as_complex(z), nq=case["level"] + 1)
    elif kind == "client":
        shape = (case["rows"], case["cols"])
        s.update(H=_hemmer(log_n), m=[rng.uniform(-1, 1, shape) for _ in range(1 + case["pair"])])
    elif kind in ("ccmm", "pcmm"):
        H = _hemmer(log_n)
        m = [rng.uniform(-1, 1, (H.dim, H.dim)) for _ in range(4)]
        a = H.encrypt2(m[0], m[1]) if case["pair"] else H.encrypt(m[0])
        if kind == "pcmm":
            b = H.encode2(m[2], m[3]) if case["pair"] else H.encode(m[2])
        else:
            b = H.encrypt2(m[2], m[3]) if case["pair"] else H.encrypt(m[2])
        if case["level"] < CHAIN - 1:
            a, b = H.level_down(a, case["level"]), H.level_down(b, case["level"]) if kind == "ccmm" else b
        s.update(H=H, a=a, b=b, pair=case["pair"], target=case["target"])
    elif kind == "projection":
        H, t_in, t_out = _hemmer(log_n), case["tiles_in"], case["tiles_out"]
        n = H.dim
        X, W = 0.1 * rng.normal(size=(n, n * t_in)), 0.02 * rng.normal(size=(n * t_in, n * t_out))
        x = [X[:, i * n:(i + 1) * n] for i in range(t_in)]
        w = lambda i, j: W[i * n:(i + 1) * n, j * n:(j + 1) * n]
        x = [H.complex_packing(H.encrypt2(x[i], x[i]), H.encrypt2(x[i + 1], x[i + 1])) for i in range(0, t_in, 2)]
        s.update(H=H, target=case["target"], x=[H.level_down(c, case["level"]) for c in x] if case["level"] < CHAIN - 1 else x,
                 w=[[H.encode_diagonal_to_row4(w(i, j), w(i, j + 1), w(i + 1, j), w(i + 1, j + 1), level=case["target"] + 1)
                     for i in range(0, t_in, 2)] for j in range(0, t_out, 2)])
    else:
        H = _hemmer(log_n, lowest=0)
        n = H.dim
        # heads of n / 2 columns; squared distances of queries and keys lie around 1.28 whatever the width
        q0, q1, k0, k1, v0, v1 = (0.8 / math.sqrt(n / 2) * rng.normal(size=(n, n)) for _ in range(6))
        cheb = np.polynomial.chebyshev.chebinterpolate(lambda t: np.exp(-(t + 1.5) / 16.0), case["degree"])
        s.update(H=H, table=_package()[1].chebyshev_product_basis(cheb, 4), q=H.encrypt2(q0, q1), k=H.encrypt2(k0, k1),
                 kt=H.encrypt2(k0.T, k1.T), v=H.encrypt2(v0, v1))
    return s


# ---- one pass ----------------------------------------------------------------------------------------------------------

def run(s):
    kind = s["kind"]
    if kind == "ntt":
        return s["ctx"].ntt(s["data"], s["index"], inverse=s["inverse"])
    if kind == "rotate":
        return s["ctx"].rotate(s["a"], s["key"], s["galois"], s["nq"])
    if kind == "mult":
        ctx, nq = s["ctx"], s["nq"]
        return ctx.rescale(ctx.relinearize(ctx.tensor(s["a"], s["b"], nq), s["key"], nq), nq)
    if kind == "encode":
        return s["ctx"].encode(s["slots"], float(1 << LOG_SCALE), s["nq"])
    H = s["H"]
    if kind == "client":
        m = s["m"]
        return H.decrypt2(H.encrypt2(m[0], m[1])) if len(m) == 2 else H.decrypt(H.encrypt(m[0]))
    if kind in ("ccmm", "pcmm"):
        c = (H.single_cc_matmul if kind == "ccmm" else H.single_matmul)(s["a"], s["b"], s["target"])
        return H.decrypt2(c) if s["pair"] else H.decrypt(c)
    if kind == "projection":
        pre = [H.matmul_pre(x, s["target"]) for x in s["x"]]
        out = []
        for column in s["w"]:
            acc = None
            for p, w in zip(pre, column):
                y = H.matmul_reuse(p, w, s["target"])
                acc = y if acc is None else H.add(acc, y)
            out.append(H.repack_cc(acc))
        return [H.decrypt2(y) for y in out]
    # attention: heads split by masks, |q|^2 and |k|^2 as row norms (the key norms transposed), the score
    # exp(-|q - k|^2 / 16) as a polynomial of -2 q k^T + |q|^2 + |k|^2, times the values
    score, last = 8, 1
    mq, mk, mv = H.mask_right_left(s["q"]), H.mask_right_left(s["k"]), H.mask_right_left(s["v"])
    sq, sk = [H.mult(x, x) for x in mq], [H.mult(x, x) for x in mk]
    H.one_mat_rot_sum_inplace(sq[0], sq[1])
    H.one_mat_rot_sum_inplace(sk[0], sk[1])
    out = []
    for j in (0, 1):
        H.transpose_inplace(sk[j], score)
        d = H.single_cc_matmul(mq[j], s["kt"], score)
        x = H.add(H.add(H.mult_const(d, -2.0), H.level_down(sq[j], score)), sk[j])
        p = H.eval_chebyshev(H.linear_transform(x, 0.5, 2.5), s["table"], 4)
        out.append(H.single_cc_matmul(p, mv[j], last))
    return [H.decrypt2(c) for c in out]


# ---- what a pass cannot do without -------------------------------------------------------------------------------------

def _key_words(case, nq):
    """Words of one evaluation key that a key switch of nq limbs reads."""
    chain, special, dnum = case.get("chain", CHAIN), case.get("special", SPECIAL), case.get("dnum", DNUM)
    alpha = -(-chain // dnum)
    return 2 * -(-nq // alpha) * (nq + special) << case["log_n"]


def work(case):
    """Bytes: operands read once, results written once, each key that the method needs read once.  Operations: a modular
    multiplication and an addition for each butterfly and each residue of a key, floating ones where the path has them."""
    kind, log_n = case["kind"], case["log_n"]
    n_ring = 1 << log_n
    n = 1 << max(0, (log_n - 2) // 2)

    def products(count, level):   # `count` products of n x n tiles: n / 2 shifts of two columns, each a key of its own
        keys = count * (n // 2) * _key_words(case, level + 3)
        return {"bytes": 8 * (keys + 2 * count * 2 * (level + 3) * n_ring), "flops": 2 * keys}

    if kind == "ntt":
        words = case["polys"] * case["limbs"] * n_ring
        return {"bytes": 16 * words, "flops": 3 * words * log_n / 2}
    if kind == "rotate":
        nq = case["level"] + 1
        key = _key_words(case, nq)
        return {"bytes": 8 * (key + 4 * nq * n_ring), "flops": 2 * key}
    if kind == "mult":
        nq = case["level"] + 1
        key = _key_words(case, nq)
        return {"bytes": 8 * (key + (4 * nq + 2 * (nq - 1)) * n_ring), "flops": 2 * key}
    if kind == "encode":
        return {"bytes": case["messages"] * (8 * n_ring + 8 * (case["level"] + 1) * n_ring),
                "flops": case["messages"] * (5 * n_ring // 2 * (log_n - 1) + 1.5 * (case["level"] + 1) * n_ring * log_n)}
    if kind == "client":   # the ciphertext is written once; two of its limbs are read back
        return {"bytes": 16 * case["rows"] * case["cols"] * (1 + case["pair"]) + 8 * (2 * CHAIN + 4) * n_ring,
                "flops": 1.5 * (CHAIN + 4) * n_ring * log_n}
    if kind == "ccmm":
        return products(1, case["target"])
    if kind == "pcmm":
        return products(1, case["target"])
    if kind == "projection":
        t, cols = case["tiles_in"] // 2, case["tiles_out"] // 2
        shifts = n * 2 * (case["target"] + 2) * n_ring   # the shifted activations, read once per group of weight tiles
        w = products(t, case["target"])
        return {"bytes": w["bytes"] + 8 * t * cols * shifts, "flops": w["flops"] + 2 * t * cols * shifts}
    a, b = products(2, 8), products(2, 1)
    return {k: a[k] + b[k] for k in a}


def tolerance(case):
    """Residues are whole numbers: exact.  Decrypted matrices carry the scheme's noise, which encryption draws anew each time:
    1e-8 to 1e-7 of the entries at scale 2^42, ten times that with other roundings on the way."""
    if case["kind"] in ("ntt", "rotate", "mult", "encode"):
        return "exact"
    return {"rel": 1e-6, "max": 1e-5}
