"""Performance cases of the BFV engine, through the Python host binding.

Every case is one call (or the short call sequence) that a program makes on a
context it keeps: HomMult + relinearisation, RGSW x RLWE external product, the
batched NTT in both directions, slot rotation, and the client's round trip
(encode, encrypt, decrypt, decode).  Ring sizes and modulus chains are the
engine's own: the default sets at N = 2^12, 2^14 and 2^15, and the 60-bit
chains with one special prime and four auxiliary primes at N = 2^13..2^16.
Plans are the context's built-in ones.

All outputs are residues (whole numbers).
"""
import math

import numpy as np
import torch

import kunpbfv_amd as kb

PLAIN = 65537
AUX_PRIMES = 4
GADGET_BITS = 20
# largest number of 60-bit ciphertext primes at each ring size (the serving
# loop's and the benchmark's chains)
MAX_Q = {13: 2, 14: 6, 15: 13, 16: 28}
# limbs x coefficients x ciphertexts of the largest listed batch
MAX_WORDS = 128 * 28 << 16


def listed():
    return [
        # a single small product: the latency of one call, every launch counts
        dict(name="mult_n4096_q2_b1", op="mult", chain="default", log_n=12, q=2, batch=1),
        # what a continuous-batching server takes from its queue at once
        dict(name="mult_n8192_q2_b9", op="mult", chain="60bit", log_n=13, q=2, batch=9),
        # two special primes (K = 2), an odd batch too small for the batched inner product
        dict(name="mult_n16384_k2_b5", op="mult", chain="default", log_n=14, q=4, batch=5),
        # a mid-size ring with a full batch
        dict(name="mult_n32768_q13_b64", op="mult", chain="60bit", log_n=15, q=13, batch=64),
        # the deep ring, one product at a time
        dict(name="mult_n65536_q28_b1", op="mult", chain="60bit", log_n=16, q=28, batch=1),
        # the deep ring, batched: the benchmark's workload
        dict(name="mult_n65536_q28_b128", op="mult", chain="60bit", log_n=16, q=28, batch=128),
        # a few external products of a small ring, as a server's queue gives them
        dict(name="ext_n8192_q2_b3", op="ext", chain="60bit", log_n=13, q=2, batch=3),
        # one RGSW ciphertext applied to a whole batch of the deep ring
        dict(name="ext_n65536_q28_b128", op="ext", chain="60bit", log_n=16, q=28, batch=128),
        # transforms alone, forward: many polynomials of a short chain
        dict(name="ntt_fwd_n16384_l8_b256", op="ntt", chain="60bit", log_n=14, q=8, batch=256, direction=1, basis="q"),
        # transforms alone, inverse, over the extended basis of a few tensor products
        dict(name="ntt_inv_n65536_l57_b12", op="ntt", chain="60bit", log_n=16, q=28, batch=12, direction=-1,
             basis="qr"),
        # slot rotation of an odd batch
        dict(name="rotate_n32768_q15_b7", op="rotate", chain="default", log_n=15, q=15, batch=7),
        # the client's side: encode, encrypt, decrypt, decode
        dict(name="client_n16384_q6_b24", op="client", chain="60bit", log_n=14, q=6, batch=24),
    ]


def draw(rng):
    op = rng.choice(["mult", "mult", "mult", "ext", "ext", "ntt", "ntt", "rotate", "client"])
    if op in ("mult", "rotate", "client") and rng.random() < 0.25:
        chain, log_n, q = "default", *rng.choice([(12, 2), (14, 4), (15, 15)])
    else:
        chain, log_n = "60bit", rng.randint(13, 16)
        q = rng.randint(2, 8 if op == "ntt" and log_n < 15 else MAX_Q[log_n])
    # an external product decomposes every limb over every limb: its work grows
    # with the square of the chain
    words = q << log_n
    most = MAX_WORDS // words
    if op == "ext":
        most = most * 28 // max(28, q)
    most = max(1, min(most, 256 if op == "ntt" else 128))
    case = dict(op=op, chain=chain, log_n=log_n, q=q, batch=int(round(math.exp(rng.uniform(0, math.log(most))))))
    if op == "ntt":
        case["direction"] = rng.choice([1, -1])
        case["basis"] = rng.choice(["q", "qr"])
        case["batch"] = max(1, case["batch"] // (2 if case["basis"] == "qr" else 1))
    return case


_contexts = {}  # the one parameter set in use, as a program keeps it


def context(case):
    key = (case["chain"], case["log_n"], case["q"])
    if key not in _contexts:
        _contexts.clear()
        torch.cuda.empty_cache()
        if case["chain"] == "default":
            _contexts[key] = kb.Context.default(case["log_n"])
        else:
            _contexts[key] = kb.Context.chain60(case["log_n"], case["q"], 1, AUX_PRIMES, 2, PLAIN)
        assert _contexts[key].qn == case["q"]
    return _contexts[key]


def _basis(ctx, case):
    """(first modulus, limbs) of a transform case"""
    return (ctx.oQ, ctx.qn + ctx.rn) if case["basis"] == "qr" else (ctx.oQ, ctx.qn)


def prepare(case, seed):
    ctx = context(case)
    op, batch = case["op"], case["batch"]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    state = dict(case=case, ctx=ctx)
    if op == "ntt":
        mod0, limbs = _basis(ctx, case)
        src = ctx.empty(batch, limbs, ctx.n)
        for l in range(limbs):
            src[:, l] = torch.randint(int(ctx.mod[mod0 + l]), (batch, ctx.n), dtype=torch.int64, device="cuda",
                                      generator=gen)
        state.update(src=src, dst=torch.empty_like(src))
        return state

    def key_seed(tag):
        return int(seed).to_bytes(8, "little") + bytes([tag]) + bytes(23)

    def messages():
        return torch.randint(ctx.plain, (batch, ctx.n), dtype=torch.int64, device="cuda", generator=gen)

    sk = ctx.keygen_sk(key_seed(1))
    pk = ctx.keygen_pk(key_seed(2), sk)
    if op == "client":
        state.update(sk=sk, pk=pk, slots=messages(), seed=key_seed(3))
        return state
    state["c1"] = ctx.encrypt(key_seed(4), pk, ctx.encode(messages()))
    if op == "mult":
        state["c2"] = ctx.encrypt(key_seed(5), pk, ctx.encode(messages()))
        state["rlk"] = ctx.keygen_rlk(key_seed(6), sk)
    elif op == "rotate":
        state["g"] = ctx.galois_elt(1 + seed % 7)
        state["gkey"] = ctx.keygen_galois(key_seed(7), sk, state["g"])
    else:
        m = np.zeros(ctx.n, dtype=np.uint64)
        m[1 + seed % 7] = 1  # a monomial: the product is a shift of the slots' polynomial
        state["rgsw"] = ctx.rgsw_encrypt(key_seed(8), sk, kb.to_device(m), GADGET_BITS)
    return state


def run(state):
    case, ctx = state["case"], state["ctx"]
    op = case["op"]
    if op == "mult":
        return ctx.mult_relin(state["rlk"], state["c1"], state["c2"])
    if op == "ext":
        return ctx.external_product(state["rgsw"], state["c1"], GADGET_BITS)
    if op == "rotate":
        return ctx.rotate(state["gkey"], state["g"], state["c1"])
    if op == "ntt":
        mod0, limbs = _basis(ctx, case)
        return ctx.ntt(state["src"], state["dst"], case["direction"], mod0, limbs, polys=case["batch"])
    pt = ctx.encode(state["slots"].clone())
    ct = ctx.encrypt(state["seed"], state["pk"], pt)
    return {"ciphertexts": ct, "slots": ctx.decode(ctx.decrypt(state["sk"], ct))}


def _shape(case):
    """(special primes, auxiliary primes, digits, key blocks, extension primes) of a case's chain"""
    log_n, q = case["log_n"], case["q"]
    p, t, gamma = 1, AUX_PRIMES, 2
    if case["chain"] == "default":
        d = kb.default_params(log_n)
        p, t, gamma = len(d["p"]), len(d["t"]), d["gamma"]
    return p, t, -(-q // p), -(-(p + q) // gamma), q + 1


def work(case):
    n, q, b, op = 1 << case["log_n"], case["q"], case["batch"], case["op"]
    p, t, digits, blocks, r = _shape(case)
    ct = 2 * q * n * 8
    key = 2 * digits * blocks * t * n * 8
    butterflies = n * case["log_n"] // 2  # of one limb's transform
    # modular multiplications: transforms, then the products between them
    if op == "ntt":
        limbs = q if case["basis"] == "q" else q + r
        return {"bytes": 2 * limbs * n * 8 * b, "flops": 2 * limbs * butterflies * b}
    switch = digits * t + 2 * blocks * t + 2 * q  # limb transforms of a key switch
    inner = 2 * digits * blocks * t * n
    if op == "rotate":
        return {"bytes": 2 * b * ct + key, "flops": 2 * b * ((switch + 2 * q) * butterflies + inner)}
    if op == "mult":
        limbs = 4 * q + 4 * r + 3 * (q + r) + switch
        mults = 4 * q * r + 4 * (q + r) + 3 * (q + 1) * r + 3 * r * q
        return {"bytes": 3 * b * ct + key, "flops": 2 * b * (limbs * butterflies + mults * n + inner)}
    if op == "ext":
        rows = 2 * q * -(-60 // GADGET_BITS)
        # digits against every limb, or against two auxiliary primes: the smaller count
        return {"bytes": 2 * b * ct + rows * ct,
                "flops": 2 * b * ((2 * rows + 8 * q) * butterflies + 2 * rows * q * n)}
    # client: the messages in and out, the keys read, the ciphertexts written and read back
    return {"bytes": 2 * b * n * 8 + 3 * q * n * 8 + 2 * b * ct, "flops": 2 * b * (4 * q + 2) * butterflies}


def exact(case, seed):
    """The outputs are whole numbers: they have no rounding to be measured."""
    return None
