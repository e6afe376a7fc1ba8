"""The work this library does for its users, as timed cases.

Each case is one call (or one burst of calls) through the public entry points
of ``tmvp_amd`` (the C ABI of ``include/tmvp.h``): the products behind Saber and
Sable at the batch sizes of a key-encapsulation service, mixed work lists, the
batched KEM in its three directions, the reference-named host functions and the
serving loop.  Device data are torch tensors on the GPU; the host functions and
the serving loop take host arrays, as their users do.

``listed()`` gives the fixed cases, ``draw(rng)`` one more from the same ranges,
``prepare`` what a program holds before the call, ``run`` the call,
``work`` the bytes and operations it cannot do without, and ``exact`` the product
cases' results from a 64-bit convolution.  All outputs are whole numbers or bytes.
"""
import math
import os
import random
import sys

import numpy as np
import torch

# torch brings its own HIP runtime; the library's front end must use that one
# and not load a second runtime into the process.
_bundled = os.path.join(os.path.dirname(torch.__file__), "lib", "libamdhip64.so")
if os.path.exists(_bundled):
    os.environ.setdefault("TMVP_HIP_RUNTIME", _bundled)
sys.path.insert(0, os.path.join(os.getcwd(), "asfand-tmvp_amd"))

import tmvp_amd as T  # noqa: E402

N = 256
SETS = ("lightsaber", "saber", "firesaber", "sable1", "sable2", "sable3")
_context = None


def context():
    """The process's one context, as a program keeps it."""
    global _context
    if _context is None:
        _context = T.Context(torch.cuda.current_device())
    return _context


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # One encryption's two products (A s, then b . s with the message): an interactive handshake, where launch and
        # latency are all there is.
        {"name": "encrypt_products_saber_1", "op": "encrypt", "set": "saber", "batch": 1},
        # A s of an encapsulation service at full load, rounded to p.
        {"name": "matvec_saber_65536", "op": "matvec", "set": "saber", "batch": 65536, "transpose": False, "round": True},
        # Key generation's product (A^T s) for a ragged batch of the largest set.
        {"name": "matvec_t_firesaber_5003", "op": "matvec", "set": "firesaber", "batch": 5003, "transpose": True,
         "round": True},
        # Raw negacyclic products, the unit everything else is made of.
        {"name": "polymul_65536", "op": "polymul", "eq_bits": 13, "batch": 65536},
        # A gateway's mixed list: every Saber set's matrix-vector and inner product in one launch.
        {"name": "mixed_saber_4096", "op": "mixed", "sets": "lightsaber,saber,firesaber", "batches": "4096,4096,4096"},
        # One decapsulation: a single client's handshake.
        {"name": "kem_decaps_saber_1", "op": "decaps", "set": "saber", "batch": 1},
        # The three KEM directions at a service's batch size.
        {"name": "kem_keypair_saber_16384", "op": "keypair", "set": "saber", "batch": 16384},
        {"name": "kem_encaps_saber_16384", "op": "encaps", "set": "saber", "batch": 16384},
        {"name": "kem_decaps_saber_16384", "op": "decaps", "set": "saber", "batch": 16384},
        # A bulk job: rekeying a fleet with the largest set, a ragged batch.
        {"name": "kem_encaps_firesaber_49999", "op": "encaps", "set": "firesaber", "batch": 49999},
        # The drop-in host function over host buffers at the batch it replaces.
        {"name": "host_sable_enc_512", "op": "host_enc", "set": "sable2", "batch": 512},
        # A burst of requests to the serving loop: both schemes, both operations, sizes up to 4096.
        {"name": "serve_burst_24", "op": "serve", "requests": 24, "most": 4096, "keys": 4096},
    ]


def _spread(rng, lo, hi):
    """A whole number of [lo, hi], even over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(("matvec", "matvec", "innerprod", "encrypt", "polymul", "mixed", "kem", "kem", "kem", "kem", "host", "serve"))
    if kind == "matvec":
        return {"op": "matvec", "set": rng.choice(SETS), "batch": _spread(rng, 1, 65536),
                "transpose": rng.random() < 0.5, "round": rng.random() < 0.8}
    if kind == "innerprod":
        return {"op": "innerprod", "set": rng.choice(SETS), "batch": _spread(rng, 1, 65536),
                "epilogue": rng.choice((T.IP_RAW, T.IP_ENC, T.IP_DEC))}
    if kind == "encrypt":
        return {"op": "encrypt", "set": rng.choice(SETS), "batch": _spread(rng, 1, 32768)}
    if kind == "polymul":
        return {"op": "polymul", "eq_bits": rng.choice((9, 10, 11, 13)), "batch": _spread(rng, 1, 65536)}
    if kind == "mixed":
        sets = [rng.choice(SETS) for _ in range(rng.randint(2, 5))]
        return {"op": "mixed", "sets": ",".join(sets), "batches": ",".join(str(_spread(rng, 16, 8192)) for _ in sets)}
    if kind == "kem":
        return {"op": rng.choice(("keypair", "encaps", "decaps")), "set": rng.choice(SETS),
                "batch": _spread(rng, 1, 40000)}
    if kind == "host":
        ps = rng.choice(SETS)
        return {"op": rng.choice(("host_enc", "host_dec")), "set": ps, "batch": _spread(rng, 1, 2048)}
    return {"op": "serve", "requests": rng.randint(4, 24), "most": _spread(rng, 64, 4096), "keys": _spread(rng, 256, 4096)}


# ---------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) & 0x7FFFFFFFFFFFFFFF)
    return g


def _uniform(g, shape, bits):
    return torch.randint(0, 1 << bits, shape, generator=g, device="cuda", dtype=torch.int16)


def _bytes(g, shape):
    return torch.randint(0, 256, shape, generator=g, device="cuda", dtype=torch.uint8)


def _secret(g, shape, mu, mask=None):
    """Centred-binomial secrets: two's complement, or masked mod q (Sable)."""
    bits = torch.zeros(shape, device="cuda", dtype=torch.int16)
    for _ in range(mu // 2):
        bits += torch.randint(0, 2, shape, generator=g, device="cuda", dtype=torch.int16)
        bits -= torch.randint(0, 2, shape, generator=g, device="cuda", dtype=torch.int16)
    return bits if mask is None else torch.bitwise_and(bits, mask)


def _set_secret(g, shape, p):
    return _secret(g, shape, p["mu"], (1 << p["eq"]) - 1 if p["sable"] else None)


def _empty16(*shape):
    return torch.empty(shape, device="cuda", dtype=torch.int16)


def _empty8(*shape):
    return torch.empty(shape, device="cuda", dtype=torch.uint8)


def _keys(ps, batch, g):
    p = T.get_params(ps)
    seeds = _bytes(g, (batch, 96))
    pk, sk = _empty8(batch, p["pk_bytes"]), _empty8(batch, p["sk_bytes"])
    context().kem_keypair(pk.data_ptr(), sk.data_ptr(), seeds.data_ptr(), batch, ps)
    torch.cuda.synchronize()
    return pk, sk


def _ciphertexts(ps, batch, pk, g):
    p = T.get_params(ps)
    rnd = _bytes(g, (batch, 32))
    ct, ss = _empty8(batch, p["ct_bytes"]), _empty8(batch, 32)
    context().kem_encaps(ct.data_ptr(), ss.data_ptr(), pk.data_ptr(), rnd.data_ptr(), batch, ps)
    torch.cuda.synchronize()
    return ct


def _mixed(case):
    return list(zip(case["sets"].split(","), (int(b) for b in case["batches"].split(","))))


def _product_inputs(case, seed):
    """The tensors of a product case, from the seed alone (exact() makes them again)."""
    g = _gen(seed)
    if case["op"] == "polymul":
        b = case["batch"]
        return {"a": _uniform(g, (b, N), case["eq_bits"]), "s": _secret(g, (b, N), 8)}
    p = T.get_params(case["set"])
    b, l = case["batch"], p["l"]
    if case["op"] == "matvec":
        return {"a": _uniform(g, (b, l, l, N), p["eq"]), "s": _set_secret(g, (b, l, N), p)}
    if case["op"] == "encrypt":
        return {"a": _uniform(g, (b, l, l, N), p["eq"]), "b": _uniform(g, (b, l, N), p["ep"]),
                "s": _set_secret(g, (b, l, N), p), "aux": _uniform(g, (b, N), 1)}
    d = {"a": _uniform(g, (b, l, N), p["ep"]), "s": _set_secret(g, (b, l, N), p), "aux": None}
    if case["epilogue"] == T.IP_ENC:
        d["aux"] = _uniform(g, (b, N), 1)
    elif case["epilogue"] == T.IP_DEC:
        d["aux"] = _uniform(g, (b, N), p["et"])
    return d


def _mixed_inputs(case, seed):
    g = _gen(seed)
    jobs = []
    for ps, b in _mixed(case):
        p = T.get_params(ps)
        l = p["l"]
        jobs.append({"set": ps, "batch": b, "A": _uniform(g, (b, l, l, N), p["eq"]), "b": _uniform(g, (b, l, N), p["ep"]),
                     "s": _set_secret(g, (b, l, N), p)})
    return jobs


class Burst:
    """A server over resident keys and the requests of one burst, in pinned memory."""

    def __init__(self, case, seed):
        rng = random.Random(1000 * case["requests"] + case["most"])  # request sizes belong to the case
        g = _gen(seed)
        n = case["keys"]
        self.server = T.Server(context())
        pks = {}
        for ps in ("saber", "sable2"):
            pk, sk = _keys(ps, n, g)
            first = self.server.add_keys(ps, pk.cpu().numpy(), sk.cpu().numpy())
            pks[ps] = (pk, first)
        self.requests = []
        for i in range(case["requests"]):
            ps, op = ("saber", "sable2")[i % 2], (T.SRV_ENCAPS, T.SRV_DECAPS)[(i // 2) % 2]
            p = T.get_params(ps)
            count = rng.randint(1, case["most"])
            ids = torch.randint(0, n, (count,), generator=g, device="cuda", dtype=torch.int64)
            pk, first = pks[ps]
            data = _bytes(g, (count, 32)) if op == T.SRV_ENCAPS else _ciphertexts(ps, count, pk[ids].contiguous(), g)
            held = T.pinned_array(tuple(data.shape))
            held[...] = data.cpu().numpy()
            out = ((T.pinned_array((count, p["ct_bytes"])), T.pinned_array((count, 32))) if op == T.SRV_ENCAPS
                   else (T.pinned_array((count, 32)), T.pinned_array((count,))))
            self.requests.append((op, ps, (ids + first).to(torch.int32).cpu().numpy(), held, out))

    def run(self):
        for i, (op, ps, keys, data, out) in enumerate(self.requests):
            self.server.submit(op, ps, keys, data, tag=i, out=out)
        left = len(self.requests)
        while left:
            for c in self.server.poll(timeout_us=100000):
                if c["status"] != T.OK:
                    raise T.TmvpError(c["status"], "serving")
                left -= 1
        return [out for _, _, _, _, out in self.requests]

    def __del__(self):
        try:
            self.server.close()
        except Exception:
            pass


# ---------------------------------------------------------------- the calls

def prepare(case, seed):
    op = case["op"]
    ctx = context()
    if op in ("matvec", "innerprod", "encrypt", "polymul"):
        d = _product_inputs(case, seed)
        shape = tuple(d["a"].shape)
        if op == "encrypt":
            return {"case": case, "ctx": ctx, "bp": _empty16(shape[0], shape[1], N), "v": _empty16(shape[0], N), **d}
        if op == "matvec":
            out = _empty16(shape[0], shape[1], N)
        else:
            out = _empty16(shape[0], N)
        return {"case": case, "ctx": ctx, "out": out, **d}
    if op == "mixed":
        jobs = _mixed_inputs(case, seed)
        descs, outs = [], []
        for j in jobs:
            p = T.get_params(j["set"])
            bp, v = _empty16(j["batch"], p["l"], N), _empty16(j["batch"], N)
            descs.append(T.work(T.OP_MATVEC, bp.data_ptr(), j["A"].data_ptr(), j["s"].data_ptr(), j["batch"], j["set"],
                                epilogue=1))
            descs.append(T.work(T.OP_INNERPROD, v.data_ptr(), j["b"].data_ptr(), j["s"].data_ptr(), j["batch"], j["set"],
                                epilogue=T.IP_RAW))
            outs += [bp, v]
        return {"case": case, "ctx": ctx, "jobs": jobs, "descs": descs, "outs": outs}
    if op == "serve":
        return {"case": case, "burst": Burst(case, seed)}
    ps, b = case["set"], case["batch"]
    p = T.get_params(ps)
    g = _gen(seed)
    st = {"case": case, "ctx": ctx}
    if op == "keypair":
        st.update(seeds=_bytes(g, (b, 96)), pk=_empty8(b, p["pk_bytes"]), sk=_empty8(b, p["sk_bytes"]))
        return st
    pk, sk = _keys(ps, b, g)
    if op == "encaps":
        st.update(pk=pk, rnd=_bytes(g, (b, 32)), ct=_empty8(b, p["ct_bytes"]), ss=_empty8(b, 32))
    elif op == "decaps":
        st.update(sk=sk, ct=_ciphertexts(ps, b, pk, g), ss=_empty8(b, 32), fail=_empty8(b))
    elif op == "host_enc":
        st.update(pk=pk.cpu().numpy(), rnd=_bytes(g, (b, 32)).cpu().numpy(), ct=np.zeros((b, p["ct_bytes"]), np.uint8),
                  ss=np.zeros((b, 32), np.uint8))
    else:
        st.update(pk=pk.cpu().numpy(), sk=sk.cpu().numpy(), ct=_ciphertexts(ps, b, pk, g).cpu().numpy(),
                  ss=np.zeros((b, 32), np.uint8))
    return st


def _host_call(st):
    lib = T.load_library()
    case = st["case"]
    ps, b = T.PARAM_SET_NAMES[case["set"]], case["batch"]
    sable = case["set"].startswith("sable")
    rc = lib.tmvp_host_configure(0, 1 if sable else b, T.SABER if sable else ps, b if sable else 1, ps if sable else T.SABLE2)
    if rc:
        raise T.TmvpError(rc, "tmvp_host_configure")
    at = {k: st[k].ctypes.data for k in ("pk", "sk", "ct", "ss") if k in st}
    if case["op"] == "host_enc":
        lib.tmvp_host_set_randomness(st["rnd"].ctypes.data, b)
        if sable:
            lib.SABLE_enc(at["ss"], at["pk"], at["ct"], 0)
        else:
            lib.saber_enc(0, at["ss"], at["pk"], at["ct"])
        outs = (st["ct"], st["ss"])
    else:
        if sable:
            lib.SABLE_dec(at["ct"], at["pk"], at["sk"], at["ss"], 0)
        else:
            lib.saber_dec(0, at["ct"], at["pk"], at["sk"], at["ss"])
        outs = (st["ss"],)
    rc = lib.tmvp_host_status()
    if rc:
        raise T.TmvpError(rc, case["op"])
    return outs


def run(state):
    case = state.get("case")
    op = case["op"]
    if op == "matvec":
        state["ctx"].matvec(state["out"].data_ptr(), state["a"].data_ptr(), state["s"].data_ptr(), case["batch"],
                            case["set"], transpose=case["transpose"], round_to_p=case["round"])
        return state["out"]
    if op == "polymul":
        state["ctx"].polymul(state["out"].data_ptr(), state["a"].data_ptr(), state["s"].data_ptr(), case["batch"],
                             case["eq_bits"])
        return state["out"]
    if op == "innerprod":
        aux = state["aux"]
        state["ctx"].innerprod(state["out"].data_ptr(), state["a"].data_ptr(), state["s"].data_ptr(), case["batch"],
                               case["set"], epilogue=case["epilogue"], aux=None if aux is None else aux.data_ptr())
        return state["out"]
    if op == "encrypt":
        state["ctx"].matvec(state["bp"].data_ptr(), state["a"].data_ptr(), state["s"].data_ptr(), case["batch"],
                            case["set"], round_to_p=True)
        state["ctx"].innerprod(state["v"].data_ptr(), state["b"].data_ptr(), state["s"].data_ptr(), case["batch"],
                               case["set"], epilogue=T.IP_ENC, aux=state["aux"].data_ptr())
        return state["bp"], state["v"]
    if op == "mixed":
        state["ctx"].batch_launch(state["descs"])
        return state["outs"]
    if op == "keypair":
        state["ctx"].kem_keypair(state["pk"].data_ptr(), state["sk"].data_ptr(), state["seeds"].data_ptr(),
                                 case["batch"], case["set"])
        return state["pk"], state["sk"]
    if op == "encaps":
        state["ctx"].kem_encaps(state["ct"].data_ptr(), state["ss"].data_ptr(), state["pk"].data_ptr(),
                                state["rnd"].data_ptr(), case["batch"], case["set"])
        return state["ct"], state["ss"]
    if op == "decaps":
        state["ctx"].kem_decaps(state["ss"].data_ptr(), state["ct"].data_ptr(), state["sk"].data_ptr(), case["batch"],
                                case["set"], fail=state["fail"].data_ptr())
        return state["ss"], state["fail"]
    if op == "serve":
        return state["burst"].run()
    return _host_call(state)


# ---------------------------------------------------------------- what a call cannot do without

# 32-bit logical operations of one Keccak-f[1600]: 24 rounds of theta (55
# 64-bit operations), rho (24), chi (75) and iota (1), two 32-bit halves each.
_KECCAK_OPS = 24 * 155 * 2


def _sponge(nbytes, rate):
    return nbytes // rate + 1


def _kem_work(op, ps, b):
    p = T.get_params(ps)
    l = p["l"]
    matrix = -(-(l * l * p["eq"] * 32) // 168)
    secret = -(-(l * p["mu"] * 32) // 168)
    hpk, hct = _sponge(p["pk_bytes"], 136), _sponge(p["ct_bytes"], 136)
    if op == "keypair":
        perms, prods, nbytes = 1 + matrix + secret + hpk, l * l, 96 + p["pk_bytes"] + p["sk_bytes"]
    elif op == "encaps":
        perms, prods = matrix + 1 + hpk + 1 + secret + hct + 1, l * l + l
        nbytes = p["pk_bytes"] + 32 + p["ct_bytes"] + 32
    else:
        perms, prods = matrix + hct + 1 + secret + 1, l * l + 2 * l
        nbytes = p["sk_bytes"] + p["ct_bytes"] + 32 + 1
    return {"bytes": b * nbytes, "flops": b * (perms * _KECCAK_OPS + prods * 2 * N * N)}


def work(case):
    op = case["op"]
    if op == "polymul":
        return {"bytes": case["batch"] * 3 * N * 2, "flops": case["batch"] * 2 * N * N}
    if op in ("matvec", "innerprod"):
        l = T.get_params(case["set"])["l"]
        if op == "matvec":
            polys, prods = l * l + 2 * l, l * l
        else:
            polys, prods = 2 * l + 1 + (case["epilogue"] != T.IP_RAW), l
        return {"bytes": case["batch"] * polys * N * 2, "flops": case["batch"] * prods * 2 * N * N}
    if op == "encrypt":
        l = T.get_params(case["set"])["l"]
        return {"bytes": case["batch"] * (l * l + 3 * l + 2) * N * 2, "flops": case["batch"] * (l * l + l) * 2 * N * N}
    if op == "mixed":
        got = {"bytes": 0, "flops": 0}
        for ps, b in _mixed(case):
            l = T.get_params(ps)["l"]
            # both products of a set read the same secret
            got["bytes"] += b * (l * l + 3 * l + 1) * N * 2
            got["flops"] += b * (l * l + l) * 2 * N * N
        return got
    if op in ("keypair", "encaps", "decaps"):
        return _kem_work(op, case["set"], case["batch"])
    if op in ("host_enc", "host_dec"):
        return _kem_work("encaps" if op == "host_enc" else "decaps", case["set"], case["batch"])
    # Serving: the mean request of the burst, without the resident matrix's
    # sponge and the public key's hash.
    got = {"bytes": 0, "flops": 0}
    for i in range(case["requests"]):
        ps, enc = ("saber", "sable2")[i % 2], (i // 2) % 2 == 0
        p = T.get_params(ps)
        l, b = p["l"], (case["most"] + 1) / 2
        secret, hct = -(-(l * p["mu"] * 32) // 168), _sponge(p["ct_bytes"], 136)
        perms = (3 if enc else 2) + secret + hct
        prods = l * l + (l if enc else 2 * l)
        got["bytes"] += b * (l * l * N * 2 + p["ct_bytes"] + (p["pk_bytes"] if enc else p["sk_bytes"]) + 64)
        got["flops"] += b * (perms * _KECCAK_OPS + prods * 2 * N * N)
    return got


# ---------------------------------------------------------------- 64-bit results

def _negacyclic(a, s, l, pairs):
    """sum over the (i, j) pairs of a[:, i] * s[:, j] mod x^256 + 1, exact: a twisted FFT in complex128
    (sums stay under 2^26) rounded to int64."""
    k = torch.arange(N, device="cuda", dtype=torch.float64) * (math.pi / N)
    twist = torch.polar(torch.ones_like(k), k)
    fa = torch.fft.fft(a.double() * twist)
    fs = torch.fft.fft(s.double() * twist)
    tot = sum(fa[:, i] * fs[:, j] for i, j in pairs)
    return torch.round((torch.fft.ifft(tot) * twist.conj()).real).to(torch.int64)


def _centred(s, p):
    s = s.to(torch.int64)
    if p is not None and p["sable"]:
        q = 1 << p["eq"]
        s = torch.where(s >= q // 2, s - q, s)
    return s


def _chunked(f, n, *ts):
    return torch.cat([f(*(t[i:i + 4096] if t is not None else None for t in ts)) for i in range(0, n, 4096)])


def _exact_matvec(A, s, p, transpose, rounded):
    l, q = p["l"], 1 << p["eq"]

    def part(A, s):
        A, s = A.reshape(-1, l * l, N), _centred(s, p)
        rows = [_negacyclic(A, s, l, [((j * l + i) if transpose else (i * l + j), j) for j in range(l)]) for i in range(l)]
        x = torch.stack(rows, 1)
        x = ((x + p["h1"]) % q) >> (p["eq"] - p["ep"]) if rounded else x % q
        return x.to(torch.int16)

    return _chunked(part, A.shape[0], A, s)


def _exact_inner(b, s, aux, p, epilogue):
    def part(b, s, aux):
        v = _negacyclic(b, _centred(s, p), p["l"], [(j, j) for j in range(p["l"])])
        q = 1 << p["ep"]
        if epilogue == T.IP_ENC:
            v = ((v + p["h1"] - (aux.to(torch.int64) << (p["ep"] - 1))) % q) >> (p["ep"] - p["et"])
        elif epilogue == T.IP_DEC:
            v = ((v + p["h2"] - (aux.to(torch.int64) << (p["ep"] - p["et"]))) % q) >> (p["ep"] - 1)
        else:
            v = v % q
        return v.to(torch.int16)

    return _chunked(part, b.shape[0], b, s, aux)


def exact(case, seed):
    op = case["op"]
    if op == "polymul":
        d = _product_inputs(case, seed)
        q = 1 << case["eq_bits"]
        return _chunked(lambda a, s: (_negacyclic(a[:, None], s[:, None].to(torch.int64), 1, [(0, 0)]) % q).to(torch.int16),
                        case["batch"], d["a"], d["s"])
    if op == "matvec":
        d = _product_inputs(case, seed)
        return _exact_matvec(d["a"], d["s"], T.get_params(case["set"]), case["transpose"], case["round"])
    if op == "innerprod":
        d = _product_inputs(case, seed)
        return _exact_inner(d["a"], d["s"], d["aux"], T.get_params(case["set"]), case["epilogue"])
    if op == "encrypt":
        d = _product_inputs(case, seed)
        p = T.get_params(case["set"])
        return _exact_matvec(d["a"], d["s"], p, False, True), _exact_inner(d["b"], d["s"], d["aux"], p, T.IP_ENC)
    if op == "mixed":
        outs = []
        for j in _mixed_inputs(case, seed):
            p = T.get_params(j["set"])
            outs += [_exact_matvec(j["A"], j["s"], p, False, True), _exact_inner(j["b"], j["s"], None, p, T.IP_RAW)]
        return outs
    return None  # the KEM's bytes are hashes
