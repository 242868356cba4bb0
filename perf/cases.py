"""The work that programs built on this library have it do, as measurable cases.

A case is a dict of plain values; `prepare` makes its inputs on the GPU,
`run` takes them once through the public Python entry points, `exact` says
what the outputs are by plain integer arithmetic. The kinds:

  msm        one multi-scalar multiplication (Context.msm_g1 / msm_g2): the
             commitment of a vector, from the smallest proofs' 2^8 points to
             the 2^24 of the library's headline figure. Scalars are uniform, or
             those of a witness (70 % of them 0 or 1, as bits and flags are).
  msm_batch  many MSMs of uneven sizes in one call (Context.msm_batch), the
             shape of a prover that commits to many vectors at once.
  ntt        one transform (Context.ntt, Context.coset_ntt), forward and
             inverse, with the library's scale or the caller's: 2^9 to 2^22 points.
  ntt_batch  many transforms of uneven sizes and directions in one call
             (Context.ntt_batch), with or without the captured graph.
  prove      one Groth16 proof (Groth16.prove) of the multiplication-gate
             circuit (2^log_m rows) or of a p x p matrix product.
  serve      a burst of proof requests of mixed circuit sizes through the
             proof server (ProofServer), waited for until the last is done.

Sizes are those of the library's own tests, tuner and benchmark, odd and
ragged ones among them. All outputs are whole numbers (field elements, points).
"""
import math

import numpy as np
import torch

import liblightzk_amd as z

R = 0x30644E72E131A029B85045B68181585D2833E84879B9709143E1F593F0000001   # Fr
P = 0x30644E72E131A029B85045B68181585D97816A916871CA8D3C208C16D87CFD47   # Fq
MONT = 1 << 256
TOP = 0x30644E72E131A029   # top 64-bit limb of both moduli: a smaller top limb is a canonical value
SERVED = ((12, 0.4), (14, 0.3), (16, 0.2), (18, 0.1))   # log2 rows and share of the served circuits

_shared = {}   # the context, key and server that a program keeps from call to call


def listed():
    return [
        # the smallest commitments: latency and launches
        {"name": "msm_g1_1000", "kind": "msm", "group": 1, "n": 1000, "scalars": "uniform"},
        # a 2^16-row circuit's commitment
        {"name": "msm_g1_2e16", "kind": "msm", "group": 1, "n": 1 << 16, "scalars": "uniform"},
        # a 2^20-row circuit's witness commitment: ragged length, one huge bucket per window
        {"name": "msm_g1_witness_2e20", "kind": "msm", "group": 1, "n": (1 << 20) - 3, "scalars": "witness"},
        # the library's headline: the largest commitment
        {"name": "msm_g1_2e24", "kind": "msm", "group": 1, "n": 1 << 24, "scalars": "uniform"},
        # the G2 query of a proof of about 2^18 rows
        {"name": "msm_g2_200003", "kind": "msm", "group": 2, "n": 200003, "scalars": "uniform"},
        # 32 commitments of 2^10..2^17 points at once
        {"name": "msm_batch_g1_32", "kind": "msm_batch", "group": 1, "count": 32, "lo": 10, "hi": 17, "shape": 5, "graph": False},
        # one small transform: launches and latency
        {"name": "ntt_2e12", "kind": "ntt", "log_n": 12, "coset": False, "inverse": False, "scale": False},
        # interpolation in a 2^18-row proof
        {"name": "intt_2e18", "kind": "ntt", "log_n": 18, "coset": False, "inverse": True, "scale": False},
        # the low-degree extension of a large polynomial
        {"name": "coset_ntt_2e22", "kind": "ntt", "log_n": 22, "coset": True, "inverse": False, "scale": False},
        # 48 transforms of 2^10..2^20 points, all directions, as a captured graph
        {"name": "ntt_batch_48", "kind": "ntt_batch", "count": 48, "lo": 10, "hi": 20, "shape": 6, "graph": True},
        # one proof at a time, the library's plain prover
        {"name": "prove_2e18", "kind": "prove", "circuit": "gates", "size": 18, "public": 8},
        # a proof server under a burst of 40 requests, mostly small
        {"name": "serve_40", "kind": "serve", "requests": 40, "shape": 7},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["msm", "msm", "msm", "msm_batch", "ntt", "ntt_batch", "prove"])
    if kind == "msm":
        group = rng.choice([1, 1, 2])
        n = _log_uniform(rng, 300, (1 << 23) if group == 1 else (1 << 20))
        return {"kind": "msm", "group": group, "n": n, "scalars": rng.choice(["uniform", "uniform", "witness"])}
    if kind == "msm_batch":
        lo = rng.randint(9, 12)
        return {"kind": "msm_batch", "group": rng.choice([1, 1, 2]), "count": rng.randint(3, 40), "lo": lo,
                "hi": lo + rng.randint(2, 5), "shape": rng.randrange(1 << 16), "graph": rng.choice([False, True])}
    if kind == "ntt":
        case = {"kind": "ntt", "log_n": rng.randint(9, 22), "coset": rng.choice([False, True]),
                "inverse": rng.choice([False, True]), "scale": rng.choice([False, True])}
        case["scale"] = case["scale"] and not case["coset"]
        return draw(rng) if any(case.items() <= c.items() for c in listed()) else case
    if kind == "ntt_batch":
        lo = rng.randint(8, 13)
        return {"kind": "ntt_batch", "count": rng.randint(2, 64), "lo": lo, "hi": lo + rng.randint(1, 6),
                "shape": rng.randrange(1 << 16), "graph": rng.choice([False, True])}
    if rng.random() < 0.5:
        return {"kind": "prove", "circuit": "matmul", "size": rng.randint(9, 63)}
    return {"kind": "prove", "circuit": "gates", "size": rng.randint(10, 18), "public": rng.randint(0, 64)}


# ---------------------------------------------------------------- inputs
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _field(g, n, sparse=False):
    """n canonical field elements (int64 [n, 4], Montgomery form) on the GPU."""
    lim = torch.iinfo(torch.int64)
    x = torch.randint(lim.min, lim.max, (n, 4), generator=g, device="cuda", dtype=torch.int64)
    x[:, 3] = torch.randint(0, TOP, (n,), generator=g, device="cuda", dtype=torch.int64)
    if sparse:   # 35 % zeros, 35 % ones
        u = torch.rand(n, generator=g, device="cuda")
        one = torch.from_numpy(_limbs([MONT % R])[0].view(np.int64)).cuda()
        x[u < 0.35] = 0
        x[(u >= 0.35) & (u < 0.7)] = one
    return x


def _context():
    if "ctx" not in _shared:
        _shared["ctx"] = z.Context(0)
    return _shared["ctx"]


def _msm_inputs(ctx, g, group, n, sparse=False):
    """Scalars s, and bases k_i G with the k they come from."""
    s, k = _field(g, n, sparse), _field(g, n)
    bases = torch.empty((n, 8 * group), dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    (ctx.fixbase_g1 if group == 1 else ctx.fixbase_g2)(k.data_ptr(), n, bases.data_ptr())
    ctx.sync()
    return s, k, bases


def _shape(case):
    """Sizes of a batch: part of the case, the same for every seed."""
    rng = np.random.default_rng([case["shape"], case["count"]])
    return rng, case["count"], case["lo"], case["hi"]


def _batch_sizes(case):
    rng, count, lo, hi = _shape(case)
    return [int(2 ** (lo + (hi - lo) * u)) for u in rng.random(count)]


def _batch_transforms(case):
    rng, count, lo, hi = _shape(case)
    return [(int(k), int(d)) for k, d in zip(rng.integers(lo, hi + 1, count), rng.integers(0, 4, count))]


def _key(case):
    """The proving key of a circuit: a prover keeps one and proves many statements with it."""
    what = (case["circuit"], case["size"], case.get("public"))
    if _shared.get("key_of") != what:
        old = _shared.pop("key", None)
        if old is not None:
            old.close()
        if case["circuit"] == "matmul":
            _shared["key"] = z.Groth16.matmul(_context(), 2, case["size"])
        else:
            _shared["key"] = z.Groth16(_context(), 2, case["size"], case["public"])
        _shared["key_of"] = what
    return _shared["key"]


def _server():
    if "server" not in _shared:
        srv = z.ProofServer(0, max_batch=32)
        _shared["circuits"] = [srv.add_circuit(11 + log_m, log_m) for log_m, _ in SERVED]
        srv.start()
        _shared["server"] = srv
    return _shared["server"], _shared["circuits"]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "serve":
        srv, circuits = _server()
        rng = np.random.default_rng(case["shape"])
        which = rng.choice(len(SERVED), size=case["requests"], p=[w for _, w in SERVED])
        reqs = [(circuits[w], srv.witness(circuits[w], seed * 64 + i), z.Groth16.rs(seed * 64 + i)) for i, w in enumerate(which)]
        return {"kind": kind, "server": srv, "requests": reqs}
    ctx = _context()
    if kind == "prove":
        key = _key(case)
        return {"kind": kind, "key": key, "z": key.witness(seed), "rs": key.rs(seed)}
    g = _generator(seed)
    if kind == "msm":
        s, _, bases = _msm_inputs(ctx, g, case["group"], case["n"], case["scalars"] == "witness")
        out = torch.zeros(12 * case["group"], dtype=torch.int64, device="cuda")
        return {"kind": kind, "ctx": ctx, "group": case["group"], "n": case["n"], "s": s, "bases": bases, "out": out}
    if kind == "msm_batch":
        sizes = _batch_sizes(case)
        group, top = case["group"], sum(sizes)
        s, _, bases = _msm_inputs(ctx, g, group, top)
        out = torch.zeros((len(sizes), 12 * group), dtype=torch.int64, device="cuda")
        jobs, at = [], 0
        for i, n in enumerate(sizes):
            jobs.append((s[at].data_ptr(), bases[at].data_ptr(), n, out[i].data_ptr()))
            at += n
        return {"kind": kind, "ctx": ctx, "group": group, "jobs": jobs, "graph": case["graph"], "s": s, "bases": bases, "out": out}
    if kind == "ntt":
        x, factor = _field(g, 1 << case["log_n"]), _field(g, 1) if case["scale"] else None
        return {"kind": kind, "ctx": ctx, "x": x, "coset": case["coset"], "inverse": case["inverse"], "factor": factor}
    todo = _batch_transforms(case)
    x = _field(g, sum(1 << k for k, _ in todo))
    jobs, at = [], 0
    for k, d in todo:
        jobs.append((x[at].data_ptr(), 1 << k, d))
        at += 1 << k
    return {"kind": "ntt_batch", "ctx": ctx, "x": x, "jobs": jobs, "graph": case["graph"]}


def run(state):
    kind = state["kind"]
    if kind == "msm":
        fn = state["ctx"].msm_g1 if state["group"] == 1 else state["ctx"].msm_g2
        fn(state["s"].data_ptr(), state["bases"].data_ptr(), state["n"], state["out"].data_ptr())
        return state["out"]
    if kind == "msm_batch":
        state["ctx"].msm_batch(state["group"], state["jobs"], graph=state["graph"])
        return state["out"]
    if kind == "ntt":
        x = state["x"]
        if state["coset"]:
            state["ctx"].coset_ntt(x.data_ptr(), x.shape[0], state["inverse"])
        else:
            factor = state["factor"]
            state["ctx"].ntt(x.data_ptr(), x.shape[0], None, state["inverse"], None if factor is None else factor.data_ptr())
        return x
    if kind == "ntt_batch":
        state["ctx"].ntt_batch(state["jobs"], graph=state["graph"])
        return state["x"]
    if kind == "prove":
        return state["key"].prove(state["z"], state["rs"]).view(np.int64)
    srv = state["server"]
    ids = [srv.submit(c, w, rs) for c, w, rs in state["requests"]]
    proofs = []
    for rid in ids:
        status, proof, _ = srv.wait(rid)
        if status != 1:
            raise z.HzkError("request failed: %d" % status)
        proofs.append(proof.view(np.int64))
    return np.stack(proofs)


# ---------------------------------------------------------------- the work of one pass
# flops: 32 x 32-bit integer multiply-adds, two operations each. A product in
# either field is 8 x 8 limb products and as many for its reduction; a point
# addition takes 10 field products in G1 and 3 times that in G2.
PRODUCT = 2 * 128


def _additions(n):
    """Point additions of a bucket method with its best window: no program does with fewer."""
    return min(math.ceil(254 / c) * (n + 2.0 ** c) for c in range(2, 25))


def _msm_work(group, n):
    return n * (32 + 64 * group) + 96 * group, _additions(n) * 10 * (1 if group == 1 else 3) * PRODUCT


def _ntt_work(k):
    return 64 << k, (k << k) / 2 * PRODUCT


def _prove_work(rows):
    k = max(4, math.ceil(math.log2(rows)))
    # the witness comes in; three products with it and the quotient; G1 queries A, L and H, G2 query B
    byts, ops = 96 << k, 0
    for group, n in ((1, rows), (1, 2 * rows), (2, rows)):
        b, o = _msm_work(group, n)
        byts, ops = byts + b, ops + o
    return byts, ops + 7 * _ntt_work(k)[1]


def work(case):
    kind = case["kind"]
    if kind == "msm":
        parts = [_msm_work(case["group"], case["n"])]
    elif kind == "msm_batch":
        parts = [_msm_work(case["group"], n) for n in _batch_sizes(case)]
    elif kind == "ntt":
        parts = [_ntt_work(case["log_n"])]
    elif kind == "ntt_batch":
        parts = [_ntt_work(k) for k, _ in _batch_transforms(case)]
    elif kind == "prove":
        p = case["size"]
        parts = [_prove_work(2 ** p if case["circuit"] == "gates" else p ** 3 + p ** 2)]
    else:
        rng = np.random.default_rng(case["shape"])
        which = rng.choice(len(SERVED), size=case["requests"], p=[w for _, w in SERVED])
        parts = [_prove_work(2 ** SERVED[w][0]) for w in which]
    return {"bytes": float(sum(b for b, _ in parts)), "flops": float(sum(o for _, o in parts))}


# ---------------------------------------------------------------- plain integer arithmetic
def _limbs(values):
    return np.array([[(v >> (64 * i)) & (2 ** 64 - 1) for i in range(4)] for v in values], dtype=np.uint64)


def _ints(x):
    """Field elements on the GPU (Montgomery form) as Python integers, still in that form."""
    b = x.cpu().numpy().tobytes()
    return [int.from_bytes(b[32 * i: 32 * i + 32], "little") for i in range(len(b) // 32)]


def _g1_mul(k):
    """k (1, 2) on y^2 = x^3 + 3, affine, or None."""
    acc, q = None, (1, 2)

    def add(a, b):
        if a is None or b is None:
            return a or b
        if a[0] == b[0]:
            if (a[1] + b[1]) % P == 0:
                return None
            m = 3 * a[0] * a[0] * pow(2 * a[1], -1, P) % P
        else:
            m = (b[1] - a[1]) * pow(b[0] - a[0], -1, P) % P
        x = (m * m - a[0] - b[0]) % P
        return x, (m * (a[0] - x) - a[1]) % P

    while k:
        if k & 1:
            acc = add(acc, q)
        q = add(q, q)
        k >>= 1
    return acc


def _g1_result(s, k):
    inv = pow(MONT, -2, R)
    pt = _g1_mul(sum(a * b for a, b in zip(s, k)) * inv % R)
    x, y, w = (0, 1, 0) if pt is None else (pt[0], pt[1], 1)
    return _limbs([v * MONT % P for v in (x, y, w)]).view(np.int64).reshape(-1)


def _ntt_ints(x, k, kind, scale=None):
    """Transform kinds 0 forward, 1 inverse, 2 coset forward, 3 coset inverse (coset 5 <w>).
    scale (a plain factor) takes the place of an inverse transform's 1 / n."""
    n = 1 << k
    w = pow(5, (R - 1) >> k, R)
    if kind == 2:
        c = 1
        x = list(x)
        for j in range(n):
            x[j] = x[j] * c % R
            c = c * 5 % R
    if kind & 1:
        w = pow(w, -1, R)
    x = [x[int(format(j, "0%db" % k)[::-1], 2)] for j in range(n)] if k else list(x)
    half = 1
    while half < n:
        step = pow(w, n // (2 * half), R)
        tw = [1] * half
        for j in range(1, half):
            tw[j] = tw[j - 1] * step % R
        for b in range(0, n, 2 * half):
            for j in range(half):
                u, v = x[b + j], x[b + j + half] * tw[j] % R
                x[b + j], x[b + j + half] = (u + v) % R, (u - v) % R
        half *= 2
    if kind & 1 or scale is not None:
        c, g = pow(n, -1, R) if scale is None else scale, pow(5, -1, R) if kind == 3 else 1
        for j in range(n):
            x[j] = x[j] * c % R
            c = c * g % R
    return x


def exact(case, seed):
    kind = case["kind"]
    if kind == "msm" and case["group"] == 1 and case["n"] <= 1 << 20:
        s, k, _ = _msm_inputs(_context(), _generator(seed), 1, case["n"], case["scalars"] == "witness")
        return torch.from_numpy(_g1_result(_ints(s), _ints(k)))
    if kind == "msm_batch" and case["group"] == 1:
        sizes = _batch_sizes(case)
        s, k, _ = _msm_inputs(_context(), _generator(seed), 1, sum(sizes))
        s, k, at, out = _ints(s), _ints(k), 0, []
        for n in sizes:
            out.append(_g1_result(s[at: at + n], k[at: at + n]))
            at += n
        return torch.from_numpy(np.stack(out))
    if kind == "ntt" and case["log_n"] <= 16:
        g = _generator(seed)
        x = _ints(_field(g, 1 << case["log_n"]))
        scale = _ints(_field(g, 1))[0] * pow(MONT, -1, R) % R if case["scale"] else None
        y = _ntt_ints(x, case["log_n"], 2 * case["coset"] + case["inverse"], scale)
        return torch.from_numpy(_limbs(y).view(np.int64))
    return None   # a proof, a G2 point or a large transform takes too long here
