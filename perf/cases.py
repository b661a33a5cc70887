"""The framework's measured workloads: batched Goldilocks NTTs, coset LDEs, Poseidon2 Merkle trees,
barycentric evaluation, power vectors and uneven job batches, each through the package's public
calls on device buffers that the caller holds (torch tensors of 64-bit words).

listed() gives the named cases, draw() further ones of the same ranges; prepare() builds a case's
inputs and handles, run() is one pass over them, work() the bytes and field operations that pass
cannot do without, and exact() the same results from plain numpy integer arithmetic.
"""
import os
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.abspath("zksync-crypto-gpu_amd"))
import boojum_amd as ba  # noqa: E402

P = 0xFFFFFFFF00000001
EPS = np.uint64(0xFFFFFFFF)
RATE, CAPACITY, WIDTH, ROUNDS = 8, 4, 12, 30


def listed():
    return [
        # one witness column transformed per call: the latency of a single call
        ntt("ntt_1x2p16", 16, 1),
        # a handful of short columns interpolated in a matrix with padded rows (small lookup tables)
        ntt("ntt_inverse_5x2p11", 11, 5, bitrev_inputs=True, inverse=True, pad=24),
        # a trace's columns evaluated on the base domain, the ordinary batch
        ntt("ntt_64x2p20", 20, 64),
        # interpolation from a coset in bit-reversed order, a long trace and an odd number of columns
        ntt("ntt_coset_inverse_19x2p22", 22, 19, bitrev_inputs=True, inverse=True, log_ext=1, coset=1),
        # the commitment LDE of a small circuit: short columns, an odd count
        lde("lde_13x2p14_b4", 14, 13, 2),
        # the commitment LDE at the benchmark's size
        lde("lde_64x2p20_b2", 20, 64, 1),
        # the commitment LDE of a long trace, its monomials kept in natural order as into_monomials gives them
        lde("lde_27x2p22_b4_monomials", 22, 27, 2, natural=True),
        # the Merkle tree over the benchmark LDE's output
        merkle("merkle_64x2p21", 21, 64, 1),
        # the tree over a small oracle: few leaves, a column count that is no multiple of the hash's rate
        merkle("merkle_93x2p14", 14, 93, 0),
        # every column opened at one out-of-domain extension point (the evaluation proof's openings)
        bary("open_64x2p20_at_ext", 20, 64, 1),
        # the shifted copy of a set of columns and the domain's powers that quotient terms multiply by
        shift("omega_shift_2p26", 20, 1 << 26),
        # independent provers' transforms and LDEs of mixed sizes, planned once and launched together
        uneven("uneven_96jobs", 96, 12, 20, 3),
    ]


def ntt(name, log_n, cols, bitrev_inputs=False, inverse=False, log_ext=0, coset=0, pad=0):
    return dict(name=name, kind="ntt", log_n=log_n, cols=cols, bitrev_inputs=bitrev_inputs, inverse=inverse,
                log_ext=log_ext, coset=coset, pad=pad)


def lde(name, log_n, cols, log_blowup, natural=False):
    return dict(name=name, kind="lde", log_n=log_n, cols=cols, log_blowup=log_blowup, natural=natural)


def merkle(name, log_rows, cols, log_rows_per_leaf):
    return dict(name=name, kind="merkle", log_rows=log_rows, cols=cols, log_rows_per_leaf=log_rows_per_leaf)


def bary(name, log_n, cols, point):
    """point: 0 base columns at a base point, 1 base columns at an extension point, 2 extension columns at one"""
    return dict(name=name, kind="bary", log_n=log_n, cols=cols, point=point)


def shift(name, log_degree, count):
    return dict(name=name, kind="shift", log_degree=log_degree, count=count)


def uneven(name, jobs, log_min, log_max, mix):
    return dict(name=name, kind="uneven", jobs=jobs, log_min=log_min, log_max=log_max, mix=mix)


def draw(rng):
    def columns(log_n, log_most, most):
        """a column count spread over its logarithm, with at most 2^log_most elements in all"""
        return int(min(most, 2 ** rng.uniform(0, max(0, log_most - log_n))))

    kind = rng.choice(["ntt", "ntt", "ntt", "lde", "lde", "lde", "merkle", "merkle", "bary", "shift", "uneven"])
    if kind == "ntt":
        log_n = rng.randint(8, 24)
        log_ext = rng.choice([0, 0, 1, 2])
        case = ntt(None, log_n, columns(log_n, 26, 4096), rng.random() < 0.5, rng.random() < 0.5, log_ext,
                   rng.randrange(1 << log_ext), rng.choice([0, 0, 0, 8, 24, 7]))
    elif kind == "lde":
        log_n, log_blowup = rng.randint(10, 22), rng.randint(1, 3)
        case = lde(None, log_n, columns(log_n, 28 - log_blowup, 256), log_blowup, rng.random() < 0.3)
    elif kind == "merkle":
        log_rows = rng.randint(10, 21)
        case = merkle(None, log_rows, columns(log_rows, 27, 200), rng.choice([0, 0, 1, 2]))
    elif kind == "bary":
        log_n, point = rng.randint(10, 22), rng.choice([0, 1, 1, 2])
        case = bary(None, log_n, columns(log_n, 26 - (point == 2), 150), point)
    elif kind == "shift":
        case = shift(None, rng.randint(10, 24), int(2 ** rng.uniform(12, 26.5)))
    else:
        low = rng.randint(10, 14)
        case = uneven(None, rng.randint(8, 96), low, rng.randint(low + 3, 20), rng.randrange(1 << 16))
    del case["name"]
    return case


# ---------------------------------------------------------------- inputs
_context = None


def context():
    """The one context a program keeps: the power tables and the hasher's round constants."""
    global _context
    if _context is None:
        _context = ba.Context.create(12, 12)
        ba.poseidon2.set_round_constants(_context, round_constants())
    return _context


def round_constants():
    return np.random.default_rng(2023).integers(0, P, ROUNDS * WIDTH, dtype=np.uint64)


def words(seed, count):
    """`count` uniform 64-bit words (field elements, read mod p) in device memory"""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randint(-(1 << 63), (1 << 63) - 1, (count,), dtype=torch.int64, device="cuda", generator=g)


def empty(count):
    return torch.zeros(count, dtype=torch.int64, device="cuda")


def view(t):
    return ba.DeviceSlice(t.data_ptr(), t.numel())


class Plan:
    """A batch plan that is given back with its state."""

    def __init__(self, jobs):
        self.plan = ba.batch.BatchPlan(context(), jobs)

    def __del__(self):
        self.plan.destroy()


def uneven_jobs(case):
    """The jobs of an uneven batch: (log_n, inverse, log_blowup or 0 for a plain NTT), a third of them LDEs"""
    r = np.random.default_rng(case["mix"])
    jobs = []
    for _ in range(case["jobs"]):
        log_n, inverse = int(r.integers(case["log_min"], case["log_max"] + 1)), bool(r.integers(0, 2))
        jobs.append((log_n, inverse, int(r.integers(1, 3)) if r.random() < 0.3 else 0))
    return jobs


def prepare(case, seed):
    context()
    kind = case["kind"]
    s = {"case": case}
    if kind == "ntt":
        s["stride"] = (1 << case["log_n"]) + case["pad"]
        s["in"] = words(seed, case["cols"] * s["stride"])
        s["out"] = empty(case["cols"] * s["stride"])
    elif kind == "lde":
        n = case["cols"] << case["log_n"]
        s["in"], s["mono"], s["out"] = words(seed, n), empty(n), empty(n << case["log_blowup"])
    elif kind == "merkle":
        leaves = (1 << case["log_rows"]) >> case["log_rows_per_leaf"]
        s["in"], s["tree"] = words(seed, case["cols"] << case["log_rows"]), empty(2 * CAPACITY * leaves)
        s["stream"] = ba.CudaStream.default()
        s["layers"] = leaves.bit_length()
    elif kind == "bary":
        n, ext = 1 << case["log_n"], case["point"] > 0
        s["in"] = words(seed, (case["cols"] << case["log_n"]) * (2 if case["point"] == 2 else 1))
        s["x"] = words(seed + 1, 1 + ext)
        s["common"], s["coeffs"], s["evals"] = empty(1 + ext), empty(n * (1 + ext)), empty(case["cols"] * (1 + ext))
        s["temp"] = empty(max(1, ba.barycentric.batch_eval_temp_elems(case["point"], n, case["cols"])))
    elif kind == "shift":
        s["in"], s["out"] = words(seed, case["count"]), empty(case["count"])
        s["powers"] = empty(1 << case["log_degree"])
    else:
        jobs, sizes = [], uneven_jobs(case)
        s["in"] = words(seed, sum(1 << log_n for log_n, _, _ in sizes))
        s["out"] = empty(sum(1 << log_n + log_blowup for log_n, _, log_blowup in sizes))
        s["mono"] = empty(max(1, sum(1 << log_n for log_n, _, log_blowup in sizes if log_blowup)))
        at_in, at_out, at_mono = view(s["in"]), view(s["out"]), view(s["mono"])
        for log_n, inverse, log_blowup in sizes:
            n = 1 << log_n
            if log_blowup:
                jobs.append(ba.batch.lde_job(at_in, at_out, log_n, 1, log_blowup, monomials=at_mono))
                at_mono = at_mono.offset(n)
            else:
                jobs.append(ba.batch.ntt_job(at_in, at_out, log_n, 1, n, n, False, inverse))
            at_in, at_out = at_in.offset(n), at_out.offset(n << log_blowup)
        s["plan"] = Plan(jobs)
    # the package's views of the buffers, which a program builds once
    s["views"] = {k: view(v) for k, v in s.items() if isinstance(v, torch.Tensor)}
    return s


def run(s):
    case, v = s["case"], s["views"]
    kind = case["kind"]
    if kind == "ntt":
        ba.ntt.batch_ntt_out_of_place(v["in"], v["out"], case["log_n"], case["cols"], 0, 0, s["stride"], s["stride"],
                                      case["bitrev_inputs"], case["inverse"], case["log_ext"], case["coset"])
        return s["out"]
    if kind == "lde":
        ba.lde.lde_batch(context(), v["in"], case["log_n"], case["cols"], case["log_blowup"], v["out"],
                         monomials=v["mono"], natural_monomials=case["natural"])
        return {"out": s["out"], "mono": s["mono"]}
    if kind == "merkle":
        ba.poseidon2.build_merkle_tree(v["in"], v["tree"], case["log_rows_per_leaf"], s["stream"], s["layers"])
        return s["tree"]
    if kind == "bary":
        ba.barycentric.precompute_lagrange_coeffs(v["x"], v["common"], 7, v["coeffs"], True, ext=case["point"] > 0)
        ba.barycentric.batch_eval(case["point"], v["in"], 1 << case["log_n"], case["cols"], v["coeffs"], v["temp"],
                                  v["evals"])
        return {"coeffs": s["coeffs"], "evals": s["evals"]}
    if kind == "shift":
        ba.ops.get_powers_of_w(case["log_degree"], 0, False, True, v["powers"])
        ba.ops.omega_shift(v["in"], case["log_degree"], 0, False, 1, v["out"])
        return {"powers": s["powers"], "out": s["out"]}
    s["plan"].plan.launch()
    return {"out": s["out"], "mono": s["mono"]}


def work(case):
    """Bytes: each input read once, each output written once; flops: field additions and products."""
    kind = case["kind"]
    if kind == "ntt":
        n = case["cols"] << case["log_n"]
        return {"bytes": 16 * n, "flops": 1.5 * n * case["log_n"]}
    if kind == "lde":
        n, blowup = case["cols"] << case["log_n"], 1 << case["log_blowup"]
        return {"bytes": 8 * n * (2 + blowup), "flops": 1.5 * n * case["log_n"] * (1 + blowup)}
    if kind == "merkle":
        leaves = (1 << case["log_rows"]) >> case["log_rows_per_leaf"]
        per_leaf = -(-(case["cols"] << case["log_rows_per_leaf"]) // RATE)
        permutations = leaves * per_leaf + leaves - 1
        # a permutation: 118 seventh powers of 4 products, 9 external layers, 22 internal ones
        return {"bytes": 8 * ((case["cols"] << case["log_rows"]) + 2 * CAPACITY * leaves),
                "flops": permutations * (118 * 5 + 9 * 60 + 22 * 35)}
    if kind == "bary":
        n, planes = case["cols"] << case["log_n"], 2 if case["point"] == 2 else 1
        out = 1 + (case["point"] > 0)
        return {"bytes": 8 * (n * planes + (out << case["log_n"])), "flops": 2 * n * planes * out}
    if kind == "shift":
        return {"bytes": 16 * case["count"] + (8 << case["log_degree"]), "flops": case["count"]}
    total = {"bytes": 0, "flops": 0}
    for log_n, inverse, log_blowup in uneven_jobs(case):
        one = work(lde(None, log_n, 1, log_blowup) if log_blowup else ntt(None, log_n, 1))
        total = {k: total[k] + one[k] for k in total}
    return total


# ---------------------------------------------------------------- the same results in plain numpy
def add(a, b):
    r = a + b
    r = r + np.where(r < a, EPS, np.uint64(0))
    return np.where(r >= P, r - np.uint64(P), r)


def sub(a, b):
    r = a - b
    return r - np.where(a < b, EPS, np.uint64(0))


def mul(a, b):
    a, b = np.asarray(a, np.uint64), np.asarray(b, np.uint64)
    w = np.uint64(32)
    a0, a1, b0, b1 = a & EPS, a >> w, b & EPS, b >> w
    z = a0 * b0
    x = a1 * b0 + (z >> w)
    y = a0 * b1 + (x & EPS)
    hi = a1 * b1 + (x >> w) + (y >> w)
    lo = (y << w) | (z & EPS)
    t = lo - (hi >> w)
    t = t - np.where(lo < (hi >> w), EPS, np.uint64(0))
    r = t + (hi & EPS) * EPS
    r = r + np.where(r < t, EPS, np.uint64(0))
    return np.where(r >= P, r - np.uint64(P), r)


def power(x, e):
    r = np.ones_like(x)
    while e:
        r = mul(r, x) if e & 1 else r
        x, e = mul(x, x), e >> 1
    return r


def omega(log_n):
    return pow(pow(7, (P - 1) >> 32, P), 1 << (32 - log_n), P)


def powers_of(base, count):
    r = np.ones(1, np.uint64)
    while r.size < count:
        r = np.concatenate([r, mul(r, np.uint64(pow(base, r.size, P)))])
    return r[:count]


def reversal(log_n):
    r = np.zeros(1, np.int64)
    for _ in range(log_n):
        r = np.concatenate([2 * r, 2 * r + 1])
    return r


def transform(x, log_n, root, s=1):
    """sum_j s^j x[.., j] root^(j k), k in natural order"""
    x = mul(x, powers_of(s, 1 << log_n))[:, reversal(log_n)]
    for t in range(log_n):
        half = 1 << t
        x = x.reshape(x.shape[0], -1, 2, half)
        tw = powers_of(pow(root, 1 << (log_n - 1 - t), P), half)
        a, b = x[:, :, 0], mul(x[:, :, 1], tw)
        x = np.stack([add(a, b), sub(a, b)], axis=2).reshape(x.shape[0], -1)
    return x


def interpolate(x, log_n, s=1):
    n = 1 << log_n
    r = transform(x, log_n, pow(omega(log_n), P - 2, P))
    return mul(r, mul(powers_of(pow(s, P - 2, P), n), np.uint64(pow(n, P - 2, P))))


def exact_lde(x, log_n, log_blowup, natural):
    mono, n, rev = interpolate(x, log_n), 1 << log_n, reversal(log_n)
    cosets = [transform(mono, log_n, omega(log_n), 7 * pow(omega(log_n + log_blowup), int(c), P) % P)[:, rev]
              for c in reversal(log_blowup)]
    return np.concatenate(cosets, axis=1).reshape(-1), (mono if natural else mono[:, rev]).reshape(-1)


def permute(s, rc):
    """One Poseidon2 permutation (width 12, 4 + 22 + 4 rounds, x^7) of the states s[lane]"""
    m4 = np.array([[5, 7, 1, 3], [4, 6, 1, 1], [1, 3, 5, 7], [1, 1, 4, 6]], np.uint64)
    external = np.kron(np.ones((3, 3), np.uint64) + np.eye(3, dtype=np.uint64), m4)
    diagonal = [4, 14, 11, 8, 0, 5, 2, 9, 13, 6, 3, 12]

    def matrix(m, s):
        rows = [[mul(x, c) if c > 1 else x for x, c in zip(s, row)] for row in m]
        out = []
        for row in rows:
            acc = row[0]
            for x in row[1:]:
                acc = add(acc, x)
            out.append(acc)
        return out

    def seventh(x):
        x2 = mul(x, x)
        return mul(mul(x2, x), mul(x2, x2))

    s = matrix(external, s)
    for r in range(ROUNDS):
        if 4 <= r < 26:
            s[0] = seventh(add(s[0], rc[r][0]))
            total = s[0]
            for x in s[1:]:
                total = add(total, x)
            s = [add(total, mul(x, np.uint64(1 << d))) for x, d in zip(s, diagonal)]
        else:
            s = matrix(external, [seventh(add(x, rc[r][i])) for i, x in enumerate(s)])
    return s


def exact_tree(case, x):
    rc = round_constants().reshape(ROUNDS, WIDTH)
    rows = 1 << case["log_rows_per_leaf"]
    leaves = (1 << case["log_rows"]) // rows
    zero = np.zeros(leaves, np.uint64)
    values = x.reshape(case["cols"], leaves, rows).transpose(0, 2, 1).reshape(-1, leaves)
    s = [zero] * WIDTH
    for at in range(0, len(values), RATE):
        chunk = list(values[at:at + RATE])
        s = permute(chunk + [zero] * (RATE - len(chunk)) + s[RATE:], rc)
    layer, out = np.stack(s[:CAPACITY]), []
    while True:
        out.append(layer.reshape(-1))
        if layer.shape[1] == 1:
            return np.concatenate(out + [np.zeros(CAPACITY, np.uint64)])
        left, right, zero = layer[:, 0::2], layer[:, 1::2], np.zeros(layer.shape[1] // 2, np.uint64)
        layer = np.stack(permute(list(left) + list(right) + [zero] * 4, rc)[:CAPACITY])


def total_of(x):
    """sum over the last axis"""
    while x.shape[-1] > 1:
        x = add(x[..., 0::2], x[..., 1::2])
    return x[..., 0]


def exact_bary(case, x, ys):
    log_n, n = case["log_n"], 1 << case["log_n"]
    cn = pow(7, n, P)
    w_inv = powers_of(pow(omega(log_n), P - 2, P), n)[reversal(log_n)]
    a, b = int(x[0]) % P, int(x[1]) % P if case["point"] else 0

    def ext_mul(p, q):
        return (p[0] * q[0] + 7 * p[1] * q[1]) % P, (p[0] * q[1] + p[1] * q[0]) % P

    xn, sq = (1, 0), (a, b)
    for _ in range(log_n):
        sq = ext_mul(sq, sq)
    xn = sq
    scale = 7 * pow(n * cn, P - 2, P) % P
    c0, c1 = (xn[0] - cn) * scale % P, xn[1] * scale % P
    d0, d1 = sub(mul(w_inv, np.uint64(a)), np.uint64(7)), mul(w_inv, np.uint64(b))
    norm = power(sub(mul(d0, d0), mul(mul(d1, d1), np.uint64(7))), P - 2)
    i0, i1 = mul(d0, norm), sub(np.zeros_like(d1), mul(d1, norm))
    u = [np.uint64(v) for v in (c0, c1, 7 * c1 % P)]
    l0, l1 = add(mul(i0, u[0]), mul(i1, u[2])), add(mul(i0, u[1]), mul(i1, u[0]))
    if case["point"] == 0:
        return l0, total_of(mul(ys.reshape(-1, n), l0))
    ys = ys.reshape(case["cols"], -1, n)
    e0, e1 = total_of(mul(ys[:, 0], l0)), total_of(mul(ys[:, 0], l1))
    if case["point"] == 2:
        e0 = add(e0, mul(total_of(mul(ys[:, 1], l1)), np.uint64(7)))
        e1 = add(e1, total_of(mul(ys[:, 1], l0)))
    return np.concatenate([l0, l1]), np.stack([e0, e1], axis=1).reshape(-1)


def exact(case, seed):
    """run()'s outputs from numpy, or None where that would take long"""
    flops = work(case)["flops"]
    if flops > (2e8 if case["kind"] == "merkle" else 1e8) or case["kind"] == "uneven":
        return None

    def given(s, count):
        x = words(s, count).cpu().numpy().view(np.uint64)
        return np.where(x >= P, x - np.uint64(P), x)

    def signed(x):
        return np.ascontiguousarray(x).view(np.int64)

    kind = case["kind"]
    if kind == "ntt":
        log_n, n = case["log_n"], 1 << case["log_n"]
        stride, rev = n + case["pad"], reversal(case["log_n"])
        x = given(seed, case["cols"] * stride).reshape(case["cols"], stride)[:, :n]
        x = x[:, rev] if case["bitrev_inputs"] else x
        s = 7 * pow(omega(log_n + case["log_ext"]), case["coset"], P) % P if case["log_ext"] else 1
        r = interpolate(x, log_n, s) if case["inverse"] else transform(x, log_n, omega(log_n), s)
        out = np.zeros((case["cols"], stride), np.uint64)
        out[:, :n] = r if case["bitrev_inputs"] else r[:, rev]
        return signed(out.reshape(-1))
    if kind == "lde":
        x = given(seed, case["cols"] << case["log_n"]).reshape(case["cols"], -1)
        out, mono = exact_lde(x, case["log_n"], case["log_blowup"], case["natural"])
        return {"out": signed(out), "mono": signed(mono)}
    if kind == "merkle":
        return signed(exact_tree(case, given(seed, case["cols"] << case["log_rows"])))
    if kind == "bary":
        planes = 2 if case["point"] == 2 else 1
        ys = given(seed, (case["cols"] << case["log_n"]) * planes)
        coeffs, evals = exact_bary(case, given(seed + 1, 1 + (case["point"] > 0)), ys)
        return {"coeffs": signed(coeffs), "evals": signed(evals)}
    log_n = case["log_degree"]
    w = powers_of(omega(log_n), 1 << log_n)
    factors = np.resize(w, case["count"])
    return {"powers": signed(w[reversal(log_n)]), "out": signed(mul(given(seed, case["count"]), factors))}
