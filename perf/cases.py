"""Performance cases of the MI355X backend: the calls its users make, with
inputs, work counts, tolerances and a 64-bit restatement of each.

A case is a dict of plain values; its "kind" says which public call it times:

  evolve   DeviceState.evolve: exp(-(it + beta) H) psi by restarted Krylov,
           from a kept initial state to the result on the host
  otoc     DeviceState.otoc: F(t) = <i|A(t) B A(t) B|i>, four evolutions a point
  npoint   syk_block_npoint: one disorder realization of the parity-block SYK
           OTOC or Green's function, from the couplings' seed to v_k / v_0
  ground   DeviceState.ground_state: restarted Lanczos, energy and state
  apply    rp_apply_ops: H psi on device vectors
  arnoldi  rp_apply_ops and rp_gs_pass_fused: one Arnoldi step of a program
           that drives the C interface itself
  batch    rp_batch_*: one restart's Arnoldi steps of a batch of realizations,
           replayed as a captured graph
  train    rp_mlp_loss_grad and rp_mlp_adam: one training step of the proposer

Operators: "syk" (q = 4 SYK of n Majoranas on n/2 sites; k > 0 keeps k n
random quadruples, k = 0 all of them) and "xxz" (open random-field chain of n
sites).  Term lists are (bits, coeff) as rp_terms_upload takes them: two bits
a site, X at bit 2s and Z at bit 2s + 1, the string X^x Z^z with its phase in
the coefficient.
"""
import ctypes as c
import itertools
import math

import numpy as np
import torch

import reapers_amd as ra

GROUP, TUNED = ra.RP_TERMS_ACC_GROUP, ra.RP_TERMS_AUTOTUNE
BATCH_TUNED, BATCH_GROUP = 1, 2       # RP_BATCH_AUTOTUNE, RP_BATCH_ACC_GROUP


# --------------------------------------------------------------------------
# the cases
# --------------------------------------------------------------------------
def listed():
    return [
        # the smallest whole call: dense SYK of 24 Majoranas, checked against
        # exact diagonalization in the literature; latency and launches count
        {"name": "evolve_dense_syk24_f64", "kind": "evolve", "model": "syk", "n": 24, "k": 0, "fp": 64,
         "flags": 0, "t": 2.0, "beta": 0.0, "m": 30, "tol": 1e-12},
        # an ordinary evolution of a sparse SYK state, default upload
        {"name": "evolve_syk36_f32", "kind": "evolve", "model": "syk", "n": 36, "k": 8, "fp": 32,
         "flags": 0, "t": 5.0, "beta": 0.0, "m": 20, "tol": 1e-7},
        # a spin chain in double precision, cooled while it evolves
        {"name": "evolve_xxz19_f64", "kind": "evolve", "model": "xxz", "n": 19, "k": 0, "fp": 64,
         "flags": 0, "t": 0.7, "beta": 0.1, "m": 15, "tol": 1e-10},
        # OTOC points as the benchmark computes them (tuned upload, FP32)
        {"name": "otoc_syk38_f32", "kind": "otoc", "model": "syk", "n": 38, "k": 8, "fp": 32,
         "flags": GROUP | TUNED, "t0": 0.5, "t1": 2.0, "points": 2, "m": 12, "tol": 1e-7},
        # the n-point driver on one realization of a small sector
        {"name": "npoint_syk26_f64", "kind": "npoint", "n": 26, "k": 8, "fp": 64, "what": "otoc",
         "beta": 1.0, "tmax": 3.0, "steps": 3, "m": 16, "tol": 1e-9},
        # ground-state search of a chain
        {"name": "ground_xxz16_f64", "kind": "ground", "model": "xxz", "n": 16, "k": 0, "fp": 64,
         "flags": 0, "m": 12, "iters": 4},
        # the Pauli apply of the headline evolution: 24 qubits, tuned upload
        {"name": "apply_syk48_f32", "kind": "apply", "model": "syk", "n": 48, "k": 8, "fp": 32,
         "flags": GROUP | TUNED},
        # the same operator in double precision, default upload
        {"name": "apply_syk46_f64", "kind": "apply", "model": "syk", "n": 46, "k": 8, "fp": 64,
         "flags": 0},
        # a state beyond every cache: 28 qubits, 2 GiB a vector
        {"name": "apply_syk56_f32", "kind": "apply", "model": "syk", "n": 56, "k": 8, "fp": 32,
         "flags": GROUP},
        # one Arnoldi step of a chain, where the Gram-Schmidt sweeps dominate
        {"name": "arnoldi_xxz23_f32", "kind": "arnoldi", "model": "xxz", "n": 23, "k": 0, "fp": 32,
         "flags": 0, "vecs": 12},
        # a restart of a batch: uneven realizations, four states each
        {"name": "batch_syk32_40x4_f32", "kind": "batch", "nmin": 32, "nmax": 40, "probs": 12, "k": 8,
         "fp": 32, "flags": BATCH_TUNED | BATCH_GROUP, "rhs": 4, "m": 8},
        # one training step of the proposer network on its committed data's size
        {"name": "train_2792", "kind": "train", "samples": 2792},
    ]


def _geo(rng, lo, hi):
    return lo * (hi / lo) ** rng.random()


def draw(rng):
    """One more case of the listed kinds and ranges."""
    kind = rng.choice(["evolve", "evolve", "otoc", "npoint", "ground", "apply", "apply", "arnoldi",
                       "batch", "train"])
    fp = rng.choice([32, 64])
    flags = rng.choice([0, GROUP, GROUP | TUNED]) if fp == 32 else rng.choice([0, TUNED])
    if kind == "train":
        return {"kind": kind, "samples": int(round(_geo(rng, 64, 8192)))}
    if kind == "npoint":
        return {"kind": kind, "n": 2 * rng.randint(8, 13), "k": rng.choice([4, 8]), "fp": 64,
                "what": rng.choice(["otoc", "green"]), "beta": round(rng.uniform(0.0, 2.0), 3),
                "tmax": round(_geo(rng, 0.5, 5.0), 3), "steps": rng.randint(1, 3),
                "m": rng.randint(12, 24), "tol": 1e-9}
    if kind == "batch":
        hi = rng.randint(13, 20 if fp == 32 else 19)
        return {"kind": kind, "nmin": 2 * max(13, hi - rng.randint(0, 4)), "nmax": 2 * hi,
                "probs": rng.randint(2, 12), "k": 8, "fp": fp, "flags": BATCH_TUNED | (BATCH_GROUP if fp == 32 else 0),
                "rhs": rng.choice([2, 4]), "m": rng.randint(2, 8)}
    if kind == "otoc":
        return {"kind": kind, "model": "syk", "n": 2 * rng.randint(9, 19 if fp == 32 else 17),
                "k": rng.choice([4, 8]), "fp": fp, "flags": flags, "t0": round(_geo(rng, 0.1, 0.8), 3),
                "t1": round(_geo(rng, 0.9, 2.0), 3), "points": rng.randint(1, 2),
                "m": rng.randint(8, 20), "tol": 1e-7 if fp == 32 else 1e-10}
    model = rng.choice(["syk", "xxz"])
    case = {"kind": kind, "model": model, "n": 0, "k": 0, "fp": fp, "flags": flags}

    def size(lo, hi):
        sites = rng.randint(lo, hi)
        case["n"] = 2 * sites if model == "syk" else sites
        case["k"] = 0 if model == "xxz" or (sites <= 12 and rng.random() < 0.5) else rng.choice([4, 8])

    if kind == "evolve":
        size(7, 19)
        case.update(t=round(_geo(rng, 0.2, 5.0 if model == "syk" else 1.0), 3),
                    beta=rng.choice([0.0, 0.0, 0.1]), m=rng.randint(12, 30),
                    tol=1e-7 if fp == 32 else 1e-11)
    elif kind == "ground":
        size(8, 17)
        case.update(fp=64, flags=rng.choice([0, TUNED]), m=rng.randint(6, 16), iters=rng.randint(1, 4))
    elif kind == "apply":
        size(7, 26 if fp == 32 else 24)
    else:
        size(9, 23 if fp == 32 else 22)
        case["vecs"] = rng.randint(1, 20)
    return case


# --------------------------------------------------------------------------
# operators
# --------------------------------------------------------------------------
def _majorana(a):
    """(x, z, phase) of chi_a sqrt(2): Z on the sites below a // 2, X or Y on it."""
    s = a // 2
    return (1 << s, (1 << s) - 1, 1.0 + 0j) if a % 2 == 0 else (1 << s, (2 << s) - 1, 1j)


def _product(ops):
    x, z, ph = 0, 0, 1.0 + 0j
    for x1, z1, p1 in ops:
        ph *= p1 * (-1) ** bin(z & x1).count("1")
        x, z = x ^ x1, z ^ z1
    return x, z, ph


def _terms(model, n, k, fp, rng):
    """[(x, z, coefficient)] of the operator sum c X^x Z^z; coefficients are
    values of the state's precision."""
    out = []
    if model == "syk":
        total = math.comb(n, 4)
        if k and k * n < total:
            quads = set()
            while len(quads) < k * n:
                quads.add(tuple(sorted(rng.choice(n, 4, replace=False).tolist())))
            quads = sorted(quads)
        else:
            quads = list(itertools.combinations(range(n), 4))
        sigma = math.sqrt(6.0 / n ** 3 * total / len(quads))
        J = sigma * rng.standard_normal(len(quads))
        ms = [_majorana(a) for a in range(n)]
        for q, j in zip(quads, J):
            x, z, ph = _product([ms[a] for a in q])
            out.append((x, z, 0.25 * j * ph))
    else:
        J, delta, width = 1.0, rng.uniform(0.5, 1.5), rng.uniform(0.5, 4.0)
        for s in range(n - 1):
            pair = 3 << s
            out.append((pair, 0, J))                  # X X
            out.append((pair, pair, -J))              # Y Y = (i X Z)(i X Z)
            out.append((0, pair, J * delta))          # Z Z
        for s in range(n):
            out.append((0, 1 << s, rng.uniform(-width, width)))
    if fp == 32:
        out = [(x, z, complex(np.float32(np.real(v)), np.float32(np.imag(v)))) for x, z, v in out]
    return out


def _bits(terms):
    def spread(v):
        r = 0
        for s in range(32):
            r |= (v >> s & 1) << (2 * s)
        return r
    bits = np.array([spread(x) | spread(z) << 1 for x, z, _ in terms], np.uint64)
    return bits, np.array([v for _, _, v in terms], np.complex128)


def _sites(case):
    return case["n"] // 2 if case.get("model", "syk") == "syk" else case["n"]


def _inputs(case, seed):
    """The operator's terms and the initial state (complex128 values of the
    state's precision, on the GPU), from the seed alone."""
    rng = np.random.default_rng(seed)
    terms = _terms(case["model"], case["n"], case["k"], case["fp"], rng)
    return terms, _gauss(1 << _sites(case), case["fp"], seed)


def _gauss(dim, fp, seed, salt=1):
    g = torch.Generator(device="cuda").manual_seed(1000003 * seed + salt)
    dt = torch.float32 if fp == 32 else torch.float64
    v = torch.view_as_complex(torch.randn(dim, 2, generator=g, device="cuda", dtype=dt))
    return v / torch.linalg.vector_norm(v)


def _orthonormal(dim, k, fp, seed):
    """k orthonormal vectors, rows of a (k, dim) tensor: Cholesky QR, twice."""
    V = torch.stack([_gauss(dim, 64, seed, 10 + i) for i in range(k)])
    for _ in range(2):
        G = torch.stack([torch.stack([torch.vdot(a, b) for b in V]) for a in V])
        R = torch.linalg.cholesky(G.cpu()).conj().cuda()          # V = conj(L) Q over rows
        for i in range(k):
            for j in range(i):
                V[i] -= R[i, j] * V[j]
            V[i] /= R[i, i]
    return V.to(torch.complex64 if fp == 32 else torch.complex128)


# --------------------------------------------------------------------------
# device objects of a program that calls the C interface
# --------------------------------------------------------------------------
class _Terms:
    def __init__(self, terms, sites, fp, flags):
        bits, co = _bits(terms)
        arr = np.ascontiguousarray(np.stack([co.real, co.imag], 1).ravel())
        self.h = c.c_void_p()
        ra.check(ra.hip().rp_terms_upload_ex(c.byref(self.h), _prec(fp), sites, bits.ctypes.data,
                                             arr.ctypes.data, len(bits), flags))

    def __del__(self):
        ra.hip().rp_terms_free(self.h)


class _BatchRun:
    """A batch handle with its basis vectors and the captured restart."""

    def __init__(self, lens, terms, rhs, m, fp, flags):
        lib = ra.hip()
        flat = [_bits(t) for t in terms]
        bits = np.concatenate([b for b, _ in flat])
        co = np.concatenate([v for _, v in flat])
        arr = np.ascontiguousarray(np.stack([co.real, co.imag], 1).ravel())
        off = np.concatenate([[0], np.cumsum([len(b) for b, _ in flat])]).astype(np.int64)
        la = np.array(lens, np.int32)
        self.h, self.g = c.c_void_p(), c.c_void_p()
        ra.check(lib.rp_batch_create(c.byref(self.h), _prec(fp), len(lens), c.c_void_p(la.ctypes.data),
                                     c.c_void_p(bits.ctypes.data), c.c_void_p(arr.ctypes.data),
                                     c.c_void_p(off.ctypes.data), rhs, m, flags))
        rows = sum(1 << x for x in lens)
        dt = torch.complex64 if fp == 32 else torch.complex128
        self.V = [torch.zeros(rows, rhs, dtype=dt, device="cuda") for _ in range(m + 1)]
        self.H = torch.zeros(len(lens) * rhs, m, m + 1, 2, dtype=torch.float64, device="cuda")
        self.nrm = torch.zeros(len(lens) * rhs, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        ptrs = (c.c_void_p * (m + 1))(*[v.data_ptr() for v in self.V])
        ra.check(lib.rp_batch_set_basis(self.h, ptrs, m + 1))
        ra.check(lib.rp_batch_capture_arnoldi(self.h, 0, m, c.c_void_p(self.H.data_ptr()),
                                              c.byref(self.g)))

    def __del__(self):
        if self.g:
            ra.hip().rp_graph_free(self.g)
        if self.h:
            ra.hip().rp_batch_free(self.h)


def _prec(fp):
    return ra.RP_C64 if fp == 32 else ra.RP_C128


def _batch_inputs(case, seed):
    rng = np.random.default_rng(seed)
    span = (case["nmax"] - case["nmin"]) // 2
    sites = [case["nmin"] // 2 + i % (span + 1) for i in range(case["probs"])]
    terms = [_terms("syk", 2 * s, case["k"], case["fp"], rng) for s in sites]
    dt = torch.complex64 if case["fp"] == 32 else torch.complex128
    x = torch.empty(sum(1 << s for s in sites), case["rhs"], dtype=dt, device="cuda")
    at = 0
    for p, s in enumerate(sites):
        for r in range(case["rhs"]):
            x[at:at + (1 << s), r] = _gauss(1 << s, case["fp"], seed, 100 + 4 * p + r)
        at += 1 << s
    return sites, terms, x


def _train_inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def rnd(*shape, scale=1.0):
        return scale * torch.randn(*shape, generator=g, device="cuda")
    n, npar = case["samples"], ra.MLP_NPARAMS
    return {"p": rnd(npar, scale=0.2), "X": rnd(n, ra.MLP_IN), "T": rnd(n, ra.MLP_OUT) + 2.0,
            "W": torch.rand(n, ra.MLP_OUT, generator=g, device="cuda") + 0.5,
            "g": torch.zeros(npar, device="cuda"), "m": rnd(npar, scale=1e-3),
            "v": 1e-4 * torch.rand(npar, generator=g, device="cuda") + 1e-5}


# --------------------------------------------------------------------------
# what a user's program has in hand, and one pass
# --------------------------------------------------------------------------
def prepare(case, seed):
    ra.init(0)
    kind = case["kind"]
    s = {"case": case, "seed": seed}
    if kind == "train":
        s.update(_train_inputs(case, seed))
        return s
    if kind == "npoint":
        return s
    if kind == "batch":
        sites, terms, x = _batch_inputs(case, seed)
        b = _BatchRun(sites, terms, case["rhs"], case["m"], case["fp"], case["flags"])
        s.update(b=b, x=x)
        return s
    terms, psi = _inputs(case, seed)
    sites = _sites(case)
    if kind in ("apply", "arnoldi"):
        s.update(h=_Terms(terms, sites, case["fp"], case["flags"]), v=psi, w=torch.empty_like(psi))
        if kind == "arnoldi":
            k = case["vecs"]
            s["V"] = _orthonormal(psi.numel(), k, case["fp"], seed)
            s["v"] = s["V"][k - 1]
            s["ptrs"] = (c.c_void_p * k)(*[v.data_ptr() for v in s["V"]])
        return s
    bits, co = _bits(terms)
    ra.set_upload_flags(case["flags"])
    s["ham"] = ra.Hamiltonian(sites, bits, co, fp=case["fp"])
    ops = [s["ham"]]
    if kind == "otoc":
        for a in (0, 1):
            x, z, ph = _majorana(a)
            b1, c1 = _bits([(x, z, ph * math.sqrt(0.5))])
            ops.append(ra.Hamiltonian(sites, b1, c1, fp=case["fp"]))
        s["A"], s["B"] = ops[1:]
    for h in ops:
        h.info()                      # uploads the term list
    ra.set_upload_flags(0)
    s["psi"] = ra.DeviceState(sites, fp=case["fp"])
    s["psi"].load(psi.cpu().numpy())
    s["work"] = ra.DeviceState(sites, fp=case["fp"])
    return s


def _times(case):
    return [case["t0"], case["t1"]][:case["points"]]


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    lib = ra.hip()
    if kind == "evolve":
        s["work"].copy_from(s["psi"])
        s["work"].evolve(s["ham"], case["t"], case["beta"], krydim=case["m"], tol=case["tol"])
        return s["work"].store()
    if kind == "otoc":
        return s["psi"].otoc(s["ham"], s["A"], s["B"], _times(case), krydim=case["m"],
                             tol=case["tol"])[0]
    if kind == "npoint":
        return ra.syk_block_npoint(case["n"], case["what"], sp=case["k"], seed=s["seed"],
                                   state_seed=s["seed"] + 1, beta=case["beta"], tmax=case["tmax"],
                                   nsteps=case["steps"], krylov_dim=case["m"], tol=case["tol"],
                                   fp=case["fp"])[1]
    if kind == "ground":
        s["work"].copy_from(s["psi"])
        e = s["work"].ground_state(s["ham"], case["m"], 1e-14, case["iters"])
        return {"energy": e, "state": s["work"].store()}
    if kind == "apply":
        ra.check(lib.rp_apply_ops(s["h"].h, s["w"].data_ptr(), s["v"].data_ptr(), 0))
        return s["w"]
    if kind == "arnoldi":
        k = case["vecs"]
        h, norm, done = np.empty(2 * k), c.c_double(), c.c_int()
        ra.check(lib.rp_apply_ops(s["h"].h, s["w"].data_ptr(), s["v"].data_ptr(), 0))
        ra.check(lib.rp_gs_pass_fused(_prec(case["fp"]), s["ptrs"], k, s["w"].data_ptr(),
                                      s["w"].numel(), h.ctypes.data, c.byref(norm), 1e-300,
                                      c.byref(done)))
        return {"w": s["w"], "h": h, "norm": norm.value, "normalized": done.value}
    if kind == "batch":
        b, x = s["b"], s["x"]
        ra.check(lib.rp_memcpy(b.V[0].data_ptr(), x.data_ptr(), x.numel() * x.element_size(),
                               ra.RP_D2D))
        ra.check(lib.rp_batch_normalize(b.h, 0, c.c_void_p(b.nrm.data_ptr())))
        ra.check(lib.rp_graph_launch(b.g))
        return {"H": b.H, "V": b.V, "norm": b.nrm}
    loss = c.c_double()
    ra.check(lib.rp_mlp_loss_grad(s["p"].data_ptr(), s["X"].data_ptr(), s["T"].data_ptr(),
                                  s["W"].data_ptr(), case["samples"], s["g"].data_ptr(),
                                  c.byref(loss)))
    ra.check(lib.rp_mlp_adam(s["p"].data_ptr(), s["g"].data_ptr(), s["m"].data_ptr(),
                             s["v"].data_ptr(), ra.MLP_NPARAMS, 1e-3, 0.9, 0.999, 1e-8, 1e-4, 100))
    return {"loss": loss.value, "grad": s["g"], "params": s["p"], "m": s["m"], "v": s["v"]}


# --------------------------------------------------------------------------
# what the path cannot do without
# --------------------------------------------------------------------------
def _nterms(case, n=None):
    n = case["n"] if n is None else n
    if case.get("model", "syk") == "xxz":
        return 4 * n - 3
    return min(case["k"] * n, math.comb(n, 4)) if case["k"] else math.comb(n, 4)


def work(case):
    """Bytes: inputs read and outputs written once.  Flops: a term application
    is 4 (a real or imaginary coefficient times a complex amplitude, added);
    a Krylov case counts the applies and sweeps of one basis of m vectors for
    every evolution (its restart count depends on the operator)."""
    kind = case["kind"]
    if kind == "train":
        n, npar = case["samples"], ra.MLP_NPARAMS
        return {"bytes": 4.0 * (n * (ra.MLP_IN + 2 * ra.MLP_OUT) + 8 * npar), "flops": 6.0 * n * npar}
    S = 8 if case["fp"] == 32 else 16
    if kind == "batch":
        b = f = 0.0
        span = (case["nmax"] - case["nmin"]) // 2
        for i in range(case["probs"]):
            n = case["nmin"] + 2 * (i % (span + 1))
            D, m = case["rhs"] * 2.0 ** (n // 2), case["m"]
            b += D * S * (m + 2)
            f += D * (4.0 * m * _nterms(case, n) + 16.0 * m * (m + 1) / 2)
        return {"bytes": b, "flops": f}
    if kind == "npoint":
        D, m = 2.0 ** (case["n"] // 2 - 1), case["m"]
        evolutions = (case["steps"] + 1) * (4 if case["what"] == "otoc" else 2) + 1
        return {"bytes": D * S, "flops": evolutions * D * (4.0 * m * case["k"] * case["n"] + 8.0 * m * m)}
    D, T = 2.0 ** _sites(case), _nterms(case)
    if kind == "apply":
        return {"bytes": 2 * D * S, "flops": 4.0 * D * T}
    if kind == "arnoldi":
        k = case["vecs"]
        return {"bytes": (k + 2) * D * S, "flops": D * (4.0 * T + 16.0 * k)}
    m = case["m"]
    one = D * (4.0 * m * T + 8.0 * m * m)
    if kind == "ground":
        return {"bytes": 2 * D * S, "flops": case["iters"] * D * m * (4.0 * T + 24.0)}
    if kind == "otoc":
        return {"bytes": D * S, "flops": 4 * case["points"] * one}
    return {"bytes": 2 * D * S, "flops": one}


def tolerance(case):
    """About four times the difference of two correct implementations, from
    the error of the FP32 and FP64 paths against exact()."""
    kind, f32 = case["kind"], case.get("fp") == 32
    if kind == "train":       # FP32 sums in another order: 1e-7 in the gradient
        return {"rel": 1e-6, "max": 1e-4}
    if kind == "npoint":      # each point is four evolutions to tol 1e-9
        return {"rel": 2e-8, "max": 2e-7}
    if kind == "ground":      # the recurrence without reorthogonalization amplifies rounding
        return {"rel": 1e-10, "max": 1e-8}
    if kind in ("evolve", "otoc"):        # 1.2e-7 in FP32; tol 1e-10 to 1e-12 in FP64
        return {"rel": 1e-6, "max": 4e-5} if f32 else {"rel": 4e-10, "max": 1e-8}
    if kind == "batch":       # 2.2e-7 in the last Krylov vector
        return {"rel": 1e-6, "max": 4e-5} if f32 else {"rel": 1e-13, "max": 1e-11}
    return {"rel": 4e-7, "max": 1e-5} if f32 else {"rel": 4e-15, "max": 1e-12}


# --------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# --------------------------------------------------------------------------
class _Exact:
    """sum c X^x Z^z on complex128 vectors of 2^sites amplitudes."""

    def __init__(self, terms, sites):
        self.sites, self.by_x = sites, {}
        for x, z, v in terms:
            self.by_x.setdefault(x, []).append((z, complex(v)))
        self.lb = sites // 2
        n = 1 << (sites - self.lb)
        par = torch.zeros(1, dtype=torch.float64, device="cuda") + 1.0
        while par.numel() < n:
            par = torch.cat([par, -par])              # (-1)^popcount(i)
        self.par = par
        self.idx = torch.arange(n, device="cuda")
        self.kept = None
        if len(self.by_x) * 16 << sites < 12 << 30:
            self.kept = {x: self._diag(ts) for x, ts in self.by_x.items()}

    def _diag(self, ts):
        """sum c (-1)^popcount(i & z) over the input index i, as (high, low)."""
        lo = self.idx[:1 << self.lb]
        hi = self.idx[:1 << (self.sites - self.lb)]
        zl = torch.tensor([z & ((1 << self.lb) - 1) for z, _ in ts], device="cuda")
        zh = torch.tensor([z >> self.lb for z, _ in ts], device="cuda")
        co = torch.tensor([v for _, v in ts], dtype=torch.complex128, device="cuda")
        sl = self.par[lo[None, :] & zl[:, None]]
        sh = self.par[hi[None, :] & zh[:, None]]
        if len(ts) == 1:
            return (co[0] * sh[0]).reshape(-1, 1) * sl[0].reshape(1, -1)
        return (sh.to(torch.complex128) * co[:, None]).T @ sl.to(torch.complex128)

    def __call__(self, v):
        nh, nl = 1 << (self.sites - self.lb), 1 << self.lb
        v = v.reshape(nh, nl)
        out = torch.zeros_like(v)
        for x, ts in self.by_x.items():
            # the input amplitude i lands at i ^ x
            t = v * (self.kept[x] if self.kept else self._diag(ts))
            xl, xh = x & (nl - 1), x >> self.lb
            if xh:
                t = t[self.idx[:nh] ^ xh]
            out += t[:, self.idx[:nl] ^ xl] if xl else t
        return out.reshape(-1)


def _expm_exact(H, v, z):
    """exp(z H) v for Hermitian H: Lanczos steps of 30 vectors with full
    reorthogonalization, each as long as its error estimate allows."""
    left = 1.0
    while left > 0:
        V, al, be = [v / torch.linalg.vector_norm(v)], [], []
        for j in range(30):
            w = H(V[j])
            al.append(torch.vdot(V[j], w).real.item())
            for _ in range(2):
                for u in V:
                    w = w - torch.vdot(u, w) * u
            b = torch.linalg.vector_norm(w).item()
            if b < 1e-13:
                break
            be.append(b)
            V.append(w / b)
        k = len(al)
        T = np.diag(al) + np.diag(be[:k - 1], 1) + np.diag(be[:k - 1], -1)
        ev, Q = np.linalg.eigh(T)
        step = left
        while True:
            f = Q @ (np.exp(z * step * ev) * Q[0])
            if len(be) < k or be[k - 1] * abs(z) * step * abs(f[-1]) < 1e-14 * np.linalg.norm(f):
                break
            step /= 2
        nv = torch.linalg.vector_norm(v).item()
        v = sum((nv * f[i]).item() * V[i] for i in range(k))
        left = left - step if step < left else 0.0
    return v


def exact(case, seed):
    kind = case["kind"]
    if kind == "npoint":
        return None                   # its couplings and state come from the driver's own seeds
    if kind == "train":
        return _train_exact(case, seed)
    if kind == "batch":
        return _batch_exact(case, seed)
    terms, psi = _inputs(case, seed)
    H = _Exact(terms, _sites(case))
    v = psi.to(torch.complex128)
    if kind == "apply":
        return H(v)
    if kind == "arnoldi":
        V = _orthonormal(v.numel(), case["vecs"], case["fp"], seed).to(torch.complex128)
        w = H(V[-1])
        h = torch.stack([torch.vdot(u, w) for u in V])
        for a, u in zip(h, V):
            w = w - a * u
        n = torch.linalg.vector_norm(w)
        h = torch.view_as_real(h).reshape(-1).cpu().numpy()
        return {"w": w / n, "h": h, "norm": n.item(), "normalized": None}
    if kind == "evolve":
        return _expm_exact(H, v, -(case["beta"] + 1j * case["t"])).cpu().numpy()
    if kind == "otoc":
        ops = []
        for a in (0, 1):
            x, z, ph = _majorana(a)
            r = ph * math.sqrt(0.5)
            if case["fp"] == 32:
                r = complex(np.float32(r.real), np.float32(r.imag))
            ops.append(_Exact([(x, z, r)], _sites(case)))
        A, B = ops
        out = []
        for t in _times(case):
            u = A(_expm_exact(H, B(v), -1j * t))
            u = B(_expm_exact(H, u, 1j * t))
            u = A(_expm_exact(H, u, -1j * t))
            out.append(torch.vdot(v, _expm_exact(H, u, 1j * t)).item())
        return np.array(out)
    # restarted Lanczos of m vectors without reorthogonalization
    m = case["m"]
    for _ in range(case["iters"]):
        V, al, be = [v], [], []
        for i in range(m):
            w = H(V[i])
            al.append(torch.vdot(V[i], w).real.item())
            if i == m - 1:
                break
            w = w - al[i] * V[i] - (be[i - 1] * V[i - 1] if i else 0.0)
            be.append(torch.linalg.vector_norm(w).item())
            V.append(w / be[i])
        ev, Q = np.linalg.eigh(np.diag(al) + np.diag(be, 1) + np.diag(be, -1))
        v = sum(Q[i, 0].item() * V[i] for i in range(m))
        v = v / torch.linalg.vector_norm(v)
    # an eigenvector's sign is free: the state has no value of its own
    return {"energy": ev[0].item(), "state": None}


def _batch_exact(case, seed):
    sites, terms, x = _batch_inputs(case, seed)
    m, rhs = case["m"], case["rhs"]
    V = [torch.zeros(x.shape, dtype=torch.complex128, device="cuda") for _ in range(m + 1)]
    Hs = torch.zeros(len(sites) * rhs, m, m + 1, 2, dtype=torch.float64, device="cuda")
    norms = torch.zeros(len(sites) * rhs, dtype=torch.float64, device="cuda")
    at = 0
    for p, s in enumerate(sites):
        H, D = _Exact(terms[p], s), 1 << s
        for r in range(rhs):
            q = p * rhs + r
            v = x[at:at + D, r].to(torch.complex128)
            norms[q] = torch.linalg.vector_norm(v)
            B = [v / norms[q]]
            for j in range(m):
                w = H(B[j])
                col = torch.zeros(j + 1, dtype=torch.complex128, device="cuda")
                first = None
                for _ in range(2):
                    h = torch.stack([torch.vdot(u, w) for u in B])
                    for a, u in zip(h, B):
                        w = w - a * u
                    col += h
                    n = torch.linalg.vector_norm(w)
                    first = n if first is None else first
                Hs[q, j, :j + 1] = torch.view_as_real(col)
                Hs[q, j, j + 1, 0], Hs[q, j, j + 1, 1] = n, first
                B.append(w / n)
            for j, u in enumerate(B):
                V[j][at:at + D, r] = u
        at += D
    return {"H": Hs, "V": V, "norm": norms}


def _train_exact(case, seed):
    d = {k: t.double() for k, t in _train_inputs(case, seed).items()}
    p = d["p"].clone().requires_grad_(True)
    cut = np.cumsum([0, 768, 64, 4096, 64, 128, 2]).tolist()
    w1, b1, w2, b2, w3, b3 = [p[a:b] for a, b in zip(cut, cut[1:])]
    h = torch.tanh(d["X"] @ w1.reshape(64, 12).T + b1)
    h = torch.tanh(h @ w2.reshape(64, 64).T + b2)
    y = h @ w3.reshape(2, 64).T + b3
    loss = (d["W"] * (y - d["T"]) ** 2).sum() / case["samples"]
    g, = torch.autograd.grad(loss, p)
    m, v = 0.9 * d["m"] + 0.1 * g, 0.999 * d["v"] + 0.001 * g * g
    mh, vh = m / (1 - 0.9 ** 100), v / (1 - 0.999 ** 100)
    new = d["p"] - 1e-3 * (mh / (vh.sqrt() + 1e-8) + 1e-4 * d["p"])
    return {"loss": loss.item(), "grad": g, "params": new, "m": m, "v": v}
