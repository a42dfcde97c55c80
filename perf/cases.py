"""Timed workloads of the TLR Cholesky library, through its public entry points.

A case is a dict of plain values; "path" names what a program does with the
library:

  generate    STARSH_gen, then STARSH_check into a dense matrix that is copied
              to the host (the generation half of the harness's --check)
  factor      HiCMA_dpotrf_L of a generated matrix (copied first, since the
              factorization works in place) and the log-likelihood of one z
  likelihood  one step of a maximum-likelihood fit: STARSH_gen, band choice,
              band regeneration, HiCMA_dpotrf_L, log-likelihood
  solve       triangular solves, Sigma^-1 B or the log-likelihood on a factor
              the program holds
  demote      mixed-precision storage: copy of a factor, norms, demotion, and
              the log-likelihood on the demoted factor
  serve       a batch of log-likelihood requests of mixed size through the
              server

kind is the reference's -D number: 2 = 2-D sqexp, 3 = 3-D sqexp, 4 = 3-D exp.
band: 0 = the reference's op-count auto-tuning, -1 = the device time model,
otherwise the band size itself.
"""
import ctypes
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hicma-parsec_amd"))
import hicma_tlr as H  # noqa: E402

NUGGET = 1e-2
EXACT_MAX_N = 34000  # dense FP64 Cholesky up to here


# --------------------------------------------------------------------------
# the cases

def _c(name, path, N, NB, maxrank, kind=2, beta=0.1, eps=1e-8, band=1, **more):
    return dict(name=name, path=path, N=N, NB=NB, maxrank=maxrank, kind=kind, beta=beta, eps=eps, band=band, **more)


def listed():
    return [
        # the smallest call: one kriging / GLS solve on the factor of the reference's CTest problem
        _c("potrs_1rhs_n2700", "solve", 2700, 270, 130, op="potrs", nrhs=1),
        # the log-likelihood of one vector on the factor of the headline problem
        _c("loglik_n90000", "solve", 90000, 900, 150, op="loglik", nrhs=1),
        # cross-validation / prediction: several right-hand sides, ragged last tile, dense band
        _c("potrs_8rhs_ragged_n30011", "solve", 30011, 512, 256, band=-1, op="potrs", nrhs=8),
        # conditional simulation: L^-T of a batch of draws, odd tile size
        _c("backward_20rhs_n8091", "solve", 8091, 465, 160, band=-1, op="backward", nrhs=20),
        # mixed-precision storage of a factor, then the likelihood on it
        _c("demote_loglik_n8100", "demote", 8100, 450, 150, band=-1),
        # the reference's CTest problem in its 3-flow form: every off-diagonal tile low rank, ranks up to NB/3
        _c("factor_3flow_n2700", "factor", 2700, 270, 130),
        # the same with the auto-tuned dense band (2-flow), ragged last tile
        _c("factor_2flow_ragged_n2600", "factor", 2600, 270, 130, band=0),
        # the headline factorization
        _c("factor_n90000", "factor", 90000, 900, 150),
        # 3-D squared-exponential field: high ranks, auto-tuned band
        _c("factor_3d_sqexp_n4096", "factor", 4096, 512, 256, kind=3, beta=0.05, band=0),
        # one step of a maximum-likelihood fit of a 2-D field at the serving tile size
        _c("likelihood_n16384", "likelihood", 16384, 512, 256, beta=0.05, band=-1),
        # compression of a 3-D exponential field (ranks above a third of the tile)
        _c("generate_3d_exp_n4096", "generate", 4096, 512, 256, kind=4),
        # serving: a batch of likelihood requests of mixed size and range on four slots
        _c("serve_6_requests", "serve", 12288, 512, 256, requests=6),
    ]


def _odd(rng, lo, hi):
    """An integer of lo .. hi, spread over its logarithm."""
    return int(round(lo * (hi / lo) ** rng.random()))


def _size(rng, lo, hi, nb_lo, nb_hi, nt_lo):
    """(N, NB): the last tile is ragged but keeps at least 0.7 NB rows, so that
    its ranks stay below half of its rows."""
    while True:
        N, NB = _odd(rng, lo, hi), _odd(rng, nb_lo, nb_hi)
        NT = -(-N // NB)
        if NT >= nt_lo and N - (NT - 1) * NB >= 0.7 * NB:
            return N, NB


def _cubes(rng):
    """(N, NB) of a 3-D problem: tiles of 8 x 8 x 8 grid points, whose ranks stay below half of their rows, the
    last one a few rows short."""
    return 512 * rng.randint(6, 8) - rng.randint(0, 40), 512


def draw(rng):
    path = rng.choice(["solve", "solve", "factor", "factor", "likelihood", "generate", "demote", "serve"])
    eps = rng.choice([1e-8, 1e-8, 1e-8, 1e-6])
    beta = round(rng.uniform(0.06, 0.15), 4)
    c = dict(path=path, kind=2, beta=beta, eps=eps, band=-1)
    if path == "solve":
        c["N"], c["NB"] = _size(rng, 2400, 40000, 270, 900, 8)
        c["op"] = rng.choice(["loglik", "potrs", "forward", "backward"])
        c["nrhs"] = 1 if c["op"] == "loglik" else rng.choice([1, 1, 2, 3, 5, 8, 13])
    elif path == "factor":
        form = rng.choice(["3flow", "2flow", "model", "3d"])
        if form == "3flow":      # every off-diagonal tile low rank
            c["N"], c["NB"] = _size(rng, 2000, 2800, 250, 300, 8)
            c["band"], c["eps"], c["beta"] = 1, 1e-8, 0.1
        elif form == "2flow":    # the reference's band
            c["N"], c["NB"] = _size(rng, 2000, 2800, 250, 300, 8)
            c["band"], c["beta"] = 0, 0.1
        elif form == "model":
            c["N"], c["NB"] = _size(rng, 4000, 40000, 300, 900, 12)
        else:
            c["kind"], c["beta"], c["eps"] = 3, 0.05, 1e-8
            c["N"], c["NB"] = _cubes(rng)
    elif path == "likelihood":
        c["N"], c["NB"] = _size(rng, 4000, 30000, 300, 640, 10)
    elif path == "generate":
        c["kind"] = rng.choice([2, 2, 3, 4])
        if c["kind"] == 2:
            c["N"], c["NB"] = _size(rng, 2400, 10000, 270, 640, 8)
        else:
            c["beta"] = 0.05 if c["kind"] == 3 else 0.1
            c["N"], c["NB"] = _cubes(rng)
    elif path == "demote":
        c["N"], c["NB"] = _size(rng, 4000, 12000, 300, 600, 10)
    else:
        c["N"], c["NB"], c["eps"] = 512 * rng.randint(8, 20), 512, 1e-8
        c["requests"] = rng.randint(2, 6)
    c["maxrank"] = c["NB"] // 2 // 16 * 16  # at most NB / 2, as the factorization asks
    return c


# --------------------------------------------------------------------------
# the workloads

_keep = {}


def _context():
    """The program's one library context."""
    if "ctx" not in _keep:
        _keep["ctx"] = H.Context(0)
    return _keep["ctx"]


def _server():
    if "srv" not in _keep:
        _keep["srv"] = H.Server(0, slots=4, hbm_budget_gb=120.0)
    return _keep["srv"]


def _matrix(case, seed):
    return H.TLRMatrix(_context(), case["N"], case["NB"], case["maxrank"], case["kind"], 1.0, case["beta"], NUGGET,
                       seed)


def _generate(A, case):
    """STARSH_gen and the band the case asks for; info of STARSH_gen."""
    info = A.generate(case["eps"], case["maxrank"], 1)
    band = case["band"]
    if band == 0:
        band = A.auto_tune()
    elif band < 0:
        band = H.band_autotune_model(A.rank_gather(), A.NT, A.NB, H.SERVE_DENSE_TFLOPS, H.SERVE_LR_TFLOPS)
    if band != 1:
        A.regenerate(band)
    return info


def _factored(case, seed):
    A = _matrix(case, seed)
    if _generate(A, case) != 0 or A.potrf(case["eps"], 0, case["maxrank"]) != 0:
        raise RuntimeError("the problem cannot be factored: %r" % (case,))
    return A


def _normal(seed, shape):
    g = torch.Generator().manual_seed(int(seed) * 7919 + 17)
    return torch.randn(shape, generator=g, dtype=torch.float64)


def _requests(case, seed):
    """The requests of a serving batch: sizes from a third of N up to N."""
    r = np.random.default_rng(int(seed))
    q = case["requests"]
    frac = np.linspace(0.34, 1.0, q) if q > 1 else np.array([1.0])
    return [dict(N=int(case["NB"] * max(6, round(f * case["N"] / case["NB"]))), sigma2=0.5 + 1.5 * ((i * 5) % q) / q,
                 beta=0.04 + 0.16 * ((i * 3) % q) / q, seed=int(r.integers(1 << 30)),
                 z=_normal(seed * 31 + i, (int(case["NB"] * max(6, round(f * case["N"] / case["NB"]))),)).numpy())
            for i, f in enumerate(frac)]


def prepare(case, seed):
    s = {"case": case}
    path, N = case["path"], case["N"]
    if path == "serve":
        s["srv"], s["requests"] = _server(), _requests(case, seed)
        return s
    if path == "generate":
        s["A"] = _matrix(case, seed)
        s["D"] = H.Dense(_context(), N)
        s["host"] = torch.zeros((N, N), dtype=torch.float64, pin_memory=True)
        return s
    s["B"] = _normal(seed, (case.get("nrhs", 1), N)).cuda()  # row q: right-hand side q (column major for the library)
    if path == "solve":
        s["A"] = _factored(case, seed)
    elif path == "factor":
        s["P"], s["A"] = _matrix(case, seed), _matrix(case, seed)
        if _generate(s["P"], case) != 0:
            raise RuntimeError("a tile is not compressible: %r" % (case,))
    elif path == "likelihood":
        s["A"] = _matrix(case, seed)
    elif path == "demote":
        s["F"], s["A"] = _factored(case, seed), _matrix(case, seed)
    return s


def _rhs(s):
    """A copy of the right-hand sides for the library to work in."""
    X = s["B"].clone()
    torch.cuda.current_stream().synchronize()  # the library runs on its own streams
    return X


def _ok(rc, what):
    if rc != 0:
        raise RuntimeError("%s: %d" % (what, rc))


def _loglik(s):
    X = _rhs(s)
    ld, qd, ll = ctypes.c_double(), ctypes.c_double(), ctypes.c_double()
    _ok(H.lib().hicma_tlr_loglik(_context().h, s["A"].h, X.data_ptr(), ctypes.byref(ld), ctypes.byref(qd),
                                 ctypes.byref(ll)), "hicma_tlr_loglik")
    return {"y": X, "logdet_quad_loglik": np.array([ld.value, qd.value, ll.value])}


def run(s):
    case = s["case"]
    path, A = case["path"], s.get("A")
    if path == "serve":
        srv = s["srv"]
        tickets = [srv.submit(NB=case["NB"], maxrank=case["maxrank"], eps=case["eps"], nugget=NUGGET, **q)
                   for q in s["requests"]]
        got = [srv.wait(t) for t in tickets]
        return {"values": np.array([[g["logdet"], g["quad"], g["loglik"]] for g in got]),
                "status_band": np.array([[g["status"], g["band"]] for g in got])}
    if path == "generate":
        info = A.generate(case["eps"], case["maxrank"], 1)
        s["D"].uncompress(A)
        _ok(H.lib().hicma_dense_get(s["D"].h, s["host"].data_ptr()), "hicma_dense_get")
        return {"dense": s["host"], "ranks": A.rank_gather(), "info": info}
    if path == "solve":
        if case["op"] == "loglik":
            return _loglik(s)
        X, L, ctx, n, N = _rhs(s), H.lib(), _context().h, case["nrhs"], case["N"]
        if case["op"] == "potrs":
            _ok(L.hicma_tlr_potrs(ctx, A.h, n, X.data_ptr(), N), "hicma_tlr_potrs")
        else:
            _ok(L.hicma_tlr_trsm(ctx, A.h, int(case["op"] == "backward"), n, X.data_ptr(), N), "hicma_tlr_trsm")
        return {"x": X}
    if path == "demote":
        A.copy_from(s["F"])
        normA = A.normf()
        counts = A.demote(1e-5 * normA, 1e-8 * normA)
        return dict(_loglik(s), norm=np.array([normA]), counts=np.array(counts))
    if path == "likelihood":
        _ok(_generate(A, case), "STARSH_gen")
    else:
        A.copy_from(s["P"])
    _ok(A.potrf(case["eps"], 0, case["maxrank"]), "HiCMA_dpotrf_L")
    return _loglik(s)


# --------------------------------------------------------------------------
# what a pass cannot do without

def _rank(case):
    """A typical off-band rank of the problem (2-D sqexp at eps 1e-8: 19 at 100 tile rows, 46 at 10)."""
    NT = -(-case["N"] // case["NB"])
    return min({2: 1.0, 3: 2.0, 4: 3.4}[case["kind"]] * (10.0 + 110.0 / NT ** 0.5), 0.45 * case["NB"])


def _factor_flops(N, NB, r):
    """Dense potrf per diagonal tile, low-rank trsm and syrk per panel tile, and per low-rank update the two
    small products, two QRs of a stack of 2 r columns, the product of their R factors, its SVD and the two new
    factors (the reference's op_counts)."""
    NT = -(-N // NB)
    s = 2 * r
    update = 4.0 * NB * r * r + 2 * (2.0 * NB * s * s - 2.0 * s ** 3 / 3) + s ** 3 + 22.0 * s ** 3 + \
        2 * (4.0 * NB * s * r - 2.0 * r * s * s)
    pairs, triples = NT * (NT - 1) / 2, NT * (NT - 1) * (NT - 2) / 6
    return NT * NB ** 3 / 3.0 + pairs * (NB * NB * r + 4.0 * NB * r * r + 2.0 * NB * NB * r) + triples * update


def work(case):
    N, NB, path = case["N"], case["NB"], case["path"]
    NT = -(-N // NB)
    if path == "serve":
        parts = [work(dict(case, path="likelihood", N=q["N"])) for q in _requests(case, 0)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    r, pairs = _rank(case), NT * (NT - 1) / 2
    diag, low = 8.0 * NT * NB * NB, 8.0 * pairs * 2 * NB * r
    held = diag / 2 + low                       # one triangle of the diagonal tiles, every low-rank tile
    gen = pairs * (10.0 * NB * NB + 4.0 * NB * NB * (r + 10) + 8.0 * NB * (r + 10) ** 2)  # kernel, sketch, two QRs
    once = 2.0 * held / 8                       # one multiply-add per element of the factor
    if path == "generate":
        return {"bytes": diag + low + 2 * 8.0 * N * N, "flops": gen + 2.0 * pairs * NB * NB * r}
    if path == "solve":
        n, passes = case["nrhs"], 2 if case["op"] == "potrs" else 1
        return {"bytes": passes * held + 16.0 * N * n, "flops": passes * n * once}
    if path == "demote":
        return {"bytes": 2 * (diag + low) + held + 16.0 * N, "flops": 2 * once + pairs * 4.0 * NB * r * r}
    flops = _factor_flops(N, NB, r) + once
    if path == "factor":
        return {"bytes": 2 * (diag + low) + held + 16.0 * N, "flops": flops}
    return {"bytes": diag + low + held + 16.0 * N, "flops": flops + gen}


# --------------------------------------------------------------------------
# the same in 64 bits, by dense linear algebra

def _points(N, ndim, seed):
    """The jittered grid in Morton order, (ndim, N)."""
    s = max(1, int(np.ceil(N ** (1.0 / ndim) - 1e-9)))
    while s ** ndim < N:
        s += 1
    g = np.arange(s ** ndim, dtype=np.uint64)
    coord = [(g // np.uint64(s ** d)) % np.uint64(s) for d in range(ndim)]
    code = np.zeros_like(g)
    for d in range(ndim):
        for b in range(int(s).bit_length()):
            code |= ((coord[d] >> np.uint64(b)) & np.uint64(1)) << np.uint64(b * ndim + d)
    order = np.argsort(code, kind="stable")[:N]
    out = np.empty((ndim, N))
    with np.errstate(over="ignore"):
        for d in range(ndim):
            x = np.uint64(seed) * np.uint64(0x632BE59BD9B4E019) + g[order] * np.uint64(ndim) + np.uint64(d)
            z = x + np.uint64(0x9E3779B97F4A7C15)
            z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
            z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
            z = z ^ (z >> np.uint64(31))
            u = (z >> np.uint64(11)).astype(np.float64) * 2.0 ** -53
            out[d] = (coord[d][order].astype(np.float64) + 0.5 + 0.8 * u - 0.4) / s
    return out


def _covariance(N, kind, sigma2, beta, seed):
    p = torch.from_numpy(_points(N, 2 if kind == 2 else 3, seed)).cuda()
    S = torch.zeros((N, N), dtype=torch.float64, device="cuda")
    for x in p:
        S += (x[:, None] - x[None, :]) ** 2
    S = sigma2 * torch.exp(-torch.sqrt(S) / beta) if kind == 4 else sigma2 * torch.exp(S / (-2.0 * beta * beta))
    S.diagonal().add_(NUGGET)
    return S


def _exact_loglik(S, z):
    L = torch.linalg.cholesky(S)
    y = torch.linalg.solve_triangular(L, z.cuda().reshape(-1, 1), upper=False)[:, 0]
    ld, qd = 2.0 * float(L.diagonal().log().sum()), float(y.square().sum())
    return y, [ld, qd, -0.5 * (ld + qd + len(y) * float(np.log(2.0 * np.pi)))]


def exact(case, seed):
    path, N = case["path"], case["N"]
    if N > EXACT_MAX_N:
        return None
    if path == "serve":
        got = [_exact_loglik(_covariance(q["N"], 2, q["sigma2"], q["beta"], q["seed"]), torch.from_numpy(q["z"]))[1]
               for q in _requests(case, seed)]
        return {"values": np.array(got), "status_band": None}
    S = _covariance(N, case["kind"], 1.0, case["beta"], seed)
    if path == "generate":
        return {"dense": torch.triu(S), "ranks": None, "info": None}  # column major: the lower triangle
    B = _normal(seed, (case.get("nrhs", 1), N))
    if path == "solve" and case["op"] != "loglik":
        L, X = torch.linalg.cholesky(S), B.cuda().T.contiguous()
        if case["op"] != "backward":
            X = torch.linalg.solve_triangular(L, X, upper=False)
        if case["op"] != "forward":
            X = torch.linalg.solve_triangular(L.T, X, upper=True)
        return {"x": X.T.contiguous()}
    y, v = _exact_loglik(S, B)
    out = {"y": y.reshape(1, N), "logdet_quad_loglik": np.array(v)}
    if path == "demote":
        out.update(norm=None, counts=None)
    return out
