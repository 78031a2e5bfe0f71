"""Performance cases: the randomized-SVD work that programs have this framework do, from one small panel to
the 50,000 x 1,000,000 headline, through the public Python view of the C ABI (pcaone_amd.api).

Kinds of work (the "kind" of a case):

- "run": `Context.run` on genotypes that are resident in HBM (--svd 1 or 2, with or without missing
  genotypes, --emu), each precision form that is used in earnest; what a PCA job does per data set.
- "batch": many independent cohorts in one `Context.batch_run`, then every cohort's U.
- "step": one computeGandH for a caller that keeps its own computeUSV (the reference-side binding): Omega in,
  G and H out.
- "read": .bed rows in host memory made resident (upload, allele counts, both packed layouts).

Genotypes are drawn from a Balding-Nichols model: ancestral frequencies U(0.05, 0.5), Fst 0.1 between
populations, optional missingness at random.
"""
import numpy as np
import torch

from pcaone_amd import api, synth

FST = 0.1
SEED = 112  # the --seed default


def listed():
    return [
        # The smallest calls: a few hundred samples on a chip's worth of markers, plain settings; launches,
        # synchronisations and host steps count here.
        dict(name="svd1_fp32_small", kind="run", svd=1, form="fp32", n=501, m=5003, pops=3, k=4, miss=0.0, emu=False,
             maxp=20, tol=1e-4, v=False),
        # The program's default settings (winSVD, 64 windows, k = 10, FP32) on the small benchmark size.
        dict(name="svd2_fp32_default", kind="run", svd=2, form="fp32", n=2000, m=20000, pops=3, k=10, miss=0.0,
             emu=False, maxp=20, tol=1e-4, v=False),
        # The FP64 form with loadings (-V), as it is used to check the reduced forms; ragged sizes.
        dict(name="svd1_fp64_loadings", kind="run", svd=1, form="fp64", n=3001, m=50021, pops=4, k=10, miss=0.0,
             emu=False, maxp=20, tol=1e-4, v=True),
        # The default precision on an ordinary cohort: array data of 12,001 samples.
        dict(name="svd1_fp32_array", kind="run", svd=1, form="fp32", n=12001, m=150001, pops=5, k=10, miss=0.0,
             emu=False, maxp=20, tol=1e-4, v=False),
        # Real genotype calls: 2 % missing, k = 20 (L = 40).
        dict(name="svd1_bf16_missing", kind="run", svd=1, form="bf16", n=10007, m=120011, pops=4, k=20, miss=0.02,
             emu=False, maxp=20, tol=1e-4, v=False),
        # The fastest form of --svd 1 on an imputed panel of 20,000 samples, a fixed number of passes.
        dict(name="svd1_int8_panel", kind="run", svd=1, form="int8", n=20000, m=500000, pops=6, k=20, miss=0.0,
             emu=False, maxp=7, tol=0.0, v=False),
        # winSVD at its benchmark size (64 windows).
        dict(name="svd2_bf16", kind="run", svd=2, form="bf16", n=10000, m=500000, pops=5, k=20, miss=0.0, emu=False,
             maxp=20, tol=1e-4, v=False),
        # The largest: the headline benchmark, eight passes at L = 80.
        dict(name="svd1_fp8_headline", kind="run", svd=1, form="fp8", n=50000, m=1000000, pops=8, k=40, miss=0.0,
             emu=False, maxp=7, tol=0.0, v=False),
        # EM imputation (--emu) of 10 % missing genotypes; U and V come back.
        dict(name="emu_bf16", kind="run", svd=1, form="bf16", n=6000, m=60000, pops=3, k=10, miss=0.10, emu=True,
             maxp=20, tol=1e-4, v=True),
        # Many cohorts at once.
        dict(name="batch_bf16", kind="batch", form="bf16", cohorts=32, n=500, n_hi=8000, m=10000, m_hi=100000, pops=3,
             k=10, maxp=5, tol=0.0),
        # computeGandH for a caller that keeps its own computeUSV: G and H go back to the host.
        dict(name="step_bf16", kind="step", form="bf16", n=20001, m=100003, pops=4, k=20, miss=0.0),
        # Reading: 1 GB of .bed rows in host memory.
        dict(name="read_rows", kind="read", n=20011, m=200003, pops=2, miss=0.01),
    ]


def _log(rng, lo, hi):
    v = int(round(lo * (hi / lo) ** rng.random()))
    return v + 1 if v < hi and rng.random() < 0.5 and v % 2 == 0 else v


def draw(rng):
    kind = rng.choice(["run", "run", "run", "run", "batch", "step", "read"])
    if kind == "batch":
        n, m = _log(rng, 400, 1500), _log(rng, 5000, 20000)
        return dict(kind=kind, form=rng.choice(["bf16", "fp32", "fp8"]), cohorts=rng.randint(3, 32), n=n,
                    n_hi=n * rng.randint(2, 5), m=m, m_hi=m * rng.randint(2, 5), pops=rng.randint(2, 6),
                    k=rng.randint(3, 16), maxp=rng.randint(3, 7), tol=0.0)
    n = _log(rng, 400, 30000)
    m = min(_log(rng, 5000, 600000), 4 * 10**9 // n)
    pops = rng.randint(2, 8)
    if kind == "read":
        return dict(kind=kind, n=n, m=m, pops=pops, miss=rng.choice([0.0, 0.01, 0.05]))
    k = rng.choice([3, 5, 10, 16, 20, 33, 40])
    if kind == "step":
        return dict(kind=kind, form=rng.choice(["bf16", "fp32", "fp64", "fp8", "int8"]), n=n, m=min(m, 150000),
                    pops=pops, k=k, miss=rng.choice([0.0, 0.02]))
    svd = rng.choice([1, 1, 2])
    emu = svd == 1 and rng.random() < 0.15
    if emu:
        n, m, k = min(n, 6000), min(m, 40000), min(k, 10)
    miss = 0.08 if emu else rng.choice([0.0, 0.0, 0.02])
    return dict(kind=kind, svd=svd, form=rng.choice(["bf16", "fp32", "fp64", "fp8"] + (["int8"] if svd == 1 else [])),
                n=n, m=m, pops=pops, k=k, miss=miss, emu=emu, maxp=20, tol=1e-4, v=emu or rng.random() < 0.3)


# ---------------------------------------------------------------------------------------------------- inputs
def _codes(n, m, pops, miss, seed, each):
    """Calls each(j0, codes) with blocks of PLINK 2-bit codes (rows = SNPs, uint8 values 0..3) on the GPU."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    pop = torch.arange(n, device="cuda") * pops // n
    step = max(1, (1 << 27) // n)
    for j0 in range(0, m, step):
        r = min(step, m - j0)
        p = 0.05 + 0.45 * torch.rand(r, 1, device="cuda", generator=g)
        f = p + torch.sqrt(FST * p * (1 - p)) * torch.randn(r, pops, device="cuda", generator=g)
        f = f.clamp_(0.01, 0.99)[:, pop]
        u = torch.rand(r, n, device="cuda", generator=g)
        # two copies of A1 -> code 00, one -> 10, none -> 11; missing -> 01
        c = torch.where(u < f * f, 0, torch.where(u < f * (2 - f), 2, 3)).to(torch.uint8)
        if miss > 0:
            c.masked_fill_(torch.rand(r, n, device="cuda", generator=g) < miss, 1)
        each(j0, c)


def _rows(n, m, pops, miss, seed):
    """.bed rows (m x ceil(n / 4) bytes) in host memory."""
    out = np.empty((m, (n + 3) // 4), dtype=np.uint8)
    dst = torch.from_numpy(out)

    def pack(j0, c):
        if n % 4:
            c = torch.nn.functional.pad(c, (0, 4 - n % 4))
        q = c.view(c.shape[0], -1, 4)
        dst[j0:j0 + c.shape[0]] = (q[:, :, 0] | q[:, :, 1] << 2 | q[:, :, 2] << 4 | q[:, :, 3] << 6).cpu()

    _codes(n, m, pops, miss, seed, pack)
    return out


def _cohort_sizes(case):
    """Sizes log-spaced over the case's ranges, the two orders interleaved."""
    c = case["cohorts"]
    t = np.arange(c) / max(c - 1, 1)
    n = np.round(case["n"] * (case["n_hi"] / case["n"]) ** t).astype(int)
    m = np.round(case["m"] * (case["m_hi"] / case["m"]) ** ((t * 7919) % 1.0)).astype(int)
    return list(zip(n.tolist(), m.tolist()))


def _params(case):
    kw = dict(svd=case.get("svd", 1), k=case["k"], oversamples=10, maxp=case["maxp"], tol=case["tol"], seed=SEED,
              precision=case["form"])
    if case["kind"] == "batch":
        # chunks named, so that results do not depend on which of the timed candidates wins
        kw.update(kchunk_g=4096, kchunk_h=8192)
    if case.get("emu"):
        kw.update(emu=1, maxiter=20)
    if case.get("v"):
        kw.update(printv=1)
    return api.default_params(**kw)


def _width(case):
    return case["k"] + max(10, case["k"])


def _huge(case):
    return case["n"] * case["m"] > 12 * 10**9


def _omega(case, seed):
    return np.asfortranarray(np.random.default_rng(seed).standard_normal((case["n"], _width(case))))


def prepare(case, seed):
    state = {"case": case}
    if case["kind"] == "read":
        state["rows"] = _rows(case["n"], case["m"], case["pops"], case["miss"], seed)
        state["ctx"] = api.Context(0)
        return state
    ctx = state["ctx"] = api.Context(0)
    if case["kind"] == "batch":
        ctx.batch_upload([(_rows(n, m, case["pops"], 0.0, seed * 1000 + i), n)
                          for i, (n, m) in enumerate(_cohort_sizes(case))])
        state["params"] = _params(case)
        return state
    if _huge(case):  # the framework's own generator: 12.5 GB need not cross the host
        ctx.generate(synth.Spec(seed=seed + 1, nsamples=case["n"], nsnps=case["m"], npops=case["pops"]))
    else:
        ctx.upload_packed(_rows(case["n"], case["m"], case["pops"], case["miss"], seed), case["n"])
    if case["kind"] == "step":
        ctx.standardize()
        ctx.configure(case["form"], _width(case))
        state["omega"] = _omega(case, seed)
    else:
        state["params"] = _params(case)
    return state


def run(state):
    case, ctx = state["case"], state["ctx"]
    if case["kind"] == "read":
        ctx.upload_packed(state["rows"], case["n"])
        n, m, nmiss = ctx.dims()
        return {"n": n, "m": m, "nmiss": nmiss, "F": ctx.allele_freq()}
    if case["kind"] == "batch":
        r = ctx.batch_run(state["params"])
        return {"S": r["S"], "E": r["E"], "epochs": r["epochs"], "status": r["status"],
                "U": [ctx.batch_get_u(c) for c in range(case["cohorts"])]}
    if case["kind"] == "step":
        ctx.set_omega(state["omega"])
        ctx.sketch(0, case["m"], 0)
        return {"G": ctx.get_g(0, case["m"], _width(case)), "H": ctx.get_h(0, _width(case))}
    r = ctx.run(state["params"], want_v=case["v"])
    out = {"U": r.U, "S": r.S, "E": r.E, "epochs": r.info["total_epochs"]}
    if case["v"]:
        out["V"] = r.V
    return out


# ----------------------------------------------------------------------------------------------------- floors
def work(case):
    if case["kind"] == "batch":
        b = f = 0
        L = _width(case)
        for n, m in _cohort_sizes(case):
            b += m * ((n + 3) // 4) + 8 * n * case["k"]
            f += 4 * n * m * L * (case["maxp"] + 1)
        return {"bytes": b, "flops": f}
    n, m = case["n"], case["m"]
    rows = m * ((n + 3) // 4)
    if case["kind"] == "read":
        return {"bytes": rows + 8 * m, "flops": 0}
    L = _width(case)
    if case["kind"] == "step":
        return {"bytes": rows + 8 * L * (2 * n + m), "flops": 4 * n * m * L}
    # one pass over the matrix is two products; a run that stops by its tolerance takes at least two passes
    passes = case["maxp"] + 1 if case["tol"] == 0 else (7 if case["svd"] == 2 else 2)
    return {"bytes": rows + 8 * n * case["k"] + (8 * m * case["k"] if case["v"] else 0),
            "flops": 4 * n * m * L * passes}


# ------------------------------------------------------------------------------------------- values in 64 bits
def _normals(seed, count):
    """std::normal_distribution<double> over std::minstd_rand0 (libstdc++): the order of the Omega draw."""
    p, a = np.uint64(2147483647), 16807
    need = 4 * (int(count / 2 / 0.77) + 4096)
    seq = np.array([seed * a % int(p)], dtype=np.uint64)
    while len(seq) < need:
        seq = np.concatenate([seq, seq * np.uint64(pow(a, len(seq), int(p))) % p])
    r = 2147483646.0
    d = (seq[:need] - np.uint64(1)).astype(np.float64).reshape(-1, 2)
    u = 2.0 * ((d[:, 0] + d[:, 1] * r) / (r * r)) - 1.0
    x, y = u[0::2], u[1::2]
    r2 = x * x + y * y
    keep = (r2 <= 1.0) & (r2 != 0.0)
    x, y, r2 = x[keep], y[keep], r2[keep]
    mult = np.sqrt(-2.0 * np.log(r2) / r2)
    return np.stack([y * mult, x * mult], axis=1).reshape(-1)[:count]


def _dense(case, seed):
    """The standardized genotypes (m x n) in float64: sqrt(2 / (F (1 - F))) (x - F), x = copies / 2, missing 0."""
    A = torch.empty(case["m"], case["n"], dtype=torch.float64, device="cuda")
    val = torch.tensor([1.0, 0.0, 0.5, 0.0], dtype=torch.float64, device="cuda")

    def put(j0, c):
        seen = c != 1
        x = val[c.to(torch.int32)]
        F = x.sum(1, keepdim=True) / seen.sum(1, keepdim=True).clamp(min=1)
        sd = torch.sqrt(F * (1 - F))
        sc = torch.where(sd > 1e-9, 2.0 ** 0.5 / sd, torch.ones_like(sd))
        A[j0:j0 + c.shape[0]] = (x - F) * seen * sc

    _codes(case["n"], case["m"], case["pops"], case["miss"], seed, put)
    return A


def exact(case, seed):
    if case["kind"] == "batch" or case["n"] * case["m"] > 3 * 10**9 and case["kind"] != "read":
        return None
    if case["kind"] == "read":
        F, nmiss = [], []

        def count(j0, c):
            two, one, no = (c == 0).sum(1), (c == 2).sum(1), (c == 1).sum(1)
            F.append((two.double() + 0.5 * one.double()) / (c.shape[1] - no).double().clamp(min=1))
            nmiss.append(int(no.sum()))

        _codes(case["n"], case["m"], case["pops"], case["miss"], seed, count)
        return {"n": case["n"], "m": case["m"], "nmiss": sum(nmiss), "F": torch.cat(F)}
    if case["kind"] == "step":
        A = _dense(case, seed)
        G = A @ torch.from_numpy(_omega(case, seed)).cuda()
        return {"G": G, "H": A.T @ G}
    if case["svd"] != 1 or case["emu"]:
        return None
    # computeUSV of --svd 1 by dense QR and SVD.  U and V are unique up to their signs only: the singular values.
    A, k, L = _dense(case, seed), case["k"], _width(case)
    Q = torch.from_numpy(_normals(SEED, case["n"] * L).reshape(L, case["n"]).T.copy()).cuda()
    prev = None
    for pi in range(case["maxp"] + 1):
        if pi:
            Q = torch.linalg.qr(H)[0]
        G = A @ Q
        H = A.T @ G
        R = torch.linalg.qr(G, mode="r")[1]
        B = torch.linalg.solve_triangular(R.T, H.T, upper=False)
        w, s, _ = torch.linalg.svd(B.T, full_matrices=False)
        u = w[:, :k]
        if prev is not None and 1.0 - float((u.T @ prev).norm(dim=0).mean()) < case["tol"]:
            break
        prev = u
    out = {"U": None, "S": s[:k], "E": s[:k] ** 2 / case["m"], "epochs": pi + 1}
    if case["v"]:
        out["V"] = None
    return out
