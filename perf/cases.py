"""The measured cases: what a program built on this library has it do.

A case is one pass through the public entry points of include/cl2qcd.h (bound by cl2qcd_amd.abi) on
device buffers that the caller owns, or one whole solver call of the C++ drop-in (cl2qcd_amd._host).
Inputs are made with plain torch from the seed alone: SU(3) links disordered around the unit matrix and
Gaussian sources.  `exact` gives the same results in complex128 torch from the same inputs.

Kinds:
  hop          cl2_dslash_eo on one parity, then on the other (the reference's dslash benchmark)
  operator     QplusQminus_eo of the twisted-mass action on one field
  cg           CG iterations on QplusQminus_eo in reduced precision between two reliable updates: source
               in from FP64, `steps` fused iterations (recorded as a graph), correction out to FP64
  block        the same for a block of nrhs right-hand sides in lockstep, one mass or a mass each
  mdagm        MdagM_eo of the staggered action on one field
  cgm          multi-shift CG-M iterations on MdagM_eo, FP32 recurrence with FP64 solutions
  stagg_block  lockstep CG iterations on MdagM_eo + sigma_r for a block of right-hand sides
  solve        a whole solver call on QplusQminus_eo: `cg` (FP64, the reference's algorithm) or the
               reliable-update CG with an FP32 or FP16 inner loop
"""
import ctypes
import math

import torch

from cl2qcd_amd import abi

KAPPA, MU = 0.16, 0.005
MUBAR = 2 * KAPPA * MU
MASS = 0.01
DISORDER = 0.35  # links are unitarised (1 + DISORDER * Gaussian)
FORMATS = {"f64_18": (abi.GAUGE_F64_18, abi.F64), "f64_12": (abi.GAUGE_F64_12, abi.F64),
           "f32": (abi.GAUGE_F32_12, abi.F32), "f16": (abi.GAUGE_F16_12, abi.F16)}
LINK_BYTES = {"f64_18": 144, "f64_12": 96, "f32": 48, "f16": 24}
SPINOR_BYTES = {"f64_18": 192, "f64_12": 192, "f32": 96, "f16": 52}
VEC_BYTES = {"f64_18": 48, "f64_12": 48, "f32": 24}


def listed():
    return [
        # the headline kernel: FP64 hopping term with 18-real links on the largest lattice in use
        {"name": "hop_f64_48x96", "kind": "hop", "ns": 48, "nt": 96, "fmt": "f64_18"},
        # the smallest operator call: an 8^4 test lattice, where launches and latency are everything
        {"name": "operator_f64_8x8", "kind": "operator", "ns": 8, "nt": 8, "fmt": "f64_18"},
        # an ordinary FP32 operator on a ragged lattice (extents not multiples of 4 or 8)
        {"name": "operator_f32_14x22", "kind": "operator", "ns": 14, "nt": 22, "fmt": "f32"},
        # the inner loop of the mixed-precision solve on the largest lattice
        {"name": "cg_f32_48x96", "kind": "cg", "ns": 48, "nt": 96, "fmt": "f32", "steps": 4},
        # the FP16 inner loop of a served single-source request
        {"name": "cg_f16_24x48", "kind": "cg", "ns": 24, "nt": 48, "fmt": "f16", "steps": 10},
        # a propagator: 12 spin-colour sources in lockstep
        {"name": "block_f32_12_32x64", "kind": "block", "ns": 32, "nt": 64, "fmt": "f32", "nrhs": 12, "steps": 2,
         "masses": False},
        # requests of different masses merged into one FP16 block, on a ragged lattice
        {"name": "block_f16_8_18x30", "kind": "block", "ns": 18, "nt": 30, "fmt": "f16", "nrhs": 8, "steps": 4,
         "masses": True},
        # the staggered operator in the reference's precision
        {"name": "mdagm_f64_20x36", "kind": "mdagm", "ns": 20, "nt": 36, "fmt": "f64_18"},
        # the 16 shifts of a rational approximation on a finite-temperature lattice
        {"name": "cgm_16_48x12", "kind": "cgm", "ns": 48, "nt": 12, "fmt": "f32", "nshift": 16, "steps": 10},
        # the lockstep refinement of those shifts
        {"name": "stagg_block_f32_16_48x12", "kind": "stagg_block", "ns": 48, "nt": 12, "fmt": "f32", "nrhs": 16,
         "steps": 4},
        # the plain method, a whole solve: FP64 CG on 8^4
        {"name": "solve_cg_8x8", "kind": "solve", "ns": 8, "nt": 8, "solver": "cg"},
        # a whole mixed-precision solve on the smallest served lattice
        {"name": "solve_f16_16x32", "kind": "solve", "ns": 16, "nt": 32, "solver": "f16"},
    ]


def _even(rng, lo, hi):
    """An even extent in [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, 2 * round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / 2)))


def draw(rng):
    kind = rng.choice(["hop", "operator", "cg", "block", "mdagm", "cgm", "stagg_block", "solve"])
    c = {"kind": kind}
    if kind == "solve":
        c.update(ns=_even(rng, 6, 14), nt=_even(rng, 6, 32), solver=rng.choice(["cg", "f32", "f16"]))
        if c["solver"] == "cg":  # the FP64 solver at the sizes of a test run
            c.update(ns=min(c["ns"], 12), nt=min(c["nt"], 16))
        return c
    if kind in ("hop", "operator", "cg"):
        c.update(ns=_even(rng, 4, 48), nt=_even(rng, 4, 96))
    elif kind in ("mdagm", "cgm"):
        c.update(ns=_even(rng, 4, 48), nt=_even(rng, 4, 48))
    else:
        c.update(ns=_even(rng, 4, 32), nt=_even(rng, 4, 64))
    if kind in ("hop", "operator"):
        c["fmt"] = rng.choice(["f64_18", "f64_12", "f32"])
    elif kind == "cg":
        c.update(fmt=rng.choice(["f32", "f16"]), steps=rng.randint(2, 4))
    elif kind == "block":
        c.update(fmt=rng.choice(["f32", "f16"]), nrhs=rng.choice([2, 4, 8, 12]), steps=2,
                 masses=rng.random() < 0.5)
    elif kind == "mdagm":
        c["fmt"] = rng.choice(["f64_18", "f64_12", "f32"])
    elif kind == "cgm":
        c.update(ns=min(c["ns"], 32), nt=min(c["nt"], 32), fmt="f32", nshift=rng.choice([5, 10, 16]), steps=10)
    else:
        c.update(nt=min(c["nt"], 32), fmt="f32", nrhs=rng.choice([2, 4, 8, 16]), steps=4)
    return c


# ---------------------------------------------------------------- inputs

def _sites(case):
    return case["ns"] ** 3 * case["nt"] // 2


def _generator(seed, what):
    g = torch.Generator(device="cuda")
    g.manual_seed(1000 * int(seed) + what)
    return g


def _randn(shape, seed, what):
    return torch.view_as_complex(torch.randn(*shape, 2, dtype=torch.float64, device="cuda",
                                             generator=_generator(seed, what)))


def _links(case, seed):
    """18-real links in the F64_18 device layout, complex128 [8 = 2 dir + parity][tiles][9][64]."""
    tiles = (_sites(case) + 63) // 64
    m = _randn((8, tiles, 9, 64), seed, 1).mul_(DISORDER)
    for k in (0, 4, 8):
        m[:, :, k] += 1.0
    r0, r1 = m[:, :, 0:3], m[:, :, 3:6]
    r0 /= r0.abs().square().sum(2, keepdim=True).sqrt()
    r1 -= r0 * (r0.conj() * r1).sum(2, keepdim=True)
    r1 /= r1.abs().square().sum(2, keepdim=True).sqrt()
    for k in range(3):
        a, b = (k + 1) % 3, (k + 2) % 3
        m[:, :, 6 + k] = (r0[:, :, a] * r1[:, :, b] - r0[:, :, b] * r1[:, :, a]).conj()
    return m


def _source(case, seed):
    """The FP64 input field or block: complex128 [ncomp][Veo] or [ncomp][Veo][nrhs]."""
    ncomp = 3 if case["kind"] in ("mdagm", "cgm", "stagg_block") else 12
    n = (case["nrhs"],) if "nrhs" in case else ()
    return _randn((ncomp, _sites(case)) + n, seed, 2)


def _shifts(n):
    return [10 ** (-4 + 4 * k / max(1, n - 1)) for k in range(n)]


def _masses(case):
    """kappa and mubar of each right-hand side of a block"""
    n = case["nrhs"]
    if not case["masses"]:
        return [KAPPA] * n, [MUBAR] * n
    kappas = [0.15 + 0.01 * r / (n - 1) for r in range(n)]
    return kappas, [2 * k * (0.003 + 0.017 * r / (n - 1)) for r, k in enumerate(kappas)]


class Lattice:
    """One context, its links in the case's format, and device buffers that outlive the calls on them."""

    def __init__(self, case, seed):
        self.case = case
        self.fmt, self.prec = FORMATS[case["fmt"]]
        self.ctx = abi.Context(case["ns"], case["nt"], theta_t=1.0)
        self.kept, self.graph = [], None
        links = _links(case, seed)
        self.source = _source(case, seed)
        if self.fmt == abi.GAUGE_F64_18:
            self.links = links
        else:
            nbytes = self.ctx.lib.cl2_field_bytes(self.ctx.handle, abi.FIELD_GAUGE, self.fmt)
            self.links = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
            torch.cuda.synchronize()
            self.ctx.gauge_convert(self.links.data_ptr(), self.fmt, links.data_ptr())
            self.ctx.sync()
        self.g = self.links.data_ptr()

    def like_source(self, prec):
        """A zeroed buffer of the source's shape in another precision, in the device layout of that precision."""
        s = self.source
        if prec == abi.F64:
            t = torch.zeros_like(s)
        elif prec == abi.F32:
            shape = (6,) + tuple(s.shape[1:]) + (2,) if s.shape[0] == 12 else tuple(s.shape)
            t = torch.zeros(shape, dtype=torch.complex64, device="cuda")
        else:
            t = torch.zeros(52 * s[0].numel(), dtype=torch.uint8, device="cuda")
        return t

    def field(self, prec, copies=1):
        t = [self.like_source(prec) for _ in range(copies)] if copies > 1 else [self.like_source(prec)]
        t = torch.cat([x.reshape(-1) for x in t]) if copies > 1 else t[0]
        self.kept.append(t)
        return t.data_ptr()

    def scalars(self, values):
        t = torch.tensor(values, dtype=torch.float64, device="cuda")
        self.kept.append(t)
        return t.data_ptr()

    def record(self, body):
        body()  # once before recording, as the solvers do
        self.ctx.graph_begin()
        body()
        g = ctypes.c_void_p()
        self.ctx.graph_end(ctypes.byref(g))
        self.graph = g

    def __del__(self):
        try:
            if self.graph is not None:
                self.ctx.sync()
                self.ctx.lib.cl2_graph_destroy(self.graph)
            self.ctx.close()
        except Exception:
            pass


def _array(values):
    return (ctypes.c_double * len(values))(*values)


def prepare(case, seed):
    if case["kind"] == "solve":
        return _prepare_solve(case, seed)
    L = Lattice(case, seed)
    kind, prec, ctx = case["kind"], L.prec, L.ctx
    lo_bytes = L.like_source(prec).nbytes
    if kind in ("hop", "operator", "mdagm"):
        if prec != abi.F64:  # such a program holds its input in the operator's precision
            given = L.source
            t = L.like_source(prec)
            torch.cuda.synchronize()
            field = abi.FIELD_SU3VEC_EO if kind == "mdagm" else abi.FIELD_SPINOR_EO
            ctx.convert_precision_eo(field, t.data_ptr(), prec, given.data_ptr(), abi.F64)
            ctx.sync()
            L.source = t
            L.like_source = lambda p, t=t: torch.zeros_like(t)
        L.out, L.other = L.like_source(prec), L.like_source(prec)
        L.tmp = L.field(prec, 2)
    elif kind == "cg":
        L.x64 = torch.zeros_like(L.source)
        L.r, L.p, L.x, L.tmp = L.field(prec), L.field(prec), L.field(prec), L.field(prec, 2)
        L.minus_one, L.r2, L.pap = L.scalars([-1.0, 0.0]), L.scalars([1.0, 0.0]), L.scalars([0.0, 0.0])
        L.alpha, L.malpha, L.mbeta = L.scalars([0.0, 0.0]), L.scalars([0.0, 0.0]), L.scalars([0.0, 0.0])
        L.norms = torch.zeros(4, dtype=torch.float64, device="cuda")
        L.bytes = lo_bytes
        torch.cuda.synchronize()
        _start_cg(L)
        L.record(lambda: _cg_iteration(L))
    elif kind in ("block", "stagg_block"):
        n = case["nrhs"]
        L.x64 = torch.zeros_like(L.source)
        L.r, L.p, L.x, L.tmp = L.field(prec), L.field(prec), L.field(prec), L.field(prec, 2)
        L.r2, L.active, L.pap = L.scalars([1.0] * n), L.scalars([1.0] * n), L.scalars([0.0] * 2 * n)
        L.alpha, L.beta = L.scalars([0.0] * 2 * n), L.scalars([0.0] * 2 * n)
        L.norms = torch.zeros(2 * n, dtype=torch.float64, device="cuda")
        L.bytes = lo_bytes
        if kind == "block":
            kappas, mubars = _masses(case)
            L.kappas, L.mubars = (_array(kappas), _array(mubars)) if case["masses"] else (None, None)
        else:
            L.sigma = _array(_shifts(n))
    elif kind == "cgm":
        n = case["nshift"]
        L.solutions = torch.zeros((n,) + tuple(L.source.shape), dtype=torch.complex128, device="cuda")
        L.directions = torch.zeros((n,) + tuple(L.source.shape), dtype=torch.complex64, device="cuda")
        L.xs = (ctypes.c_void_p * n)(*[L.solutions[k].data_ptr() for k in range(n)])
        L.ps = (ctypes.c_void_p * n)(*[L.directions[k].data_ptr() for k in range(n)])
        L.r, L.p, L.tmp = L.field(prec), L.field(prec), L.field(prec)
        # beta, alpha, zeta, zeta_prev: what every solve starts from, in one vector with the running values
        L.state = L.scalars([1.0, 0.0] + [1.0] * 2 * n)
        L.begin = L.scalars([1.0, 0.0] + [1.0] * 2 * n)
        L.beta, L.alpha, L.zeta, L.zeta_prev = (L.state + 8 * k for k in (0, 1, 2, 2 + n))
        L.rr, L.rr_new, L.pap = L.scalars([1.0]), L.scalars([0.0]), L.scalars([0.0])
        L.beta_prev, L.alpha_prev = L.scalars([0.0]), L.scalars([0.0])
        L.sigma, L.active = L.scalars(_shifts(n)), L.scalars([1.0] * n)
        L.zeta_foll, L.beta_vec, L.alpha_vec = (L.scalars([0.0] * n) for _ in range(3))
        L.bytes = lo_bytes
    torch.cuda.synchronize()
    return L


def _prepare_solve(case, seed):
    from cl2qcd_amd import _host as H

    l = H.Lattice([f"--nSpace={case['ns']}", f"--nTime={case['nt']}", "--fermionAction=twistedmass",
                   f"--kappa={KAPPA}", f"--mu={MU}", "--thetaFermionTemporal=1", "--solverMaxIterations=100000"])
    gf = H.Gaugefield(l, False)
    by_site, _ = _geometry(case)
    links = _untiled(case, _links(case, seed))
    aos = torch.empty((2 * _sites(case), 4, 9), dtype=torch.complex128, device="cuda")
    for parity in (0, 1):
        for mu in range(4):
            aos[by_site[parity], mu] = links[2 * mu + parity].reshape(-1, 9)
    gf.import_(torch.view_as_real(aos).reshape(-1, 18).cpu().numpy())
    b, x = H.Spinorfield_eo(l), H.Spinorfield_eo(l)
    source = _source(case, seed)
    b.import_(torch.view_as_real(source.T.contiguous()).reshape(-1, 24).cpu().numpy())
    return {"H": H, "case": case, "lattice": l, "gauge": gf, "b": b, "x": x, "b2": H.squarenorm(b),
            "operator": H.QplusQminus_eo(l), "parameters": l.wilson_parameters()}


# ---------------------------------------------------------------- passes

def _start_cg(L):
    ctx = L.ctx
    ctx.convert_precision_eo(abi.FIELD_SPINOR_EO, L.r, L.prec, L.source.data_ptr(), abi.F64)
    ctx.copy(L.p, L.r, L.bytes)
    ctx.set_zero_eo(L.x, L.prec)
    ctx.squarenorm_eo(L.r2, L.r, L.prec)


def _cg_iteration(L):
    ctx = L.ctx
    ctx.fermionmatrix_eo_cg_step(abi.OP_QPLUSQMINUS_EO, L.r, L.p, L.g, L.fmt, abi.ACTION_TWISTEDMASS, KAPPA, MUBAR,
                                 L.tmp, L.r2, L.pap, L.alpha, L.norms.data_ptr())
    ctx.complex_op(abi.SCALAR_OP_PRODUCT, L.malpha, L.minus_one, L.alpha)
    ctx.cg_beta(L.mbeta, L.r2, L.norms.data_ptr())
    ctx.cg_update_xp(abi.FIELD_SPINOR_EO, L.x, L.p, L.r, L.prec, abi.scalar(dev=L.malpha), abi.scalar(dev=L.mbeta))


def _run_block(L):
    ctx, c, n = L.ctx, L.case, L.case["nrhs"]
    stagg = c["kind"] == "stagg_block"
    if stagg:
        ctx.block_convert_stagg_eo(L.r, L.prec, L.source.data_ptr(), abi.F64, n)
        ctx.block_set_zero_stagg_eo(L.x, L.prec, n)
        ctx.block_squarenorm_stagg_eo(L.r2, L.r, L.prec, n)
    else:
        ctx.block_convert_eo(L.r, L.prec, L.source.data_ptr(), abi.F64, n)
        ctx.block_set_zero_eo(L.x, L.prec, n)
        ctx.block_squarenorm_eo(L.r2, L.r, L.prec, n)
    ctx.copy(L.p, L.r, L.bytes)
    for _ in range(c["steps"]):
        if stagg:
            ctx.MdagM_eo_mrhs_cg_step(L.r, L.p, L.g, L.fmt, MASS, abi.EVEN, L.sigma, L.tmp, n, L.r2, L.active, L.pap,
                                      L.alpha, L.norms.data_ptr())
        else:
            ctx.fermionmatrix_eo_mrhs_cg_step(abi.OP_QPLUSQMINUS_EO, L.r, L.p, L.g, L.fmt, abi.ACTION_TWISTEDMASS,
                                              KAPPA, MUBAR, L.kappas, L.mubars, L.tmp, n, L.r2, L.active, L.pap,
                                              L.alpha, L.norms.data_ptr())
        ctx.block_cg_beta(L.beta, L.r2, L.norms.data_ptr(), L.active, n)
        if stagg:
            ctx.block_cg_update_xp_stagg_eo(L.x, L.p, L.r, L.prec, n, L.alpha, L.beta)
        else:
            ctx.block_cg_update_xp_eo(L.x, L.p, L.r, L.prec, n, L.alpha, L.beta)
    if stagg:
        ctx.block_convert_stagg_eo(L.x64.data_ptr(), abi.F64, L.x, L.prec, n)
    else:
        ctx.block_convert_eo(L.x64.data_ptr(), abi.F64, L.x, L.prec, n)
    return {"x": L.x64, "norms": L.norms}


def _run_cgm(L):
    ctx, n = L.ctx, L.case["nshift"]
    ctx.convert_precision_eo(abi.FIELD_SU3VEC_EO, L.r, L.prec, L.source.data_ptr(), abi.F64)
    ctx.copy(L.p, L.r, L.bytes)
    for k in range(n):
        ctx.set_zero_stagg_eo(L.xs[k], abi.F64)
        ctx.copy(L.ps[k], L.r, L.bytes)
    ctx.scalar_copy(L.state, L.begin, 2 + 2 * n)
    ctx.squarenorm_stagg_eo(L.rr, L.r, L.prec)
    for _ in range(L.case["steps"]):
        ctx.MdagM_eo_cgm_step(L.r, L.p, L.g, L.fmt, MASS, 0.0, abi.EVEN, L.tmp, L.rr, L.pap, L.beta, L.beta_prev,
                              L.rr_new)
        ctx.cgm_alpha_step(n, L.alpha, L.alpha_prev, L.rr_new, L.rr, L.beta, L.beta_prev, L.sigma, L.zeta,
                           L.zeta_prev, L.zeta_foll, L.beta_vec, L.alpha_vec)
        ctx.saxpy_stagg_eo(L.p, L.p, L.r, L.prec, abi.scalar(dev=L.alpha, kind=abi.SCALAR_DEV_REAL))
        ctx.multishift_update_stagg_eo(L.xs, abi.F64, L.ps, L.r, L.prec, n, L.beta_vec, L.zeta_foll, L.alpha_vec,
                                       L.active)
    return {"x": L.solutions}


def _run_solve(s):
    H, solver = s["H"], s["case"]["solver"]
    s["x"].zero()
    if solver == "cg":
        H.cg(s["x"], s["operator"], s["gauge"], s["b"], s["lattice"], 1e-20 * s["b2"], s["parameters"])
    else:
        H.cg_reliable_update(s["x"], s["operator"], s["gauge"], s["b"], s["lattice"], 1e-10, s["parameters"],
                             H.F32 if solver == "f32" else H.F16)
    return {"x": s["x"].get_host()}


def run(state):
    if isinstance(state, dict):
        return _run_solve(state)
    L, ctx, kind = state, state.ctx, state.case["kind"]
    if kind == "hop":
        ctx.dslash_eo(L.out.data_ptr(), L.source.data_ptr(), L.g, L.fmt, abi.EVEN, KAPPA)
        ctx.dslash_eo(L.other.data_ptr(), L.out.data_ptr(), L.g, L.fmt, abi.ODD, KAPPA)
        return {"odd": L.out, "even": L.other}
    if kind == "operator":
        ctx.fermionmatrix_eo(abi.OP_QPLUSQMINUS_EO, L.out.data_ptr(), L.source.data_ptr(), L.g, L.fmt,
                             abi.ACTION_TWISTEDMASS, KAPPA, MUBAR, L.tmp)
        return {"out": L.out}
    if kind == "mdagm":
        ctx.MdagM_eo(L.out.data_ptr(), L.source.data_ptr(), L.g, L.fmt, MASS, abi.EVEN, L.tmp)
        return {"out": L.out}
    if kind == "cg":
        _start_cg(L)
        ctx.graph_launch(L.graph, L.case["steps"])
        ctx.convert_precision_eo(abi.FIELD_SPINOR_EO, L.x64.data_ptr(), abi.F64, L.x, L.prec)
        return {"x": L.x64, "norms": L.norms}
    if kind == "cgm":
        return _run_cgm(L)
    return _run_block(L)


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    """Bytes: every hop reads its links and one field and writes one; an iteration also reads and writes its vectors."""
    v, kind = _sites(case), case["kind"]
    if kind == "solve":  # ~100 iterations of the FP32-sized operator; the solution out
        return {"bytes": v * 100.0 * (4 * (8 * 48 + 2 * 96) + 6 * 96), "flops": v * 100.0 * (4 * 1400 + 400)}
    link, n = 8 * LINK_BYTES[case["fmt"]], case.get("nrhs", 1)
    if kind in ("hop", "operator", "cg", "block"):
        s, hop = n * SPINOR_BYTES[case["fmt"]], n * 1400.0
        if kind == "hop":
            return {"bytes": v * 2.0 * (link + 2 * s), "flops": v * 2 * hop}
        if kind == "operator":
            return {"bytes": v * (4.0 * (link + 2 * s) + 2 * s), "flops": v * (4 * hop + 150)}
        step = 4.0 * (link + 2 * s) - s + 3 * s + 5 * s  # the last hop updates r instead of writing A p
        ends = 2 * n * 192 + 4 * s
        return {"bytes": v * (case["steps"] * step + ends), "flops": v * case["steps"] * (4 * hop + n * 400)}
    s = n * VEC_BYTES[case["fmt"]]
    if kind == "mdagm":
        return {"bytes": v * (2.0 * (link + 2 * s) + s), "flops": v * (2 * 570.0 + 20)}
    if kind == "stagg_block":
        step = 2.0 * (link + 2 * s) + 2 * s + 5 * s
        return {"bytes": v * (case["steps"] * step + 2 * n * 48 + 4 * s), "flops": v * case["steps"] * n * 1300.0}
    k = case["nshift"]
    step = 2.0 * (link + 2 * s) + 2 * s + 3 * s + s + k * (2 * s + 2 * 48)
    return {"bytes": v * (case["steps"] * step + k * (48 + s) + 3 * s), "flops": v * case["steps"] * (1300.0 + 24 * k)}


def tolerance(case):
    """About four times the distance from the 64-bit result that one rounding in the case's types makes."""
    if case["kind"] == "solve":  # both sides stop at |r| <= 1e-10 |b|; the solution's error is that times the condition
        return {"rel": 1e-8 if case["solver"] == "cg" else 5e-8}
    fmt, kind = case["fmt"], case["kind"]
    if fmt in ("f64_18", "f64_12"):
        return {"rel": 2e-15}
    if fmt == "f16":
        return {"rel": 4e-3}
    return {"rel": 5e-7 if kind in ("hop", "operator", "mdagm") else 2e-6}


# ---------------------------------------------------------------- the same in 64 bits

def _geometry(case):
    """Per parity: the site number of each eo index, and the eo indices of its neighbours [parity][0 up, 1 down][mu]."""
    ns, nt = case["ns"], case["nt"]
    s0 = 2 * torch.arange(_sites(case), device="cuda")
    x0, y, z, t = s0 % ns, s0 // ns % ns, s0 // ns ** 2 % ns, s0 // ns ** 3

    def site(x, y, z, t):
        return x % ns + ns * (y % ns + ns * (z % ns + ns * (t % nt)))

    sites, near = [], []
    for parity in (0, 1):
        x = x0 + ((y + z + t) % 2 ^ parity)
        sites.append(site(x, y, z, t))
        near.append([[site(x, y, z, t + d) // 2, site(x + d, y, z, t) // 2, site(x, y + d, z, t) // 2,
                      site(x, y, z + d, t) // 2] for d in (1, -1)])
    return sites, near


def _untiled(case, m):
    """Links [8][Veo][3][3] from the tiled layout."""
    v = _sites(case)
    return m.permute(0, 1, 3, 2).reshape(8, -1, 9)[:, :v].reshape(8, v, 3, 3)


#: rows (A, B, C) of (1 - gamma_mu): h = s_A + C s_B; backward hops take -C.  Directions T, X, Y, Z.
_ROWS = [[(0, 2, 1), (1, 3, 1)], [(0, 3, 1j), (1, 2, 1j)], [(0, 3, 1), (1, 2, -1)], [(0, 2, 1j), (1, 3, -1j)]]


class Exact:
    """The operators in complex128 on fields [ncomp][Veo]."""

    def __init__(self, case, seed):
        self.case = case
        self.links = _untiled(case, _links(case, seed))
        self.sites, self.near = _geometry(case)
        phase = math.pi / case["nt"]  # antiperiodic in time
        self.phase = [complex(math.cos(phase), math.sin(phase)), 1.0, 1.0, 1.0]

    def _times(self, u, h, dagger):
        """u [Veo][3][3] times h [rows][3][Veo]"""
        out = torch.empty_like(h)
        for a in range(3):
            e = [(u[:, b, a].conj() if dagger else u[:, a, b]) for b in range(3)]
            out[:, a] = e[0] * h[:, 0] + e[1] * h[:, 1] + e[2] * h[:, 2]
        return out

    def hop(self, psi, parity, kappa):
        """the Wilson hopping term into the sites of `parity`"""
        psi = psi.reshape(4, 3, -1)
        out = torch.zeros_like(psi)
        for mu in range(4):
            for d in (0, 1):
                to = self.near[parity][d][mu]
                u = self.links[2 * mu + parity] if d == 0 else self.links[2 * mu + 1 - parity][to]
                w = -kappa * (self.phase[mu] if d == 0 else complex(self.phase[mu]).conjugate())
                for a, b, c in _ROWS[mu]:
                    c = c if d == 0 else -c
                    h = (psi[a] + c * psi[b])[None, :, to]
                    r = w * self._times(u, h, d == 1)[0]
                    out[a] += r
                    out[b] += complex(c).conjugate() * r
        return out.reshape(12, -1)

    @staticmethod
    def diagonal(psi, mubar, inverse=False):
        """1 + i mubar gamma5, or its inverse"""
        f = torch.full((12, 1), complex(1, mubar), dtype=torch.complex128, device="cuda")
        f[6:] = complex(1, -mubar)
        return psi / f if inverse else psi * f

    def q(self, psi, kappa, mubar):
        """gamma5 Aee on the odd sublattice (mubar < 0: the minus operator)"""
        out = self.diagonal(psi, mubar) - self.hop(self.diagonal(self.hop(psi, 0, kappa), mubar, True), 1, kappa)
        out[6:] *= -1
        return out

    def qq(self, psi, kappa=KAPPA, mubar=MUBAR):
        return self.q(self.q(psi, kappa, -mubar), kappa, mubar)

    def dks(self, chi, parity):
        ns = self.case["ns"]
        s = self.sites[parity]
        x, y, z = s % ns, s // ns % ns, s // ns ** 2 % ns
        eta = [1 - 2 * ((x + y + z) % 2), torch.ones_like(x), 1 - 2 * (x % 2), 1 - 2 * ((x + y) % 2)]
        out = torch.zeros_like(chi)
        for mu in range(4):
            up, dn = self.near[parity][0][mu], self.near[parity][1][mu]
            w = 0.5 * complex(self.phase[mu])
            f = w * self._times(self.links[2 * mu + parity], chi[None, :, up], False)[0]
            b = w.conjugate() * self._times(self.links[2 * mu + 1 - parity][dn], chi[None, :, dn], True)[0]
            out += eta[mu] * (f - b)
        return out

    def mdagm(self, chi, sigma=0.0):
        return (MASS ** 2 + sigma) * chi - self.dks(self.dks(chi, 1), 0)


def _cg(op, b, steps, rel_tol=0.0):
    """x and (|r|^2, <r, r_old>) after CG iterations"""
    x, r = torch.zeros_like(b), b.clone()
    p, rr = r.clone(), float(torch.linalg.vector_norm(b)) ** 2
    stop, last = rel_tol ** 2 * rr, (rr, 0.0)
    for _ in range(steps):
        ap = op(p)
        alpha = rr / float(torch.vdot(p.reshape(-1), ap.reshape(-1)).real)
        old = r
        x, r = x + alpha * p, r - alpha * ap
        new = float(torch.linalg.vector_norm(r)) ** 2
        last = (new, float(torch.vdot(r.reshape(-1), old.reshape(-1)).real))
        if new <= stop:
            break
        p, rr = r + (new / rr) * p, new
    return x, last


def _pairs(case, psi):
    """a Wilson spinor [12][Veo] in the case's device layout"""
    return psi if case["fmt"] != "f32" else psi.reshape(6, 2, -1).permute(0, 2, 1).contiguous()


def exact(case, seed):
    kind = case["kind"]
    if kind == "solve":
        E = Exact(case, seed)
        x, _ = _cg(E.qq, _source(case, seed), 5000, 1e-14)
        return {"x": torch.view_as_real(x.T.contiguous()).reshape(-1, 24)}
    E, b = Exact(case, seed), _source(case, seed)
    if kind == "hop":
        odd = E.hop(b, 1, KAPPA)
        return {"odd": _pairs(case, odd), "even": _pairs(case, E.hop(odd, 0, KAPPA))}
    if kind == "operator":
        return {"out": _pairs(case, E.qq(b))}
    if kind == "mdagm":
        return {"out": E.mdagm(b)}
    if kind == "cg":
        # <r, r_old> is zero but for rounding, so only |r|^2 has a value to compare with: the vector as a whole
        # is dominated by it
        x, (rr, _) = _cg(E.qq, b, case["steps"])
        return {"x": x, "norms": torch.tensor([rr, 0.0, rr, 0.0], dtype=torch.float64)}
    if kind == "cgm":
        return {"x": _exact_cgm(E, b, _shifts(case["nshift"]), case["steps"])}
    xs, norms = [], []
    for r in range(case["nrhs"]):
        if kind == "block":
            kappas, mubars = _masses(case)
            x, (rr, _) = _cg(lambda p: E.qq(p, kappas[r], mubars[r]), b[..., r].contiguous(), case["steps"])
        else:
            sigma = _shifts(case["nrhs"])[r]
            x, (rr, _) = _cg(lambda p: E.mdagm(p, sigma), b[..., r].contiguous(), case["steps"])
        xs.append(x)
        norms += [rr, 0.0]
    return {"x": torch.stack(xs, -1), "norms": torch.tensor(norms, dtype=torch.float64)}


def _exact_cgm(E, b, sigma, steps):
    """multi-shift CG by its zeta recurrence"""
    n = len(sigma)
    r, p, ps = b.clone(), b.clone(), [b.clone() for _ in sigma]
    xs = [torch.zeros_like(b) for _ in sigma]
    rr, beta, alpha, zeta, before = float(torch.linalg.vector_norm(b)) ** 2, 1.0, 0.0, [1.0] * n, [1.0] * n
    for _ in range(steps):
        ap = E.mdagm(p)
        old_beta, beta = beta, -rr / float(torch.vdot(p.reshape(-1), ap.reshape(-1)).real)
        r = r + beta * ap
        new = float(torch.linalg.vector_norm(r)) ** 2
        old_alpha, alpha = alpha, new / rr
        for k in range(n):
            z, zp = zeta[k], before[k]
            zf = z * zp * old_beta / (beta * old_alpha * (zp - z) + zp * old_beta * (1 - sigma[k] * beta))
            bk = -beta * zf / z
            xs[k] = xs[k] + bk * ps[k]
            ps[k] = zf * r + (-alpha * zf * bk / (z * beta)) * ps[k]
            before[k], zeta[k] = z, zf
        p, rr = alpha * p + r, new
    return torch.stack(xs)
