"""The work a user of this library has it do, as cases that can be timed.

Every case goes through the public entry points of the Python binding: single
kernels (a Dslash, an even-odd operator, a clover build) and whole solves, from
the 8^4 Wilson lattice, where launches and host calls are what counts, to the
48^3x96 lattice of the headline Dslash and mixed-precision solve. Lattices,
kappas, tolerances and source counts are those of this repository's tests and
benchmark; `draw` spreads them over the same ranges with uneven extents.

Inputs come from the seed alone: links U = reunit(exp(0.4 i A)), A traceless
Hermitian with unit-variance Gaussian entries, Gaussian sources, and clover
terms built from the links. Up to 32^3x64 the links and sources are made in
torch and packed through the public packers; the 48^3x96 lattice (6 GB of
canonical links) uses the library's own seeded generators. Spinors come back as
the library stores them: 16-byte words in blocks of 4096 sites (the half
precisions as the stored values beside their per-site FP32 scales).
"""
import ctypes
import functools
import math

import torch

import qphix_amd as q

PRECS = {"f64": q.F64, "f32": q.F32, "f16": q.F16, "bf16": q.BF16}
REAL_BYTES = {"f64": 8, "f32": 4, "f16": 2, "bf16": 2}
STORED = {"f64": torch.float64, "f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
KINDS = {"wilson": q.OP_WILSON, "clover": q.OP_CLOVER, "tmwilson": q.OP_TMWILSON, "tmclover": q.OP_TMCLOVER,
         "ndtmclover": q.OP_NDTMCLOVER}
CSW = 1.0
SITE_BLOCK = 4096
PACKED_VOLUME = 1 << 21  # up to this volume the inputs are made in torch

# lattices of the uneven batch, four sources each
BATCH = ((8, 8, 8, 8), (12, 12, 12, 24), (16, 16, 16, 32), (24, 24, 24, 48))


def _case(name, path, lattice, **more):
    return {"name": name, "path": path, "x": lattice[0], "y": lattice[1], "z": lattice[2], "t": lattice[3], **more}


def listed():
    return [
        # the smallest operator: 2048 sites a parity, the cost is launches and host calls
        _case("wilson_op_8x8x8x8_f64", "op", (8, 8, 8, 8), kind="wilson", prec="f64", c12=False, isign=1, kappa=0.12),
        # CG on M^+M of the same lattice to 1e-12: the smallest solve, bound by the latency of its chain
        _case("wilson_cg_8x8x8x8_f64", "cg", (8, 8, 8, 8), kind="wilson", prec="f64", c12=False, isign=1, kappa=0.12,
              tol=1e-12),
        # an ordinary operator application on a lattice that does not fill the device for long
        _case("clover_op_16x16x16x32_f32", "op", (16, 16, 16, 32), kind="clover", prec="f32", c12=True, isign=1,
              kappa=0.124),
        # the daggered twisted-mass clover operator in the inner-solve precision, on uneven extents
        _case("tmclover_op_20x12x14x22_f16", "op", (20, 12, 14, 22), kind="tmclover", prec="f16", c12=True, isign=-1,
              kappa=0.124, mu=0.005),
        # the non-degenerate doublet: two flavours through one set of links
        _case("doublet_op_16x16x16x32_f64", "op", (16, 16, 16, 32), kind="ndtmclover", prec="f64", c12=False, isign=1,
              kappa=0.124, mu=0.01, eps=0.005),
        # the headline kernel: one clover Dslash of the production lattice
        _case("clover_dslash_48x48x48x96_f32", "dslash", (48, 48, 48, 96), kind="clover", prec="f32", c12=True,
              isign=1, kappa=0.1245),
        # twelve sources (one propagator) through one operator application
        _case("clover_op_12rhs_32x32x32x64_f32", "op_multi", (32, 32, 32, 64), kind="clover", prec="f32", c12=True,
              isign=1, kappa=0.124, nrhs=12),
        # the inverse clover term, rebuilt for every new gauge field (each trajectory's step)
        _case("clover_inverse_24x24x24x48_f64", "clover_build", (24, 24, 24, 48), prec="f64", c12=False, kappa=0.124),
        # the shifted systems of a rational approximation: 12 shifts from 1e-4 to 1
        _case("multishift_cg_12_32x32x32x64_f64", "multishift", (32, 32, 32, 64), kind="clover", prec="f64", c12=False,
              isign=1, kappa=0.124, nshift=12, tol=1e-8),
        # 12 point and 16 Gaussian sources in one block Krylov space
        _case("block_cg_28_24x24x24x48_f32", "block_cg", (24, 24, 24, 48), kind="clover", prec="f32", c12=True,
              isign=1, kappa=0.124, nrhs=28, tol=1e-6),
        # many small systems at once: 16 twisted-mass clover systems on four lattices, FP16 inside FP64
        _case("tmclover_batch_4_lattices_f16", "batch", (24, 24, 24, 48), kind="tmclover", prec="f16", c12=True,
              isign=1, kappa=0.124, nrhs=4, tol=1e-10),
        # the headline solve: FP16 BiCGStab inside FP64 defect correction on the production lattice
        _case("mixed_solve_48x48x48x96_f16", "mixed", (48, 48, 48, 96), kind="clover", prec="f16", c12=True, isign=1,
              kappa=0.1245, tol=1e-10),
    ]


def _log_even(rng, lo, hi):
    return 2 * int(round(math.exp(rng.uniform(math.log(lo / 2), math.log(hi / 2)))))


def draw(rng):
    path = rng.choice(["op", "op", "op", "dslash", "dslash", "op_multi", "op_multi", "clover_build", "cg", "multishift",
                       "block_cg", "mixed", "batch"])
    top = {"op": 1 << 21, "dslash": 1 << 21, "op_multi": 1 << 20, "clover_build": 1 << 19, "cg": 1 << 16,
           "multishift": 1 << 19, "block_cg": 1 << 18, "mixed": 1 << 20, "batch": 1 << 17}[path]
    while True:
        lattice = tuple(_log_even(rng, 4, hi) for hi in (48, 48, 48, 96))
        volume = lattice[0] * lattice[1] * lattice[2] * lattice[3]
        if 1024 <= volume <= top:
            break
    case = {"path": path, "x": lattice[0], "y": lattice[1], "z": lattice[2], "t": lattice[3]}
    case["kappa"] = rng.choice([0.12, 0.124, 0.1245])
    case["isign"] = rng.choice([1, -1])
    case["prec"] = rng.choice(["f64", "f32", "f32", "f16", "bf16"])
    case["kind"] = rng.choice(["wilson", "clover", "clover", "tmwilson", "tmclover"])
    if path == "op":
        case["kind"] = rng.choice([case["kind"], case["kind"], "ndtmclover"])
    elif path == "dslash":
        case["kind"] = rng.choice(["wilson", "clover", "tmwilson", "tmclover"])
    elif path == "op_multi":
        case["nrhs"] = rng.choice([2, 3, 4, 6, 7, 8, 12, 13, 16])
    elif path == "clover_build":
        case["prec"] = rng.choice(["f64", "f32"])
        case.pop("kind")
    elif path == "cg":
        case["prec"] = rng.choice(["f64", "f64", "f32"])
        case["tol"] = 1e-10 if case["prec"] == "f64" else 1e-6
    elif path == "multishift":
        case["prec"] = "f64"
        case["nshift"] = rng.randrange(2, 13)
        case["tol"] = 1e-8
    elif path == "block_cg":
        case["prec"] = rng.choice(["f64", "f32", "f32"])
        case["nrhs"] = rng.randrange(2, 29)
        case["tol"] = 1e-8 if case["prec"] == "f64" else 1e-6
    elif path in ("mixed", "batch"):
        case["prec"] = rng.choice(["f16", "bf16"])
        case["kind"] = rng.choice(["clover", "tmclover"])
        case["tol"] = 1e-10
        if path == "batch":
            case["nrhs"] = rng.randrange(1, 5)
    case["c12"] = True if case["prec"] in ("f16", "bf16") else rng.random() < 0.5
    if case.get("kind") in ("tmwilson", "tmclover", "ndtmclover"):
        case["mu"] = round(rng.uniform(0.001, 0.01), 5)
    if case.get("kind") == "ndtmclover":
        case["eps"] = round(rng.uniform(0.001, 0.009), 5)
    return case


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _lattice(case):
    return [case["x"], case["y"], case["z"], case["t"]]


def _volume(lattice):
    return lattice[0] * lattice[1] * lattice[2] * lattice[3]


def _mass(case):
    return 1.0 / (2.0 * case["kappa"]) - 4.0


def _shifts(case):
    n = case["nshift"]
    return [10.0 ** (-4.0 + 4.0 * k / (n - 1)) for k in range(n)]


@functools.lru_cache(maxsize=8)
def _cb_sites(lattice):
    """Places of the two checkerboards' sites, in canonical order, in a [t][z][y][x] array."""
    nx, ny, nz, nt = lattice
    t, z, y, x = torch.meshgrid(*(torch.arange(n, device="cuda") for n in (nt, nz, ny, nx)), indexing="ij")
    odd = ((x + y + z + t) & 1).reshape(-1)
    return torch.nonzero(odd == 0).reshape(-1), torch.nonzero(odd == 1).reshape(-1)


def _mul3(a, b):
    """Products of 3x3 complex matrices, element by element of the leading axes."""
    return (a[..., :, 0, None] * b[..., None, 0, :] + a[..., :, 1, None] * b[..., None, 1, :]
            + a[..., :, 2, None] * b[..., None, 2, :])


def _links(lattice, rng):
    """U[mu] of shape [t, z, y, x, 3, 3]."""
    shape = (lattice[3], lattice[2], lattice[1], lattice[0], 3, 3)
    eye = torch.eye(3, dtype=torch.complex128, device="cuda")
    links = []
    for _ in range(4):
        g = torch.complex(torch.randn(shape, generator=rng, device="cuda", dtype=torch.float64),
                          torch.randn(shape, generator=rng, device="cuda", dtype=torch.float64))
        h = 0.5 * (g + g.mH)
        m = 0.4j * (h - eye * (h.diagonal(dim1=-2, dim2=-1).sum(-1) / 3.0)[..., None, None])
        u = eye + m / 16.0
        for n in range(15, 0, -1):  # exp by Horner's rule; the rows are made orthonormal below
            u = eye + _mul3(m / n, u)
        r0 = u[..., 0, :] / u[..., 0, :].abs().square().sum(-1, keepdim=True).sqrt()
        r1 = u[..., 1, :] - (r0.conj() * u[..., 1, :]).sum(-1, keepdim=True) * r0
        r1 = r1 / r1.abs().square().sum(-1, keepdim=True).sqrt()
        r2 = torch.linalg.cross(r0, r1, dim=-1).conj()
        links.append(torch.stack([r0, r1, r2], dim=-2))
    return links


def _source(vh, rng):
    """A Gaussian source of one checkerboard: [site, 4, 3]."""
    return torch.complex(torch.randn((vh, 4, 3), generator=rng, device="cuda", dtype=torch.float64),
                         torch.randn((vh, 4, 3), generator=rng, device="cuda", dtype=torch.float64))


def _sources(case, vh, rng):
    n = case.get("nrhs", 2 if case.get("kind") == "ndtmclover" else 1)
    got = []
    if case["path"] == "block_cg":  # up to 12 point sources, one for each spin and colour of a site
        site = int(torch.randint(vh, (1,), generator=rng, device="cuda"))
        for k in range(min(12, n // 2)):
            p = torch.zeros((vh, 12), dtype=torch.complex128, device="cuda")
            p[site, k] = 1.0
            got.append(p.reshape(vh, 4, 3))
    return got + [_source(vh, rng) for _ in range(n - len(got))]


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _host(x):
    return torch.view_as_real(x.contiguous()).reshape(-1).cpu().numpy()


def _canonical_links(links, lattice):
    sites = torch.cat(_cb_sites(tuple(lattice)))
    return _host(torch.stack([u.reshape(-1, 3, 3)[sites] for u in links], dim=1))


def _fields(lattice, case, seed):
    """(FP64 geometry, its links, the sources on the odd checkerboard) of one lattice."""
    g64 = q.Geometry(lattice, q.F64, False)
    if _volume(lattice) <= PACKED_VOLUME:
        rng = _generator(seed)
        u = q.pack_gauge(g64, _canonical_links(_links(lattice, rng), lattice))
        b = [g64.spinor().upload(_host(s), 1) for s in _sources(case, g64.vh, rng)]
    else:
        u = q.gen_gauge(g64, seed)
        b = [q.gen_spinor(g64, seed + 1 + k, 1) for k in range(case.get("nrhs", 1))]
    return g64, u, b


def _spinors_of(g, g64, fields):
    if g.prec == q.F64:
        return fields
    got = []
    for f in fields:
        got.append(g.spinor())
        q.convert_spinor(g, got[-1], 1.0, g64, f)
    return got


class _Terms:
    """The fields of one operator kind in the precision of `g`, made from FP64 links."""

    def __init__(self, case, kind, g, g64, u64, made=None):
        self.u = u64 if g.prec == q.F64 and not g.compress12 else q.convert_gauge(g, g64, u64)
        self.clov = self.invclov = self.full = self.offd = None
        mass, mu, eps = _mass(case), case.get("mu", 0.0), case.get("eps", 0.0)
        made = {} if made is None else made

        def term(cb, what, *, full=False, **kw):
            key = (cb, what, tuple(kw.values()))
            if key not in made:
                made[key] = q.clover_build(g64, u64, CSW, mass, cb, what, **kw)
            return made[key] if g.prec == q.F64 else q.convert_clover(g, g64, made[key], full=full)

        if kind in ("clover", "tmclover", "ndtmclover"):
            self.clov = [None, term(1, q.CLOV_A)]
        if kind == "clover":
            self.invclov = [term(0, q.CLOV_AINV), None]
        elif kind == "tmclover":
            self.full = [[term(0, q.CLOV_TMINV, full=True, mu=s * mu) for s in (1.0, -1.0)], None]
        elif kind == "ndtmclover":
            self.full = [[term(0, w, full=True, mu=mu, eps=eps) for w in (q.CLOV_ND_UP, q.CLOV_ND_DN)], None]
            self.offd = [term(0, q.CLOV_ND_OFF, mu=mu, eps=eps), None]
        self.made = made

    def operator(self, case, kind, g):
        mu = case.get("mu", 0.0)
        return q.Operator(g, KINDS[kind], self.u, mass=_mass(case), twisted_mass=mu, epsilon=case.get("eps", 0.0),
                          prec_mass_rho=mu if kind == "tmclover" else 0.0, t_boundary=-1.0, clov=self.clov,
                          invclov=self.invclov, fullclov=self.full, clov_odiag=self.offd)


class _DeviceBytes:
    """A library field's device memory, for torch."""

    def __init__(self, field, nbytes):
        self.field = field
        self.__cuda_array_interface__ = {"shape": (nbytes,), "typestr": "|u1", "data": (field.p.value, False),
                                         "version": 2, "strides": None}


def _stored(field, prec):
    """What a field holds, in place: its values, and the per-site scales of a half precision."""
    g = field.geom
    nbytes = g.bytes[0] if field.kind == "spinor" else g.bytes[2]
    raw = torch.as_tensor(_DeviceBytes(field, nbytes), device="cuda")
    if prec in ("f64", "f32"):
        return raw.view(STORED[prec])
    reals = 24 if field.kind == "spinor" else 72
    padded = nbytes // (2 * reals + 4)
    return {"values": raw[:2 * reals * padded].view(STORED[prec]), "scales": raw[2 * reals * padded:].view(torch.float32)}


class _State:
    pass


def _prepare_batch(case, seed):
    s = _State()
    s.case, s.keep = case, []
    inner, s.outer, s.b, s.x = [], [], [], []
    lattices = BATCH if _lattice(case) == list(BATCH[-1]) else ((8, 8, 8, 8), tuple(_lattice(case)))
    mus = torch.rand(len(lattices), generator=torch.Generator().manual_seed(seed), dtype=torch.float64)
    for i, lattice in enumerate(lattices):
        c = dict(case, mu=0.001 + 0.009 * float(mus[i]))
        g64, u, b = _fields(list(lattice), c, seed + 1000 * (i + 1))
        gi = q.Geometry(lattice, PRECS[case["prec"]], True)
        outer_terms = _Terms(c, case["kind"], g64, g64, u)
        inner_terms = _Terms(c, case["kind"], gi, g64, u, outer_terms.made)
        mo, mi = outer_terms.operator(c, case["kind"], g64), inner_terms.operator(c, case["kind"], gi)
        s.keep += [g64, gi, outer_terms, inner_terms]
        for f in b:
            s.outer.append(mo)
            inner.append(mi)
            s.b.append(f)
            s.x.append(g64.spinor())
    s.batch = q.Batch(inner)
    s.out = [_stored(x, "f64") for x in s.x]
    return s


def prepare(case, seed):
    path = case["path"]
    if path == "batch":
        return _prepare_batch(case, seed)
    s = _State()
    s.case = case
    prec, lattice = case["prec"], _lattice(case)
    g64, u64, b64 = _fields(lattice, dict(case, nrhs=0) if path == "clover_build" else case, seed)
    g = g64 if prec == "f64" and not case["c12"] else q.Geometry(lattice, PRECS[prec], case["c12"])
    s.g, s.g64 = g, g64
    if path == "clover_build":
        s.u = u64 if g is g64 else q.convert_gauge(g, g64, u64)
        s.inverse = g.clover()  # rebuilt in place, as a program with a field for it does
        s.out = _stored(s.inverse, prec)
        q.sync()
        return s
    kind = case["kind"]
    s.terms = _Terms(case, kind, g, g64, u64)
    if path == "dslash":
        s.hop = q.Dslash(g, t_boundary=-1.0, mass=_mass(case), twisted_mass=case.get("mu", 0.0))
    else:
        s.op = s.terms.operator(case, kind, g)
    if path == "mixed":
        s.outer_terms = _Terms(case, kind, g64, g64, u64, s.terms.made)
        s.outer = s.outer_terms.operator(case, kind, g64)
        s.inner = q.InvBiCGStab(s.op, 5000)
        s.solver = q.InvRichardsonMultiPrec(s.outer, s.inner, 1e-2, 200)
        s.b, s.x = b64, [g64.spinor()]
        s.out = [_stored(x, "f64") for x in s.x]
    else:
        s.b = _spinors_of(g, g64, b64)
        s.x = [g.spinor() for _ in range(case.get("nshift", len(s.b)))]
        s.out = [_stored(x, prec) for x in s.x]
    if path == "cg":
        s.solver = q.InvCG(s.op, 5000)
    elif path == "block_cg":
        s.solver = q.InvBlockCG(s.op, 5000)
    elif path == "multishift":
        s.shifts = _shifts(case)
        s.solver = q.MInvCG(s.op, 5000, len(s.shifts))
    s.terms.made = None  # the operators keep the fields they use
    q.sync()
    return s


def run(s):
    c = s.case
    path = c["path"]
    if path == "op":
        s.op(s.x, s.b, c["isign"], 1)
        return s.out
    if path == "op_multi":
        s.op.apply_multi(s.x, s.b, c["isign"], 1)
        return s.out
    if path == "dslash":
        x, b, u, kind = s.x[0], s.b[0], s.terms.u[0], c["kind"]
        if kind == "wilson":
            s.hop.dslash(x, b, u, c["isign"], 0)
        elif kind == "clover":
            s.hop.clov_dslash(x, b, u, s.terms.invclov[0], c["isign"], 0)
        elif kind == "tmwilson":
            s.hop.tm_dslash(x, b, u, c["isign"], 0)
        else:
            s.hop.tmclov_dslash(x, b, u, s.terms.full[0], c["isign"], 0)
        return s.out
    if path == "clover_build":
        csw = ctypes.c_double(CSW)
        q.call("qphix_clover_build", s.g.h, s.u[0].p, s.u[1].p, csw, csw, ctypes.c_double(4.0 + _mass(c)), 0,
               q.CLOV_AINV, ctypes.c_double(0.0), ctypes.c_double(0.0), s.inverse.p)
        return s.out
    for x in s.x:  # every solve starts from zero
        q.zero(x.geom, x)
    if path == "cg" or path == "mixed":
        s.solver(s.x, s.b, c["tol"], c["isign"], 1)
    elif path == "multishift":
        s.solver(s.x, s.b[0], s.shifts, [c["tol"]] * len(s.shifts), c["isign"], 1)
    elif path == "block_cg":
        s.solver.solve_multi(s.x, s.b, c["tol"], c["isign"], 1)
    else:
        s.batch.richardson(s.outer, s.x, s.b, c["tol"], delta=1e-2, isign=c["isign"], graph_steps=8)
    return s.out


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
# site values of the clover-type factor of (A^-1 D, A chi - D psi) and floating-point operations of the two hops
_CLOVER_REALS = {"wilson": (0, 0), "tmwilson": (0, 0), "clover": (72, 72), "tmclover": (144, 72), "ndtmclover": (360, 72)}
_CLOVER_FLOPS = {"wilson": (0, 24), "tmwilson": (72, 96), "clover": (504, 552), "tmclover": (552, 600),
                 "ndtmclover": (2 * 1080, 2 * 648)}
# operator applications of a solve to its tolerance (measured; M and M^+ count as one each)
_APPLICATIONS = {"cg": 84, "multishift": 82, "block_cg": 62, "mixed": 48, "batch": 130}


def _op_work(case, kind, prec, c12, nrhs, halves=2):
    """Bytes and operations of an even-odd operator (halves = 1: of its first hop alone) on nrhs sources."""
    vh = _volume(_lattice(case)) // 2
    scales = 4 if prec in ("f16", "bf16") else 0
    real = REAL_BYTES[prec]
    links = (96 if c12 else 144) * real + scales
    spinor = 24 * real + scales
    flav = 2 if kind == "ndtmclover" else 1
    nbytes = flops = 0
    for h in range(halves):
        n = _CLOVER_REALS[kind][h]
        # the source is read once for the operator and its result written once
        nbytes += links + n * real + (scales if n else 0)
        flops += nrhs * (flav * 1320 + _CLOVER_FLOPS[kind][h])
    nbytes += 2 * flav * nrhs * spinor
    return {"bytes": vh * nbytes, "flops": vh * flops}


def work(case):
    path, prec = case["path"], case["prec"]
    vh = _volume(_lattice(case)) // 2
    if path == "clover_build":
        real = REAL_BYTES[prec]
        links = 4 * 2 * (12 if case["c12"] else 18) * real
        # six planes of four leaves: 13 products of 3x3 matrices a plane, and a 6x6 inverse per block
        return {"bytes": vh * (links + 72 * real), "flops": vh * (6 * 13 * 198 + 2 * 1100)}
    kind = case["kind"]
    if path == "op":
        return _op_work(case, kind, prec, case["c12"], 1)
    if path == "dslash":
        return _op_work(case, kind, prec, case["c12"], 1, halves=1)
    if path == "op_multi":
        return _op_work(case, kind, prec, case["c12"], case["nrhs"])
    n = _APPLICATIONS[path]
    nrhs = case.get("nrhs", 1)
    if path == "batch":
        lattices = BATCH if _lattice(case) == list(BATCH[-1]) else ((8, 8, 8, 8), tuple(_lattice(case)))
        w = [_op_work(dict(case, x=a, y=b, z=c, t=d), kind, prec, True, nrhs) for a, b, c, d in lattices]
        w = {k: sum(v[k] for v in w) for k in ("bytes", "flops")}
    else:
        w = _op_work(case, kind, prec, case["c12"], nrhs)
    more = 0
    if path == "multishift":  # p and x of each shift, read and written once an iteration
        more = vh * (n // 2) * case["nshift"] * 4 * 24 * 8
    elif path == "block_cg":  # P, Z and Q through the products of an iteration
        w["flops"] += vh * 12 * 8 * nrhs * nrhs * 6
    return {"bytes": n * w["bytes"] + more, "flops": n * w["flops"]}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _gammas():
    """DeGrand-Rossi: rows of (column, phase)."""
    rows = [[(3, 1j), (2, 1j), (1, -1j), (0, -1j)], [(3, -1), (2, 1), (1, 1), (0, -1)],
            [(2, 1j), (3, -1j), (0, -1j), (1, 1j)], [(2, 1), (3, 1), (0, 1), (1, 1)]]
    g = torch.zeros((4, 4, 4), dtype=torch.complex128)
    for mu in range(4):
        for row, (col, phase) in enumerate(rows[mu]):
            g[mu, row, col] = phase
    return g.cuda()


def _spin(m, psi):
    """A 4x4 spin matrix times [..., 4, 3]."""
    return sum(m[:, k, None] * psi[..., k, None, :] for k in range(4))


def _colour(u, psi, dagger=False):
    """Links times [..., 4, 3]."""
    u = u.conj() if dagger else u
    return sum((u[..., k, :] if dagger else u[..., :, k])[..., None, :] * psi[..., :, k, None] for k in range(3))


class _Exact:
    """The operators of one lattice on [t, z, y, x] arrays in complex128."""

    def __init__(self, lattice, links):
        self.lattice, self.links = tuple(lattice), links
        self.gamma, self.one = _gammas(), torch.eye(4, dtype=torch.complex128, device="cuda")
        self.axis = [3, 2, 1, 0]  # of x, y, z, t
        self.clover = {}

    def full(self, v, cb):
        nx, ny, nz, nt = self.lattice
        f = torch.zeros((nt * nz * ny * nx,) + tuple(v.shape[1:]), dtype=v.dtype, device="cuda")
        f[_cb_sites(self.lattice)[cb]] = v
        return f.reshape((nt, nz, ny, nx) + tuple(v.shape[1:]))

    def half(self, f, cb):
        return f.reshape((-1,) + tuple(f.shape[4:]))[_cb_sites(self.lattice)[cb]]

    def hop(self, psi, cb, isign):
        """D psi on checkerboard cb, antiperiodic in t."""
        psi = self.full(psi, 1 - cb)
        out = torch.zeros_like(psi)
        for mu in range(4):
            ax = self.axis[mu]
            fwd = psi.roll(-1, ax)
            if mu == 3:
                fwd[-1] = -fwd[-1]
            out += _colour(self.links[mu], _spin(self.one - isign * self.gamma[mu], fwd))
            back = _colour(self.links[mu], _spin(self.one + isign * self.gamma[mu], psi), dagger=True).roll(1, ax)
            if mu == 3:
                back[0] = -back[0]
            out += back
        return self.half(out, cb)

    def strength(self, mu, nu):
        a, b, um, un = self.axis[mu], self.axis[nu], self.links[mu], self.links[nu]
        p = _mul3(_mul3(um, un.roll(-1, a)), _mul3(un, um.roll(-1, b)).mH)  # the plaquette at x
        # the other three leaves at x are the same loop of the neighbouring plaquettes, begun at x
        u2 = _mul3(_mul3(un, um.roll((1, -1), (a, b)).mH), _mul3(un.roll(1, a).mH, um.roll(1, a)))
        u3 = _mul3(_mul3(un.roll((1, 1), (a, b)), um.roll(1, a)).mH, _mul3(um.roll((1, 1), (a, b)), un.roll(1, b)))
        u4 = _mul3(_mul3(un.roll(1, b).mH, um.roll(1, b)), _mul3(un.roll((-1, 1), (a, b)), um.mH))
        s = p + u2 + u3 + u4
        return 0.125 * (s - s.mH)

    def blocks(self, cb, mass):
        """The clover term of checkerboard cb: [site, 2, 6, 6]."""
        if cb not in self.clover:
            n = _volume(self.lattice) // 2
            a = (4.0 + mass) * torch.eye(12, dtype=torch.complex128, device="cuda").reshape(4, 3, 4, 3)
            a = a.expand(n, 4, 3, 4, 3).clone()
            for mu in range(4):
                for nu in range(mu + 1, 4):
                    sigma = 0.5 * (self.gamma[mu] @ self.gamma[nu] - self.gamma[nu] @ self.gamma[mu])
                    f = self.half(self.strength(mu, nu), cb)
                    a -= 0.5 * CSW * sigma[None, :, None, :, None] * f[:, None, :, None, :]
            self.clover[cb] = torch.stack([a[:, :2, :, :2].reshape(n, 6, 6), a[:, 2:, :, 2:].reshape(n, 6, 6)], dim=1)
        return self.clover[cb]


def _inverse(m):
    """Inverses of [..., 6, 6] by elimination (the blocks are far from singular)."""
    n = m.shape[-1]
    a = torch.cat([m, torch.eye(n, dtype=m.dtype, device=m.device).expand(m.shape)], dim=-1)
    for k in range(n):
        row = a[..., k, :] / a[..., k, k, None]
        col = a[..., :, k].clone()
        col[..., k] = 0.0
        a = a - col[..., :, None] * row[..., None, :]
        a[..., k, :] = row
    return a[..., n:]


def _apply6(m, psi):
    """Blocks [site, 2, 6, 6] times [site, 4, 3]."""
    v = psi.reshape(-1, 2, 6)
    return sum(m[..., k] * v[..., k, None] for k in range(6)).reshape(psi.shape)


def _g5():
    return torch.tensor([1.0, 1.0, -1.0, -1.0], dtype=torch.float64, device="cuda")[:, None]


def _mul6(a, b):
    return sum(a[..., :, k, None] * b[..., None, k, :] for k in range(6))


class _ExactOp:
    """An even-odd operator on the odd checkerboard; sources and results are lists over flavours."""

    def __init__(self, case, links, lattice=None):
        self.e = _Exact(lattice or _lattice(case), links)
        self.case, self.kind, self.mass = case, case["kind"], _mass(case)
        self.mu, self.eps = case.get("mu", 0.0), case.get("eps", 0.0)
        self.kept = {}

    def _inner(self, key):
        if key not in self.kept:
            a = self.e.blocks(0, self.mass)
            eye = torch.eye(6, dtype=torch.complex128, device="cuda")
            tw = 1j * torch.tensor([1.0, -1.0], dtype=torch.float64, device="cuda")[:, None, None] * self.mu * eye
            if key == "inverse":
                self.kept[key] = _inverse(a)
            elif key in (1, -1):
                self.kept[key] = _inverse(a + key * tw)
            else:
                n = _inverse(_mul6(a, a) + (self.mu ** 2 - self.eps ** 2) * eye)
                self.kept["up"], self.kept["dn"] = _mul6(n, a - tw), _mul6(n, a + tw)
                self.kept["off"] = self.eps * n
        return self.kept[key]

    def inner(self, psi, isign):
        """The first half: the even checkerboard's factor times D psi."""
        d = [self.e.hop(p, 0, isign) for p in psi]
        if self.kind == "wilson":
            return d
        if self.kind == "tmwilson":
            al = 4.0 + self.mass
            return [(al * v - 1j * isign * self.mu * _g5() * v) / (al * al + self.mu * self.mu) for v in d]
        if self.kind == "clover":
            return [_apply6(self._inner("inverse"), v) for v in d]
        if self.kind == "tmclover":
            return [_apply6(self._inner(isign), v) for v in d]
        up, dn, off = self._inner("up"), self._inner("dn"), self._inner("off")
        up, dn = (up, dn) if isign == 1 else (dn, up)
        return [_apply6(up, d[0]) + _apply6(off, d[1]), _apply6(dn, d[1]) + _apply6(off, d[0])]

    def __call__(self, psi, isign):
        al = 4.0 + self.mass
        back = [self.e.hop(v, 1, isign) for v in self.inner(psi, isign)]
        if self.kind == "wilson":
            return [al * p - (0.25 / al) * v for p, v in zip(psi, back)]
        if self.kind == "tmwilson":
            return [al * p + 1j * isign * self.mu * _g5() * p - 0.25 * v for p, v in zip(psi, back)]
        got = []
        for f, (p, v) in enumerate(zip(psi, back)):
            r = _apply6(self.e.blocks(1, self.mass), p) - 0.25 * v
            if self.kind != "clover":
                r = r + 1j * isign * (1.0 - 2.0 * f) * self.mu * _g5() * p
            if self.kind == "ndtmclover":
                r = r - self.eps * psi[1 - f]
            got.append(r)
        return got

    def normal(self, p, isign, shift=0.0):
        return self(self([p], isign), -isign)[0] + shift * p

    def solve(self, b, isign, shift=0.0, tol=1e-14):
        """(M^+M + shift) x = b by CG."""
        x, r, p = torch.zeros_like(b), b.clone(), b.clone()
        c = first = float(b.abs().square().sum())
        for _ in range(500):
            ap = self.normal(p, isign, shift)
            a = c / float((p.conj() * ap).sum().real)
            x += a * p
            r -= a * ap
            new = float(r.abs().square().sum())
            if new <= tol * tol * first:
                break
            p = r + (new / c) * p
            c = new
        return x


def _as_stored(v, prec):
    """[site, reals] as a field holds them."""
    n, reals = v.shape
    padded = -(-n // SITE_BLOCK) * SITE_BLOCK
    word = 16 // REAL_BYTES[prec]
    scales = None
    if prec in ("f16", "bf16"):
        top = v.abs().amax(dim=1)
        scales = torch.zeros(padded, dtype=torch.float64, device="cuda")
        scales[:n] = top
        v = v / torch.where(top > 0, top, 1.0)[:, None]
    full = torch.zeros((padded, reals), dtype=torch.float64, device="cuda")
    full[:n] = v
    full = full.reshape(-1, SITE_BLOCK, reals // word, word).transpose(1, 2).reshape(-1)
    return full if scales is None else {"values": full, "scales": scales}


def _spinor_as_stored(psi, prec):
    return _as_stored(torch.view_as_real(psi).reshape(-1, 24), prec)


def exact(case, seed):
    path, lattice = case["path"], _lattice(case)
    volume = _volume(lattice)
    if path == "batch" or volume > PACKED_VOLUME:
        return None
    rng = _generator(seed)
    links = _links(lattice, rng)
    vh = volume // 2
    if path == "clover_build":
        m = _inverse(_Exact(lattice, links).blocks(0, _mass(case)))
        low = [(i, j) for i in range(6) for j in range(i)]
        diag = torch.stack([m[..., i, i].real for i in range(6)], dim=-1)
        offd = torch.view_as_real(torch.stack([m[..., i, j] for i, j in low], dim=-1)).reshape(vh, 2, 30)
        return _as_stored(torch.cat([diag, offd], dim=-1).reshape(vh, 72), case["prec"])
    b = _sources(case, vh, rng)
    op, isign = _ExactOp(case, links), case["isign"]
    if path == "op":
        return [_spinor_as_stored(v, case["prec"]) for v in op(b, isign)]
    if path == "dslash":
        return [_spinor_as_stored(v, case["prec"]) for v in op.inner(b, isign)]
    if path == "op_multi":
        return [_spinor_as_stored(op([v], isign)[0], case["prec"]) for v in b]
    if volume > 1 << 17:
        return None
    if path == "cg":
        return [_spinor_as_stored(op.solve(b[0], isign), case["prec"])]
    if path == "multishift":
        return [_spinor_as_stored(op.solve(b[0], isign, sh), "f64") if k % 4 == 0 else None
                for k, sh in enumerate(_shifts(case))]
    if path == "block_cg":  # the first point source and the last Gaussian one stand for the others
        return [_spinor_as_stored(op.solve(v, isign), case["prec"]) if k in (0, len(b) - 1) else None
                for k, v in enumerate(b)]
    # mixed: M x = b through the normal equations
    return [_spinor_as_stored(op.solve(op(b, -isign)[0], isign), "f64")]
