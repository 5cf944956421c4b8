"""The work that a program gives this framework, as measured cases.

Each case is one call sequence through the public interface (`ch_swe_amd`):
the tendency of a state, RK4 integrations (small, ordinary, large, odd sizes,
both precisions, compensated, all three SBP orders), an ensemble, an uneven
batch, Crank-Nicolson steps with the conjugate-gradient solve, the
diagnostics of a run, and served requests.  `prepare` builds what such a
program holds (operator, device states with their initial fields), `run` is
one pass and returns the fields that the program reads back, `exact` is the
same computation in 64 bits with dense one-dimensional SBP matrices in plain
torch.  Fields of single-precision plans are returned as float32 (the values
the device holds); `download` hands them over as float64.
"""
import math

import numpy as np
import torch

import ch_swe_amd as cs

RADIUS, GRAV, DEPTH, OMEGA = 6.371e6, 9.81, 1000.0, 7.292e-5
DIAG_GRAV = 9.80616  # the gravity that the diagnostics are printed with


def listed():
    return [
        # the smallest call: one tendency on the grid of the Gaussian-hill
        # runs, read back (a host program stepping with its own scheme)
        dict(name="tendency N=32", kind="apply", N=32, order=21, fp32=False),
        # the Gaussian-hill configuration: N=32, sbp21, FP64, dt = 600 s, 100
        # steps; launches and latency count
        dict(name="rk4 N=32 sbp21 fp64", kind="rk4", N=32, order=21, fp32=False, steps=100, comp=False),
        # an ordinary single run in double precision
        dict(name="rk4 N=96 sbp42 fp64", kind="rk4", N=96, order=42, fp32=False, steps=200, comp=False),
        # an odd size in single precision with the compensated update
        dict(name="rk4 N=191 compensated", kind="rk4", N=191, order=42, fp32=True, steps=200, comp=True),
        # the large solve in both precisions (the benchmark's default workload)
        dict(name="rk4 N=384 sbp42 fp32", kind="rk4", N=384, order=42, fp32=True, steps=400, comp=False),
        dict(name="rk4 N=384 sbp42 fp64", kind="rk4", N=384, order=42, fp32=False, steps=200, comp=False),
        # the sixth-order operators (the paper's third convergence curve)
        dict(name="rk4 N=96 sbp63 fp64", kind="rk4", N=96, order=63, fp32=False, steps=64, comp=False),
        # a uniform ensemble: every member's steps in shared launches
        dict(name="ensemble 16 x N=96", kind="ensemble", N=96, order=42, fp32=True, steps=100, members=16),
        # an uneven batch: N in {24, 48, 96, 192}, sbp21 and sbp42, own dt and
        # step counts
        dict(name="uneven batch of 16", kind="uneven", N=192, odd=0, fp32=True, steps=120, members=16),
        # implicit time stepping: two Crank-Nicolson steps at CFL 4
        dict(name="crank-nicolson N=96", kind="implicit", N=96, order=42, fp32=False, steps=2),
        # the sums and Courant numbers of a diagnostics step (its tendencies
        # are left out: sums that cancel to a thousand-millionth of their
        # terms have no digits to compare)
        dict(name="diagnostics N=192", kind="diag", N=192, order=42),
        # requests of mixed size and precision through the server
        dict(name="serving 8 requests", kind="serve", N=96, odd=0, steps=50, requests=8),
    ]


def draw(rng):
    """One more case of the same ranges."""
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["apply", "rk4", "rk4", "rk4", "rk4", "ensemble", "uneven", "implicit", "diag", "serve"])
    order, fp32 = rng.choice([21, 42, 42]), rng.random() < 0.5
    if kind == "apply":
        return dict(kind=kind, N=size(16, 256), order=rng.choice([21, 42, 63]), fp32=fp32)
    if kind == "rk4":
        order = rng.choice([21, 42, 42, 63])
        N = size(24, 192 if order == 63 else 384)
        return dict(kind=kind, N=N, order=order, fp32=fp32, steps=rng.randint(40, 100) if order == 63 else
                    rng.randint(100, 200), comp=order != 63 and rng.random() < 0.25)
    if kind == "ensemble":
        return dict(kind=kind, N=size(32, 112), order=order, fp32=fp32, steps=rng.randint(40, 100),
                    members=rng.randint(4, 16))
    if kind == "uneven":
        return dict(kind=kind, N=size(96, 192), odd=rng.randint(0, 1), fp32=fp32, steps=rng.randint(40, 100),
                    members=rng.randint(6, 16))
    if kind == "implicit":
        return dict(kind=kind, N=size(24, 192), order=rng.choice([21, 42]), fp32=False, steps=rng.randint(1, 2))
    if kind == "diag":
        return dict(kind=kind, N=size(32, 384), order=order)
    return dict(kind=kind, N=size(48, 112), odd=rng.randint(0, 1), steps=rng.randint(25, 60),
                requests=rng.randint(4, 10))


def _time_step(N, courant):
    return courant * RADIUS * (0.5 * math.pi / N) / math.sqrt(GRAV * DEPTH)


def _solves(case):
    """The solves of a case: (N, order, fp32, dt, steps) each."""
    kind = case["kind"]
    if kind == "rk4":
        dt = 600.0 if case["N"] == 32 and case["order"] == 21 else _time_step(case["N"], 0.5)
        return [(case["N"], case["order"], case["fp32"], dt, case["steps"])]
    if kind == "ensemble":
        return [(case["N"], case["order"], case["fp32"], _time_step(case["N"], 0.5), case["steps"])] * case["members"]
    out = []
    for k in range(case["members"] if kind == "uneven" else case["requests"]):
        N = max(12, case["N"] // 2 ** (k % 4 if kind == "uneven" else k % 3)) + case["odd"] * (k % 3)
        order = 21 if (k // 4) % 2 else 42
        fp32 = case["fp32"] if kind == "uneven" else k % 2 == 0
        steps = max(2, case["steps"] * (4 + (7 * k) % 13) // 16)
        out.append((N, order, fp32, _time_step(N, 0.3 + 0.05 * (k % 5)), steps))
    return out


# ---- fields ---------------------------------------------------------------------
# panel frames of the cubed sphere: directions of increasing i and j, inward
# normal
_EX = [[-1, 0, 0], [0, 0, -1], [1, 0, 0], [0, 0, 1], [1, 0, 0], [1, 0, 0]]
_EY = [[0, 1, 0], [0, 1, 0], [0, 1, 0], [0, 1, 0], [0, 0, 1], [0, 0, -1]]
_NN = [[0, 0, 1], [-1, 0, 0], [0, 0, -1], [1, 0, 0], [0, 1, 0], [0, -1, 0]]


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _mesh(N, xt, yt):
    """X = tan(alpha), Y = tan(beta) of a mesh (xt / yt: at the cell centres
    along x / y), shape [ny, nx]."""
    hx = 0.5 * math.pi / N
    x, y = (torch.tan(-0.25 * math.pi + hx * (torch.arange(N if t else N + 1, dtype=torch.float64, device=_device())
                                              + 0.5 * t)) for t in (xt, yt))
    return x[None, :].expand(len(y), -1), y[:, None].expand(-1, len(x))


def _to_panels(a, b, c):
    """Prototype-face components [ny, nx] as vectors [6, ny, nx, 3]."""
    ex, ey, nn = (torch.tensor(m, dtype=torch.float64, device=_device())[:, None, None, :] for m in (_EX, _EY, _NN))
    return a[None, ..., None] * ex + b[None, ..., None] * ey - c[None, ..., None] * nn


def _fields(N, seed, depth=0.0):
    """(u, v, h) on the device in 64 bits: hills and hollows of up to 20 m
    with widths of 600 to 4000 km, and the non-divergent wind of a stream
    function of the same kind (a few m/s), as covariant components."""
    rng = np.random.default_rng(seed)
    k = 6
    cen = rng.standard_normal((2, k, 3))
    cen = torch.tensor(cen / np.linalg.norm(cen, axis=2, keepdims=True), device=_device())
    sharp = (RADIUS / rng.uniform(6e5, 4e6, (2, k))) ** 2
    amp = rng.uniform(-20.0, 20.0, (2, k))
    out = []
    for m, (xt, yt) in enumerate(((1, 0), (0, 1), (0, 0))):
        X, Y = _mesh(N, xt, yt)
        s2 = 1 + X * X + Y * Y
        s = torch.sqrt(s2)
        r = _to_panels(X / s, Y / s, 1 / s)
        if m == 2:
            f = sum(amp[0, q] * torch.exp(sharp[0, q] * (r @ cen[0, q] - 1)) for q in range(k))
            out.append(f + depth)
            continue
        cx, cy, s3 = 1 + X * X, 1 + Y * Y, s2 * s
        a = (_to_panels(cx * cy / s3, -X * Y * cx / s3, -X * cx / s3) if m == 0 else
             _to_panels(-X * Y * cy / s3, cx * cy / s3, -Y * cy / s3))
        # V = r x grad psi, psi = sum b exp(k (r.c - 1)) / sqrt(k)
        g = sum(0.25 * amp[1, q] * math.sqrt(sharp[1, q]) * torch.exp(sharp[1, q] * (r @ cen[1, q] - 1))[..., None]
                * cen[1, q] for q in range(k))
        out.append((torch.linalg.cross(r, g) * a).sum(-1))
    return out


def _host(fields):
    return [np.ascontiguousarray(f.cpu().numpy()) for f in fields]


def _operator(N, order, fp32, **kw):
    return cs.create_linear_swm_operator(N, order, cs.FP32 if fp32 else cs.FP64, grav=GRAV, h_mean=DEPTH,
                                         radius=RADIUS, omega=OMEGA, **kw)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("ensemble", "uneven"):
        ops, start, work, solves = {}, [], [], _solves(case)
        for k, (N, order, fp32, _, _) in enumerate(solves):
            if (N, order) not in ops:
                ops[N, order] = _operator(N, order, fp32)
            start.append(ops[N, order].create_stvec().upload(*_host(_fields(N, 1000 * seed + k))))
            work.append(start[-1].create_similar())
        return dict(case=case, solves=solves, start=start, work=work, ens=cs.Ensemble(work))
    if kind == "serve":
        solves = _solves(case)
        return dict(case=case, solves=solves, server=cs.Server(16 << 30),
                    fields=[_host(_fields(s[0], 1000 * seed + k)) for k, s in enumerate(solves)])
    if kind == "diag":
        op = _operator(case["N"], case["order"], False)
        return dict(case=case, op=op, start=op.create_stvec().upload(*_host(_fields(case["N"], seed, DEPTH))))
    op = _operator(case["N"], case["order"], case["fp32"], compensated=case.get("comp", False))
    start = op.create_stvec().upload(*_host(_fields(case["N"], seed)))
    scheme = (None if kind == "apply" else cs.create_timescheme("rk4") if kind == "rk4" else
              cs.create_timescheme("crank_nikolson", rel_tol=1e-10, max_iter=200))
    return dict(case=case, op=op, start=start, work=op.create_stvec(), scheme=scheme)


def _read(arrays, fp32):
    """Downloaded fields; float32 where the device holds single precision."""
    return [torch.from_numpy(a).to(torch.float32) for a in arrays] if fp32 else list(arrays)


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind in ("ensemble", "uneven"):
        # the members restart from their initial states, advance together
        # and are read back
        for s, w in zip(state["start"], state["work"]):
            w.assign(1.0, s)
        state["ens"].rk4([s[3] for s in state["solves"]], [s[4] for s in state["solves"]], graph=True)
        return [_read(w.download(), s[2]) for w, s in zip(state["work"], state["solves"])]
    if kind == "serve":
        srv = state["server"]
        ids = [srv.submit(*f, s[3], s[4], s[0], s[1], cs.FP32 if s[2] else cs.FP64, grav=GRAV, h_mean=DEPTH,
                          radius=RADIUS, omega=OMEGA) for f, s in zip(state["fields"], state["solves"])]
        got = [None] * len(ids)
        while any(g is None for g in got):
            srv.tick(25)
            for k, rid in enumerate(ids):
                if got[k] is None:
                    got[k] = srv.take(rid)
            srv.wait()
        return [_read(g, s[2]) for g, s in zip(got, state["solves"])]
    op = state["op"]
    if kind == "diag":
        st, dt = state["start"], _time_step(case["N"], 0.5)
        return [list(op.integrals(st)), op.integrals_diag(st, DIAG_GRAV), op.cfl_diag(st, dt, DIAG_GRAV)]
    w = state["work"]
    if kind == "apply":
        op.apply(w, state["start"])
        return _read(w.download(), case["fp32"])
    w.assign(1.0, state["start"])
    if kind == "rk4":
        state["scheme"].step(w, op, _solves(case)[0][3], case["steps"])
    else:
        state["scheme"].step(w, op, _time_step(case["N"], 4.0), case["steps"])
    return _read(w.download(), case["fp32"])


def work(case):
    """Bytes: every operator application reads a state and the nine metric
    coefficients (eight of them common to the panels) and writes a state;
    fields leave the device once.  Flops: about 130 per grid point and
    application (twelve four-point stencils and the metric products)."""
    def app(N, size):
        return 6 * (N + 1) * (3 * N + 1) * size * 2 + (8 + 6) * (N + 1) ** 2 * size

    kind = case["kind"]
    if kind in ("apply", "diag", "implicit"):
        N, size = case["N"], 4 if case.get("fp32") else 8
        count = {"apply": 1, "diag": 1, "implicit": 2 * 70 * case.get("steps", 1)}[kind]
        return dict(bytes=count * app(N, size), flops=130 * 6 * N * N * count)
    bytes_ = flops = 0
    for N, _, fp32, _, steps in _solves(case):
        bytes_ += 4 * steps * app(N, 4 if fp32 else 8)
        flops += 4 * steps * 130 * 6 * N * N
    return dict(bytes=bytes_, flops=flops)


# ---- the same computation in 64 bits, without the framework ---------------------
_C13, _C14 = 0.1264926207034815, -0.029892648949074313
# closure rows (first points of a line; mirrored at its end), interior
# stencil (symmetric or antisymmetric half, nearest first), SAT projection
# and boundary norm weights of the centre and interface points
_SBP = {
    21: dict(di=[], dc=[[-1, 1]], ii=[], ic=[[1]], dq=[1], iq=[0.5], R=[1.5, -0.5], hc=[1, 1], hi=[0.5]),
    42: dict(
        di=[[-79 / 78, 27 / 26, -1 / 26, 1 / 78], [2 / 21, -9 / 7, 9 / 7, -2 / 21],
            [1 / 75, 0, -27 / 25, 83 / 75, -1 / 25]],
        dc=[[-2, 3, -1], [-1, 1], [1 / 24, -9 / 8, 9 / 8, -1 / 24], [-1 / 71, 6 / 71, -83 / 71, 81 / 71, -3 / 71]],
        ii=[[0.5 + _C13 + 2 * _C14, 0.5 - 2 * _C13 - 3 * _C14, _C13, _C14],
            [-8 / 63 - 52 / 21 * _C13 - 104 / 21 * _C14, 29 / 42 + 104 / 21 * _C13 + 52 / 7 * _C14,
             -52 / 21 * _C13 + 0.5, -52 / 21 * _C14 - 4 / 63],
            [26 / 25 * _C13 + 52 / 25 * _C14 - 1 / 25, -1 / 50 - 52 / 25 * _C13 - 78 / 25 * _C14,
             3 / 5 + 26 / 25 * _C13, 13 / 25 + 26 / 25 * _C14, -3 / 50]],
        ic=[[39 / 28 + 39 / 14 * _C13 + 39 / 7 * _C14, -2 / 7 - 39 / 7 * _C13 - 78 / 7 * _C14,
             39 / 14 * _C13 + 39 / 7 * _C14 - 3 / 28],
            [13 / 27 - 52 / 27 * _C13 - 26 / 9 * _C14, 29 / 54 + 104 / 27 * _C13 + 52 / 9 * _C14,
             -1 / 54 - 52 / 27 * _C13 - 26 / 9 * _C14],
            [13 / 12 * _C13, 7 / 16 - 13 / 6 * _C13, 5 / 8 + 13 / 12 * _C13, -1 / 16],
            [78 / 71 * _C14, -156 / 71 * _C14 - 4 / 71, 39 / 71 + 78 / 71 * _C14, 81 / 142, -9 / 142]],
        dq=[9 / 8, -1 / 24], iq=[9 / 16, -1 / 16], R=[15 / 8, -5 / 4, 3 / 8], hc=[13 / 12, 7 / 8, 25 / 24],
        hi=[7 / 18, 9 / 8, 1, 71 / 72]),
    63: dict(
        di=[[-0.9795214020218487, 0.9597522747540616, -0.0021284121310923276, 0.04308560808739484,
             -0.02118806868851538],
            [0.10094185622089052, -1.3621007582168956, 1.480651137325344, -0.2787674248835621, 0.059275189554223895],
            [0.1050522197237869, -0.3755418649660661, -0.5066880707069372, 0.7227932046793403, 0.05138416400746168,
             0.0030003472624146313],
            [-0.010281664659776757, 0.009016888173475901, 0.1158762991569453, -1.3063741185003286,
             1.2879206487212211, -0.10361859147794651, 0.007460538586412149],
            [-0.08522272532774755, 0.2300959768599209, -0.06748505183821596, -0.28075281972041166,
             -0.77959568679678, 1.0363920760788554, -0.05757733755993641, 0.0041455683043154215],
            [0.03958146265158008, -0.10105244572213268, 0.0269485128845091, 0.10551623486389128,
             -0.009407429883264403, -1.1945625283432082, 1.1945625283432082, -0.066364584907956,
             0.004778250113372832]],
        dc=[[-3.137061163091724, 6.472195962306311, -4.476505551641335, 0.9669525120033824, 0.2921335971506185,
             -0.11771535672725233],
            [-0.8550973738466245, 0.5371097071174838, 0.4442015766629761, -0.00428923422758698, -0.1969782207705677,
             0.07505354506431924],
            [0.003267033496606009, -1.0058841165930086, 1.032532798072641, -0.09496402962593153, 0.0995309639229438,
             -0.03448264927325102],
            [-0.0460358301286618, 0.1318266207921457, -1.0252815152152988, 0.7452431221796392, 0.2882309687613436,
             -0.093983366389168],
            [0.025410671711714995, -0.031462633326690415, -0.08181244708002722, -0.8246706459806198,
             0.8983528780132024, 0.009405106598725824, 0.004777070063694267]],
        ii=[[0.4559762640735722, 0.5156609261411327, 0.09215963713516839, -0.055207108988023945,
             -0.008589718361849435],
            [-0.2329150785274282, 1.0886403314451474, 0.006569476829126231, 0.1526003661160169,
             -0.014895095862863417],
            [-0.13300622901536394, 0.24335188147388265, 0.43548086151449933, 0.4385084167668463,
             0.008164201104099517, 0.007500868156036579],
            [0.10717671074312715, -0.3332211159670528, 0.3310769312612241, 0.29067744812134255, 0.7410665665922483,
             -0.15542788721691977, 0.018651346466030373],
            [0.09305432569823871, -0.07099703081266313, -0.291616405335888, 0.3005623879587947, 0.5268027700312061,
             0.5181960380394277, -0.08636600633990461, 0.010363920760788554],
            [-0.05115521553501697, 0.05753938634775091, 0.09801308881771609, -0.1230378129758785,
             -0.08832072291927771, 0.5972812641716041, 0.5972812641716041, -0.09954687736193402,
             0.011945625283432081]],
        ic=[[1.6267303202606325, -0.3677632041998704, -0.6299565857805535, 0.2041457799345569, 0.3189794129688649,
             -0.15213572318363067],
            [0.4594313713417274, 0.42927755971902565, 0.287843512318841, -0.15850960868795075,
             -0.060778415165360984, 0.04273558047371772],
            [0.14146161692901638, 0.004462990795171873, 0.8874262064612957, 0.2713272665549153,
             -0.43009320031948844, 0.12541511957908888],
            [-0.058987332524401276, 0.07216334765484655, 0.6220237974938234, 0.16582184683346107,
             0.3085681858542267, -0.10958984531195667],
            [-0.0103015766372022, -0.007906156741522508, 0.012998815562764554, 0.47451358497362967,
             0.607051568675785, -0.0882989109926898, 0.01194267515923567]],
        dq=[75 / 64, -25 / 384, 3 / 640], iq=[75 / 128, -25 / 256, 3 / 256], R=[35 / 16, -35 / 16, 21 / 16, -5 / 16],
        hc=[325363 / 276480, 144001 / 276480, 43195 / 27648, 86857 / 138240, 312623 / 276480, 271229 / 276480],
        hi=[95 / 288, 317 / 240, 23 / 30, 793 / 720, 157 / 160]),
}


def _matrix(rows, half, n_out, n_in, sign):
    """The dense matrix of a staggered stencil: closure rows, mirrored at the
    end with `sign`, and the interior half stencil (sign: -1 derivative)."""
    m = np.zeros((n_out, n_in))
    off = 0 if n_out < n_in else -1  # centre k lies between interfaces k and k + 1
    for k in range(len(rows), n_out - len(rows)):
        for q, c in enumerate(half):
            m[k, k + off + 1 + q] += c
            m[k, k + off - q] += sign * c
    for r, row in enumerate(rows):
        for q, c in enumerate(row):
            m[r, q] += c
            m[n_out - 1 - r, n_in - 1 - q] += sign * c
    return torch.tensor(m, device=_device())


class _Exact:
    """The operator in 64 bits; fields as [6, ny, nx] tensors."""

    def __init__(self, N, order):
        self.N, n, b = N, N + 1, _SBP[order]
        self.hx = 0.5 * math.pi / N
        self.R, self.hi = b["R"], b["hi"]
        self.sat = [0.5 * r / h for r, h in zip(b["R"], b["hc"])]
        self.Di, self.Dc = _matrix(b["di"], b["dq"], N, n, -1), _matrix(b["dc"], b["dq"], n, N, -1)
        self.Ii, self.Ic = _matrix(b["ii"], b["iq"], N, n, 1), _matrix(b["ic"], b["iq"], n, N, 1)

        def metric(xt, yt):
            X, Y = _mesh(N, xt, yt)
            s2 = 1 + X * X + Y * Y
            s, cx, cy = torch.sqrt(s2), 1 + X * X, 1 + Y * Y
            return X, Y, s, cx * cy / (s2 * s), s2 / cx, s2 * X * Y / (cx * cy), s2 / cy

        def coriolis(X, Y, s):
            return 2 * OMEGA * _to_panels(X / s, Y / s, 1 / s)[..., 2]

        def norm(centre):
            e, m = (b["hc"], N) if centre else (b["hi"], n)
            w = torch.ones(m, dtype=torch.float64, device=_device())
            w[:len(e)] = torch.tensor(e, dtype=torch.float64)
            w[m - len(e):] = torch.tensor(e[::-1], dtype=torch.float64)
            return w

        X, Y, s, self.Jh, _, q12, _ = metric(0, 0)
        self.JQ12, self.fJ2 = self.Jh * q12, coriolis(X, Y, s) * self.Jh ** 2
        _, _, _, self.Ju, self.Q11, _, _ = metric(1, 0)
        _, _, _, self.Jv, _, _, self.Q22 = metric(0, 1)
        X, Y, s, self.Jo, _, _, _ = metric(1, 1)
        self.fo = coriolis(X, Y, s)
        self.w = {m: J * self.hx ** 2 * norm(yt)[:, None] * norm(xt)[None, :] for m, J, xt, yt in
                  (("h", self.Jh, 0, 0), ("u", self.Ju, 1, 0), ("v", self.Jv, 0, 1), ("o", self.Jo, 1, 1))}
        # which side of which panel meets side s of panel p, from the
        # positions of the sides' end points (0 left, 1 right, 2 bottom, 3 top)
        ends = {}
        for p in range(6):
            def at(x, y, p=p):
                return tuple(x * np.array(_EX[p]) + y * np.array(_EY[p]) - np.array(_NN[p]))
            for k, e in enumerate(((at(-1, -1), at(-1, 1)), (at(1, -1), at(1, 1)), (at(-1, -1), at(1, -1)),
                                   (at(-1, 1), at(1, 1)))):
                ends[p, k] = e
        self.q, self.qs, self.rev = (torch.zeros(6, 4, dtype=torch.long, device=_device()) for _ in range(3))
        for (p, k), e in ends.items():
            for (q, m), f in ends.items():
                if q != p and set(e) == set(f):
                    self.q[p, k], self.qs[p, k], self.rev[p, k] = q, m, int(e != f)
        side = torch.arange(4, device=_device())[None, :].expand(6, 4)
        out = (side % 2 == 1) == (self.qs % 2 == 0)  # both axes cross the edge the same way
        self.cross = torch.where(out, 1.0, -1.0).double()[..., None]
        self.along = torch.where(self.rev == 1, -1.0, 1.0).double()[..., None]
        self.swap = ((side <= 1) != (self.qs <= 1))[..., None]
        # covariant sync weights: own across-edge covariant vector . the
        # neighbour's along-edge contravariant one, the neighbour's prototype
        # face folded onto this one
        c, e = -0.25 * math.pi + self.hx * np.arange(n), np.full(n, 0.25 * math.pi)

        def basis(al, be):
            X, Y = np.tan(al), np.tan(be)
            s2, cx, cy = 1 + X * X + Y * Y, 1 + X * X, 1 + Y * Y
            s3 = s2 * np.sqrt(s2)
            a1 = np.array([cx * cy / s3, -X * Y * cx / s3, -X * cx / s3])
            a2 = np.array([-X * Y * cy / s3, cx * cy / s3, -Y * cy / s3])
            q11, q12, q22 = s2 / cx, s2 * X * Y / (cx * cy), s2 / cy
            return a1, a2, q11 * a1 + q12 * a2, q12 * a1 + q22 * a2

        qb = [basis(c, -e)[1], basis(c, e)[2]]
        qt = [basis(c, e)[1], basis(c, -e)[2]]
        ql = [basis(-e, c)[0], basis(e, c)[3]]
        qr = [basis(e, c)[0], basis(-e, c)[3]]
        self.wt = torch.tensor(np.stack([
            -ql[0][0] * ql[1][2] + ql[0][1] * ql[1][1] + ql[0][2] * ql[1][0],
            qr[0][0] * qr[1][2] + qr[0][1] * qr[1][1] - qr[0][2] * qr[1][0],
            qb[0][0] * qb[1][0] - qb[0][1] * qb[1][2] + qb[0][2] * qb[1][1],
            qt[0][0] * qt[1][0] + qt[0][1] * qt[1][2] - qt[0][2] * qt[1][1]]), device=_device())

    @staticmethod
    def _x(M, f):
        return f @ M.T

    @staticmethod
    def _y(M, f):
        return torch.matmul(M, f)

    @staticmethod
    def _sides(l, r, b, t):
        return torch.stack([l, r, b, t], 1)

    def _edge(self, f):
        return self._sides(f[:, :, 0], f[:, :, -1], f[:, 0, :], f[:, -1, :])

    def _nb(self, e):
        """What the neighbours hold at the sides' points ([6, 4, n])."""
        g = e[self.q, self.qs]
        return torch.where(self.rev[..., None] == 1, g.flip(-1), g)

    def _grad(self, f, dup, x):
        """i2c derivative along x or y with its SAT against the duplicates."""
        s = len(self.sat)
        if x:
            d = self._x(self.Di, f)
            for r in range(s):
                d[:, :, r] += self.sat[r] * (f[:, :, 0] - dup[:, 0])
                d[:, :, -1 - r] += self.sat[r] * (dup[:, 1] - f[:, :, -1])
        else:
            d = self._y(self.Di, f)
            for r in range(s):
                d[:, r, :] += self.sat[r] * (f[:, 0, :] - dup[:, 2])
                d[:, -1 - r, :] += self.sat[r] * (dup[:, 3] - f[:, -1, :])
        return d

    def contra(self, u, v):
        w1, w2 = self.JQ12 * self._y(self.Ic, v), self.JQ12 * self._x(self.Ic, u)
        return self.Q11 * u + self._x(self.Ii, w1) / self.Ju, self.Q22 * v + self._y(self.Ii, w2) / self.Jv

    def _sync(self, a, corner, lr, bt):
        """Edge points of a become lr / bt (left, right / bottom, top rows),
        corner points `corner`."""
        a = a.clone()
        a[:, 1:-1, 0], a[:, 1:-1, -1] = lr[0][:, 1:-1], lr[1][:, 1:-1]
        a[:, 0, 1:-1], a[:, -1, 1:-1] = bt[0][:, 1:-1], bt[1][:, 1:-1]
        for i in (0, -1):
            for j in (0, -1):
                a[:, j, i] = corner(i, j)
        return a

    def apply(self, u, v, h, rotate=True):
        C = 0.5 / self.hi[0]
        ut, vt = self.contra(u, v)
        ju, jv = self.Ju * ut, self.Jv * vt
        dx, dy = self._x(self.Dc, ju), self._y(self.Dc, jv)
        for r, c in enumerate(self.R):
            own = self._sides(ju[:, :, r], ju[:, :, -1 - r], jv[:, r, :], jv[:, -1 - r, :])
            jump = C * c * (own - self.cross * self._nb(own))
            dx[:, :, 0] += jump[:, 0]
            dx[:, :, -1] -= jump[:, 1]
            dy[:, 0, :] += jump[:, 2]
            dy[:, -1, :] -= jump[:, 3]
        div = (dx + dy) / (self.Jh * RADIUS * self.hx)
        e, nd = self._edge(div), self._nb(self._edge(div))
        side = {0: (0, 2), -1: (1, 3)}
        mean = 0.5 * (e + nd)
        div = self._sync(div, lambda i, j: (div[:, j, i] + nd[:, side[i][0], j] + nd[:, side[j][1], i]) / 3,
                         (mean[:, 0], mean[:, 1]), (mean[:, 2], mean[:, 3]))
        du = -GRAV / (self.hx * RADIUS) * self._grad(h, self._nb(self._edge(h)), True)
        dv = -GRAV / (self.hx * RADIUS) * self._grad(h, self._nb(self._edge(h)), False)
        if rotate:
            V, U = self.fJ2 * self._y(self.Ic, vt), -self.fJ2 * self._x(self.Ic, ut)
            nV, nU = self._nb(self._edge(V)), self._nb(self._edge(U))
            # across-edge and along-edge components in this panel's frame:
            # V is the first (x), U the second (y) component of the pair
            lr = (torch.arange(4, device=_device()) <= 1)[None, :, None]
            first, second = torch.where(self.swap, nU, nV), torch.where(self.swap, nV, nU)
            hV = torch.where(lr, self.cross, self.along) * first
            hU = torch.where(lr, self.along, self.cross) * second
            eV, eU, w = self._edge(V), self._edge(U), self.wt[None]
            mU = torch.where(lr, 0.5 * (eU + hU), 0.5 * (eU + hU + w * hV))
            mV = torch.where(lr, 0.5 * (eV + hV + w * hU), 0.5 * (eV + hV))

            def cU(i, j):
                a, b = side[i][0], side[j][1]
                return (U[:, j, i] + hU[:, a, j] + hU[:, b, i] + self.wt[b, i] * hV[:, b, i]) / 3

            def cV(i, j):
                a, b = side[i][0], side[j][1]
                return (V[:, j, i] + hV[:, a, j] + hV[:, b, i] + self.wt[a, j] * hU[:, a, j]) / 3

            U2 = self._sync(U, cU, (mU[:, 0], mU[:, 1]), (mU[:, 2], mU[:, 3]))
            V2 = self._sync(V, cV, (mV[:, 0], mV[:, 1]), (mV[:, 2], mV[:, 3]))
            du = du + self._x(self.Ii, V2) / self.Ju
            dv = dv + self._y(self.Ii, U2) / self.Jv
        return [du, dv, -DEPTH * div]

    def rk4(self, y, dt, steps):
        for _ in range(steps):
            k1 = self.apply(*y)
            k2 = self.apply(*(a + 0.5 * dt * k for a, k in zip(y, k1)))
            k3 = self.apply(*(a + 0.5 * dt * k for a, k in zip(y, k2)))
            k4 = self.apply(*(a + dt * k for a, k in zip(y, k3)))
            y = [a + dt / 6 * (p + 2 * q + 2 * r + s) for a, p, q, r, s in zip(y, k1, k2, k3, k4)]
        return y

    def solve(self, rhs, dt):
        """(I - dt L0)^-1 rhs, L0 without rotation: conjugate gradients on
        the Helmholtz problem for h, to rounding."""
        zu, zv = torch.zeros_like(rhs[0]), torch.zeros_like(rhs[1])

        def helm(z):
            g = self.apply(zu, zv, z, False)
            return z - dt * dt * self.apply(g[0], g[1], torch.zeros_like(z), False)[2]

        def dot(a, b):
            return (self.w["h"] * a * b).sum()

        b = rhs[2] + dt * self.apply(rhs[0], rhs[1], torch.zeros_like(rhs[2]), False)[2]
        x, r = b, b - helm(b)
        p, rr = r, dot(r, r)
        for _ in range(400):
            if float(rr) <= 1e-26 * float(dot(b, b)):
                break
            ap = helm(p)
            al = rr / dot(p, ap)
            x, r = x + al * p, r - al * ap
            new = dot(r, r)
            p, rr = r + new / rr * p, new
        g = self.apply(zu, zv, x, False)
        return [rhs[0] + dt * g[0], rhs[1] + dt * g[1], x]

    def curl(self, u, v):
        t = self._sides(v[:, :, 0], v[:, :, -1], u[:, 0, :], u[:, -1, :])
        dup = self.along * self._nb(t)
        return (self._grad(v, dup, True) - self._grad(u, dup, False)) / (self.hx * RADIUS * self.Jo)

    def diagnostics(self, u, v, h, dt, g):
        ut, vt = self.contra(u, v)
        w, sq = self.w, (RADIUS * self.hx) ** 2
        hu, hv = self._x(self.Ii, h), self._y(self.Ii, h)
        hq = 0.5 * (self._y(self.Ii, hu) + self._x(self.Ii, hv))
        z = self.curl(u, v) + self.fo
        mass = (h * w["h"]).sum()
        energy = 0.5 * GRAV * (h * h * w["h"]).sum() + 0.5 * DEPTH * ((u * ut * w["u"]).sum() + (v * vt * w["v"]).sum())
        ke = 0.5 * ((hu * ut * u * w["u"]).sum() + (hv * vt * v * w["v"]).sum())
        pe = 0.5 * g * (h * h * w["h"]).sum()
        ens = (0.5 * z * z / hq * w["o"]).sum()
        val = [float(a) for a in (mass, energy, h.min(), h.max(), mass, ke + pe, ke, pe, ens)]
        cfl = [math.sqrt(g * float(h.max()) / sq) * dt] + [math.sqrt(float((a * b).abs().max()) / sq) * dt
                                                           for a, b in ((ut, u), (vt, v))]
        return [val[:2], dict(zip(("hmin", "hmax", "mass", "TE", "KE", "PE", "Enstrophy"), val[2:9])),
                dict(zip(("gravity", "advective_x", "advective_y"), cfl))]


def exact(case, seed):
    kind = case["kind"]
    if kind in ("ensemble", "uneven", "serve"):
        grids, out = {}, []
        for k, (N, order, _, dt, steps) in enumerate(_solves(case)):
            if (N, order) not in grids:
                grids[N, order] = _Exact(N, order)
            out.append(_host(grids[N, order].rk4(_fields(N, 1000 * seed + k), dt, steps)))
        return out
    N = case["N"]
    grid = _Exact(N, case["order"])
    y = _fields(N, seed, DEPTH if kind == "diag" else 0.0)
    if kind == "diag":
        return grid.diagnostics(*y, _time_step(N, 0.5), DIAG_GRAV)
    if kind == "apply":
        return _host(grid.apply(*y))
    if kind == "rk4":
        return _host(grid.rk4(y, _solves(case)[0][3], case["steps"]))
    dt = _time_step(N, 4.0)
    for _ in range(case["steps"]):
        f = grid.apply(*y)
        y = grid.solve([a + 0.5 * dt * k for a, k in zip(y, f)], 0.5 * dt)
    return _host(y)
