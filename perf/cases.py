"""The evaluations that a user of this library has it do, for timing them and
for comparing two builds' outputs.

Four ways into the library are covered:
  call    one spectrum per call through rx_eval_model, host arrays in and out:
          an XSPEC / ISIS fit, which evaluates one model hundreds of times on
          one energy grid with other parameters each time (the lmod* entry
          points are this call in FP64);
  device  one spectrum on device tensors through rx_eval_model_noalloc: a
          likelihood whose data already live on the GPU;
  batch   a resident batch through rx_batch_run, every output then read into
          the caller's arrays: the walkers of an ensemble sampler, parameter
          scans and training sets;
  serve   a burst of mixed requests through the serving loop.
Parameters are drawn over the priors that the benchmark uses (spin
U[-0.998, 0.998], inclination U[5, 85] deg, Rin from the ISCO to 50, height
U[3, 100]), inputs are a cut-off power law with two iron lines.
"""
import ctypes
import math

import numpy as np
import torch

import relxill_amd as rx

_DP = ctypes.POINTER(ctypes.c_double)

MODELS = {"relline": rx.MODEL_RELLINE, "relline_lp": rx.MODEL_RELLINELP, "relconv": rx.MODEL_RELCONV,
          "relconv_lp": 12, "relxill": rx.MODEL_RELXILL, "relxilllp": rx.MODEL_RELXILLLP,
          "relxillcp": rx.MODEL_RELXILLCP, "relxilllpcp": rx.MODEL_RELXILLLPCP}
LINE = ("relline", "relline_lp")
CONV = ("relconv", "relconv_lp")
LAMP_POST = ("relline_lp", "relconv_lp", "relxilllp", "relxilllpcp")
N_RADII, N_CONV, CONV_LO, CONV_HI = 1000, 4096, 0.00035, 2000.0  # the library's default grids


def listed():
    return [
        # a fit of a single line to a narrow CCD band: the smallest call there is
        dict(name="relline call 299", path="call", model="relline", bins=299, requests=1, fp32=False, rrad=False),
        # the same with a convolution of the continuum on a full detector grid
        dict(name="relconv call 3000", path="call", model="relconv", bins=3000, requests=1, fp32=False, rrad=False),
        # a GPU-resident likelihood, one line at a time on an odd grid
        dict(name="relline_lp device 1777", path="device", model="relline_lp", bins=1777, requests=1, fp32=True,
             rrad=False),
        # the model most fits use, one call at a time
        dict(name="relxill call 3000", path="call", model="relxill", bins=3000, requests=1, fp32=False, rrad=False),
        # its lamp-post form with the returning radiation on, as the model's defaults have it
        dict(name="relxilllp call 3000", path="call", model="relxilllp", bins=3000, requests=1, fp32=False, rrad=True),
        # the same with the Comptonised primary: the most expensive single call
        dict(name="relxilllpcp call 2501", path="call", model="relxilllpcp", bins=2501, requests=1, fp32=False,
             rrad=True),
        # the benchmark's workload: 4096 convolutions on grids of 300-8000 bins
        dict(name="relconv batch 4096", path="batch", model="relconv", bins=0, requests=4096, fp32=True, rrad=False),
        # an ensemble sampler's walkers on a lamp-post line
        dict(name="relline_lp batch 256", path="batch", model="relline_lp", bins=3000, requests=256, fp32=True,
             rrad=False),
        # a parameter scan of the full model
        dict(name="relxill batch 1024", path="batch", model="relxill", bins=3000, requests=1024, fp32=True,
             rrad=False),
        # a smaller scan of its lamp-post form in double precision
        dict(name="relxilllp batch 128", path="batch", model="relxilllp", bins=3000, requests=128, fp32=False,
             rrad=False),
        # walkers of a fit with the Comptonised lamp post
        dict(name="relxilllpcp batch 64", path="batch", model="relxilllpcp", bins=1500, requests=64, fp32=False,
             rrad=True),
        # a burst of line, convolution and lamp-post requests at the serving loop
        dict(name="serve 512", path="serve", model="mixed", bins=0, requests=512, fp32=True, rrad=False),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    path = rng.choice(["call", "call", "device", "batch", "batch", "serve"])
    if path == "call":
        model = rng.choice(["relline", "relline_lp", "relconv", "relconv_lp", "relxill", "relxilllp", "relxillcp",
                            "relxilllpcp"])
        return dict(path=path, model=model, bins=size(200, 8000), requests=1, fp32=rng.random() < 0.25,
                    rrad=model in LAMP_POST and rng.random() < 0.5)
    if path == "device":
        model = rng.choice(["relline", "relline_lp", "relconv", "relconv_lp"])
        return dict(path=path, model=model, bins=size(200, 8000), requests=1, fp32=rng.random() < 0.5, rrad=False)
    if path == "batch":
        model = rng.choice(["relline", "relline_lp", "relconv", "relconv_lp", "relxill", "relxilllp", "relxilllpcp"])
        most = {"relxill": 1024, "relxilllp": 192, "relxilllpcp": 64}.get(model, 2048)
        return dict(path=path, model=model, bins=rng.choice([0, size(300, 6000)]), requests=size(8, most),
                    fp32=rng.random() < 0.5, rrad=model in LAMP_POST and rng.random() < 0.3)
    return dict(path=path, model="mixed", bins=0, requests=size(32, 1024), fp32=True, rrad=False)


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------
def kerr_rms(a):
    s = -1.0 if a < 0 else 1.0
    z1 = 1.0 + (1.0 - a * a) ** (1.0 / 3.0) * ((1.0 + a) ** (1.0 / 3.0) + (1.0 - a) ** (1.0 / 3.0))
    z2 = math.sqrt(3.0 * a * a + z1 * z1)
    return 3.0 + z2 - s * math.sqrt((3.0 - z1) * (3.0 + z1 + 2 * z2))


def log_grid(n_bins, emin, emax):
    i = np.arange(n_bins + 1, dtype=np.float64)
    return np.exp(i / n_bins * (np.log(emax) - np.log(emin)) + np.log(emin))


def continuum(e):
    """cut-off power law and two iron lines, photons per bin"""
    em = 0.5 * (e[1:] + e[:-1])
    lines = 0.02 * np.exp(-0.5 * ((em - 6.4) / 0.05) ** 2) + 0.008 * np.exp(-0.5 * ((em - 6.97) / 0.05) ** 2)
    return (em ** -2.0 * np.exp(-em / 300.0) + lines) * np.diff(e)


def parameters(model, rng, rrad):
    """one parameter array in the model's order"""
    a = rng.uniform(-0.998, 0.998)
    incl = rng.uniform(5.0, 85.0)
    # half of the fits leave Rin at the ISCO (a negative value is in units of it);
    # the returning radiation's table starts there
    rin = -1.0 if rng.uniform() < 0.5 else rng.uniform(kerr_rms(a), 50.0)
    rout = float(np.exp(rng.uniform(np.log(200.0), np.log(990.0))))
    q = [rng.uniform(2.0, 6.0), rng.uniform(2.0, 4.0), rng.uniform(5.0, 40.0)]
    h = rng.uniform(3.0, 100.0)
    gam = rng.uniform(1.4, 2.8)
    lxi, afe = rng.uniform(0.0, 4.5), rng.uniform(0.5, 10.0)
    ecut = float(np.exp(rng.uniform(np.log(20.0), np.log(800.0))))
    kte, dens = float(np.exp(rng.uniform(np.log(5.0), np.log(300.0)))), rng.uniform(15.0, 19.0)
    rr = 1.0 if rrad else 0.0
    if model == "relline":
        return [6.4] + q + [a, incl, rin, rout, 0.0, 0.0]
    if model == "relline_lp":
        return [6.4, h, a, incl, rin, rout, 0.0, 0.0, gam, rr]
    if model == "relconv":
        return q + [a, incl, rin, rout, 0.0]
    if model == "relconv_lp":
        return [h, 0.0, a, incl, rin, rout, 0.0, gam, rr]
    if model == "relxill":
        return q + [a, incl, rin, rout, 0.0, gam, lxi, afe, ecut, 3.0]
    if model == "relxilllp":
        return [h, 0.0, a, incl, rin, rout, 0.0, gam, lxi, afe, ecut, 1.0, rr, 0.0]
    if model == "relxillcp":
        return [incl, a, rin, rout, q[2], q[0], q[1], 0.0, gam, lxi, dens, afe, kte, 3.0]
    return [incl, a, rin, rout, h, 0.0, gam, lxi, dens, afe, kte, 1.0, 0.0, 0.0, 0.0, rr, 0.0]


def requests_of(case, seed):
    # the models and grids of a case are always the same, the parameters are the seed's
    rng, grids = np.random.default_rng([int(seed), 17]), np.random.default_rng(case["requests"])
    reqs, shared = [], {}
    for _ in range(case["requests"]):
        model = case["model"]
        if model == "mixed":
            model = grids.choice(["relline", "relconv", "relline_lp"], p=[0.4, 0.4, 0.2])
        n = case["bins"] or int(np.exp(grids.uniform(np.log(300), np.log(8000))))
        key = (n, model in LINE)
        if key not in shared:  # requests of one grid size share the grid, as walkers of one fit do
            e = log_grid(n, 0.1, 10.0 if model in LINE else 100.0)
            shared[key] = (e, continuum(e))
        e, f = shared[key]
        reqs.append(dict(model=MODELS[model], energy=e, params=parameters(model, rng, case["rrad"]),
                         flux_in=f if model in CONV else None))
    return reqs


_ready = False


def _library():
    """the device and every table resident, as after a program's first call of each model"""
    global _ready
    if not _ready:
        if rx.lib.rx_init(0) != 0:
            raise RuntimeError(rx.lib.rx_last_error().decode())
        e = log_grid(200, 0.5, 20.0)
        for m in ("relline_lp", "relxill", "relxilllp", "relxillcp", "relxilllpcp"):
            rx.eval_model(MODELS[m], parameters(m, np.random.default_rng(3), m == "relxilllp"), e)
        _ready = True


class _State:
    def __init__(self, case, reqs):
        self.case, self.reqs, self.precision = case, reqs, rx.FP32 if case["fp32"] else rx.FP64

    def __del__(self):
        if getattr(self, "batch", None) is not None:
            self.batch.close()
        if getattr(self, "server", None) is not None:
            self.server.stop()


def prepare(case, seed):
    _library()
    reqs = requests_of(case, seed)
    st = _State(case, reqs)
    if case["path"] == "batch":
        st.batch = rx.Batch(reqs)
        at = np.cumsum([0] + st.batch.n_flux)
        st.flux = np.zeros(int(at[-1]))
        st.rows = [st.flux[at[i]:at[i + 1]].ctypes.data_as(_DP) for i in range(len(reqs))]
    elif case["path"] == "device":
        r = reqs[0]
        st.energy = torch.from_numpy(r["energy"]).cuda()
        st.flux_in = torch.from_numpy(r["flux_in"]).cuda() if r["flux_in"] is not None else None
        st.flux = torch.zeros(r["energy"].size - 1, dtype=torch.float64, device="cuda")
        st.params = np.array(r["params"], dtype=np.float64)
    elif case["path"] == "serve":
        st.server = rx.Server(max_inflight=4096, hbm_budget=16 << 30, n_streams=4, precision=st.precision)
    return st


def run(st):
    path = st.case["path"]
    if path == "call":
        r = st.reqs[0]
        return rx.eval_model(r["model"], r["params"], r["energy"], flux_in=r["flux_in"], precision=st.precision)[0]
    if path == "device":
        s = rx.lib.rx_eval_model_noalloc(
            st.reqs[0]["model"], st.params.ctypes.data_as(_DP), ctypes.cast(st.energy.data_ptr(), _DP),
            ctypes.cast(st.flux_in.data_ptr(), _DP) if st.flux_in is not None else None,
            ctypes.cast(st.flux.data_ptr(), _DP), st.flux.numel(), st.precision,
            torch.cuda.current_stream().cuda_stream)
        if s != rx.RX_OK:
            raise RuntimeError(rx.lib.rx_last_error().decode())
        return st.flux
    if path == "batch":
        b, read = st.batch, rx.lib.rx_batch_output
        b.run(st.precision)
        b.sync()
        for i, row in enumerate(st.rows):
            if read(b.h, i, row) != rx.RX_OK:
                raise RuntimeError("request %d failed" % i)
        return st.flux
    tickets = st.server.replay(st.reqs, np.zeros(len(st.reqs)))
    st.server.drain()
    got = [st.server.poll(t) for t in tickets]
    if any(g is None or g[1] != rx.RX_OK for g in got):
        raise RuntimeError("a served request failed")
    return np.concatenate([g[0] for g in got])


# --------------------------------------------------------------------------
# work
# --------------------------------------------------------------------------
def work(case):
    """Bytes: the table corners a spectrum interpolates, its grid, input and
    output.  Operations: the integrand evaluations of the reference's bin
    integrals (20 operations each), the transforms of a convolution, the
    interpolation of the reflection table, the tridiagonal solves."""
    model = case["model"]
    n = case["bins"] or 2350  # mean of the log-uniform grids
    zones = 10 if model in ("relxilllp", "relxilllpcp") else 1
    # (radius, bin) pairs inside a radius' energy window: about 0.12 of the line
    # grids' and 0.012 of the convolution grid's, 3 to 5 evaluations each
    share = {"mixed": 0.5, **{m: 1.0 for m in LINE}}.get(model, 0.0)
    pairs = N_RADII * (share * 0.12 * n + (1.0 - share) * 0.012 * N_CONV)
    flops = 20.0 * 4.0 * pairs
    nbytes = 68800.0 + 8.0 * (n + 1) + 8.0 * n + (8.0 * n if model in CONV or model == "mixed" else 0.0)
    if model not in LINE:
        flops += (1.0 - share) * zones * 2.5 * N_CONV * math.log2(N_CONV) * 3.0
    if model.startswith("relxill"):
        rows = 16.0 * 1.4 if zones == 1 else 180.0  # table rows with a weight
        nbytes += rows * 2999 * 4.0
        flops += zones * 2.0 * rows * 2999
        if case["rrad"]:  # every inclination of every zone, for the correction factors
            nbytes += 16.0 * 10 * 2999 * 4.0
            flops += zones * 2.0 * 160 * 2999
    if model.endswith("cp"):
        flops += (1.0 + (zones if zones > 1 else 0)) * 900 * 300.0
    return {"bytes": nbytes * case["requests"], "flops": flops * case["requests"]}


# --------------------------------------------------------------------------
# the same spectra in plain 64-bit torch: lines and convolutions
# --------------------------------------------------------------------------
H, ROMB_PREC, ROMB_MAX = 5e-3, 0.02, 5


class _Plain:
    """The relativistic line and its convolution as the model defines them: the
    transfer function interpolated between its table nodes, 1000 radii, the
    integral over g* per energy bin (Romberg to 2 %, the closed form at the
    two ends, the midpoint below 0.95 of the line energy)."""

    def __init__(self):
        self.dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        self.rel, self.lp = rx.tables_view()  # the tables are input data

    def t(self, x):
        return torch.as_tensor(np.asarray(x, dtype=np.float64), device=self.dev)

    @staticmethod
    def bracket(arr, x):
        return int(np.clip(np.searchsorted(arr, np.float32(x), side="right") - 1, 0, arr.size - 2))

    def nodes(self, a, mu0):
        R = self.rel
        n_r, ng = R["n_r"], R["n_g"]
        ia, im = self.bracket(R["a"], a), self.bracket(R["mu0"], mu0)
        fa = float((np.float32(a) - R["a"][ia]) / (R["a"][ia + 1] - R["a"][ia]))
        fm = float((np.float32(mu0) - R["mu0"][im]) / (R["mu0"][im + 1] - R["mu0"][im]))

        def mix(name, shape):
            v = R[name].reshape((R["n_a"], R["n_mu0"]) + shape).astype(np.float64)
            return ((1 - fa) * (1 - fm) * v[ia, im] + fa * (1 - fm) * v[ia + 1, im] + (1 - fa) * fm * v[ia, im + 1]
                    + fa * fm * v[ia + 1, im + 1])

        r = R["r"].reshape(R["n_a"], R["n_mu0"], n_r).astype(np.float64)
        r = fa * r[ia + 1, im] + (1 - fa) * r[ia, im]
        t = np.stack([mix("trff1", (n_r, ng)), mix("trff2", (n_r, ng))], axis=-1)
        return r, mix("gmin", (n_r,)), mix("gmax", (n_r,)), t

    def lamp_post(self, a, h, gam, re):
        """emissivity of a stationary source at height h"""
        L = self.lp
        na, nh, nr = L["n_a"], L["n_h"], L["n_r"]
        ia = self.bracket(L["a"], a)
        fa = float((np.float32(a) - L["a"][ia]) / (L["a"][ia + 1] - L["a"][ia]))
        hs = L["h"].reshape(na, nh)

        def at(name):
            v, out = L[name].reshape(na, nh, nr).astype(np.float64), 0.0
            for k, w in ((ia, 1 - fa), (ia + 1, fa)):
                i = self.bracket(hs[k], h)
                f = float((np.float32(h) - hs[k][i]) / (hs[k][i + 1] - hs[k][i]))
                out = out + w * (f * v[k, i + 1] + (1 - f) * v[k, i])
            return out

        rad = L["rad"].reshape(na, nr).astype(np.float64)
        jr, je, jd = fa * rad[ia + 1] + (1 - fa) * rad[ia], at("intens"), at("del_")
        k = np.clip(np.searchsorted(jr, re, side="right") - 1, 0, nr - 2)
        lin = (re - jr[k]) / (jr[k + 1] - jr[k])
        lg = (np.log(re) - np.log(jr[k])) / (np.log(jr[k + 1]) - np.log(jr[k]))
        f = np.where(jd[k] / math.pi * 180.0 <= 75.0, lin, lg)
        sr = np.sqrt(re)
        g = (re * sr + a) / (sr * np.sqrt(re * re - 3 * re + 2 * a * sr)) / math.sqrt(
            (h * h + a * a) / (h * h - 2 * h + a * a))
        return np.exp(f * np.log(je[k + 1]) + (1 - f) * np.log(je[k])) * g ** gam

    def profile(self, E, a, incl, rin, rout, emissivity, bkn):
        """photons per bin on the grid E (line-energy units), summing to one"""
        rms = kerr_rms(a)
        tre, tgmin, tgmax, tT = self.nodes(a, math.cos(incl))
        n_r, ng, nr = tre.size, self.rel["n_g"], N_RADII
        if tre[-1] > rms and (tre[-1] - rms) / tre[-1] < 1e-3:
            tre[-1] = rms
        i_in = int(np.clip(np.sum(tre >= rin) - 1, 0, n_r - 2))
        i_out = int(np.clip(np.sum(tre >= rout) - 1, 0, n_r - 2))
        if tre[i_out] < 1000.0 < tre[i_out] * 1.01:
            tre[i_out] = 1000.0
        r1, r2 = 1.0 / math.sqrt(rout), 1.0 / math.sqrt(rin)
        re = (1.0 / (np.arange(nr) * (r2 - r1) / (nr - 1) + r1)) ** 2
        K = np.clip(np.minimum((tre[None, :] > re[:, None]).sum(1) - 1, i_in), 0, n_r - 2)
        f = (re - tre[K + 1]) / (tre[K] - tre[K + 1])
        gmin, gmax = (f * x[K] + (1 - f) * x[K + 1] for x in (tgmin, tgmax))
        T = f[:, None, None] * tT[K] + (1 - f)[:, None, None] * tT[K + 1]
        dr = np.empty(nr)
        dr[1:-1] = 0.5 * (re[:-2] - re[2:])
        dr[0], dr[-1] = 0.5 * (re[0] - re[1]), 0.5 * (re[-2] - re[-1])
        ring = re * dr * math.pi
        em = emissivity(re)
        if bkn:
            em = em / np.sum(em * ring * 2)
        coef = self.t(em / (gmax - gmin) * ring / 2)
        # pairs (radius, bin) inside the radius' window
        E = self.t(E)
        n = E.numel() - 1
        gmin, gmax, T = self.t(gmin), self.t(gmax), self.t(T).reshape(-1)
        lo = torch.clamp(torch.searchsorted(E, torch.clamp(gmin, min=float(E[0])), right=True) - 1, 0, n - 1)
        hi = torch.clamp(torch.searchsorted(E, torch.clamp(gmax, max=float(E[-1])), right=True) - 1, 0, n - 1)
        cnt = torch.where((gmax > E[0]) & (gmin < E[-1]), hi - lo + 1, torch.zeros_like(lo))
        rad = torch.repeat_interleave(torch.arange(nr, device=self.dev), cnt)
        j = torch.arange(rad.numel(), device=self.dev) - (torch.cumsum(cnt, 0) - cnt)[rad] + lo[rad]
        step = (1.0 - 2 * H) / (ng - 1)
        gs = self.t(H + step * np.arange(ng))

        def f2(e, rd):
            """both branches of the integrand at the energies e of the radii rd"""
            g = (e - gmin[rd]) * (1.0 / (gmax[rd] - gmin[rd]))
            i = torch.clamp(torch.searchsorted(gs, g, right=True) - 1, 0, ng - 2)
            w = (g - gs[i]) / (gs[i + 1] - gs[i])
            base = e ** 3 / torch.sqrt(g - g * g)
            at = (rd * ng + i) * 2
            return torch.stack([base * (w * T[at + b] + (1 - w) * T[at + 2 + b]) for b in (0, 1)])

        every = torch.arange(nr, device=self.dev)
        width = gmax - gmin
        normL = f2(H * width + gmin, every).sum(0) * math.sqrt(H)
        normU = f2((1 - H) * width + gmin, every).sum(0) * math.sqrt(H)
        w = width[rad]
        elo, ehi = E[j], E[j + 1]
        blo = torch.clamp((elo - gmin[rad]) / w, 0.0, 1.0)
        bhi = torch.clamp((ehi - gmin[rad]) / w, 0.0, 1.0)
        val = torch.zeros_like(elo)

        def edge(a_, b_):
            low = a_ <= 0.5
            l_, h_ = torch.where(low, a_, 1.0 - b_), torch.where(low, b_, 1.0 - a_)
            nrm = torch.where(low, normL[rad], normU[rad])
            return 2 * nrm * (torch.sqrt(torch.clamp(h_, min=0.0)) - torch.sqrt(torch.clamp(l_, min=0.0))) * w

        at_lo, at_hi = blo <= H, bhi >= 1 - H
        Ht = torch.full_like(blo, H)
        val = val + torch.where(at_lo, edge(blo, torch.minimum(bhi, Ht)), torch.zeros_like(val))
        val = val + torch.where(at_hi, edge(torch.maximum(blo, 1 - Ht), bhi), torch.zeros_like(val))
        rlo = torch.where(at_lo, H * w + gmin[rad], elo)
        rhi = torch.where(at_hi, (1 - H) * w + gmin[rad], ehi)
        inner = (bhi > H) & (blo < 1 - H)
        mid = inner & (rlo < 0.95)
        f = f2((rlo[mid] + rhi[mid]) / 2, rad[mid])
        val[mid] = val[mid] + f.sum(0) * (rhi[mid] - rlo[mid])
        rom = inner & (rlo >= 0.95)
        if bool(rom.any()):
            val[rom] = val[rom] + self.romberg(rlo[rom], rhi[rom], rad[rom], f2)
        val = torch.where(bhi > 0, val * coef[rad], torch.zeros_like(val))
        p = torch.zeros(n, dtype=torch.float64, device=self.dev).index_add_(0, j, val)
        p = p / (0.5 * (E[:-1] + E[1:]))
        return p / p.sum()

    @staticmethod
    def romberg(a, b, rd, f2):
        pas = b - a
        s = (f2(a, rd) + f2(b, rd)) / 2
        row = [s * pas]
        res, live = row[0].clone(), torch.ones_like(s, dtype=torch.bool)
        act = torch.arange(a.numel(), device=a.device)
        for n in range(1, ROMB_MAX + 2):
            pas = pas / 2
            for m in range(1 << (n - 1)):
                s = s + f2(a + pas * (2 * m + 1), rd)
            new, r = [s * pas], 1.0
            for ii in range(1, n + 1):
                r *= 4.0
                new.append((r * new[ii - 1] - row[ii - 1]) / (r - 1.0))
            top = row[n - 1]
            res[:, act] = torch.where(live, new[n], res[:, act])
            live = live & (torch.abs(new[n] - top) / new[n] > ROMB_PREC) & (n <= ROMB_MAX)
            keep = live.any(0)
            if not bool(keep.any()):
                break
            a, rd, pas, act = a[keep], rd[keep], pas[keep], act[keep]
            s, live, row = s[:, keep], live[:, keep], [x[:, keep] for x in new]
        return res.sum(0)

    @staticmethod
    def rebin(e_out, e_in, f_in):
        """photons of the bins e_in shared out over the bins e_out"""
        return np.diff(np.interp(e_out, e_in, np.concatenate([[0.0], np.cumsum(f_in)])))

    def spectrum(self, model, p, e, flux_in):
        line, lp = model in LINE, model in LAMP_POST
        if model == "relline":
            a, incl, rin, rout, q = p[4], p[5], p[6], p[7], p[1:4]
        elif model == "relconv":
            a, incl, rin, rout, q = p[3], p[4], p[5], p[6], p[0:3]
        elif model == "relline_lp":
            a, incl, rin, rout, h, gam = p[2], p[3], p[4], p[5], p[1], p[8]
        else:
            a, incl, rin, rout, h, gam = p[2], p[3], p[4], p[5], p[0], p[7]
        rms = kerr_rms(a)
        rin = max(-rin * rms if rin < 0 else rin, rms)
        if lp:
            h = max(h, 1.1 * (1 + math.sqrt(1 - a * a)))
            em = lambda re: self.lamp_post(a, h, gam, re)  # noqa: E731
        else:
            rbr = min(max(q[2], rin), rout)
            em = lambda re: (re / rbr) ** -np.where(re > rbr, q[1], q[0])  # noqa: E731
        ec = e / p[0] if line else log_grid(N_CONV, CONV_LO, CONV_HI)
        prof = self.profile(ec, a, incl * math.pi / 180, rin, rout, em, not lp).cpu().numpy()
        if line:
            return prof
        mid, de = 0.5 * (ec[1:] + ec[:-1]), np.diff(ec)
        band = (ec[:-1] >= 0.01) & (ec[1:] < 1000.0)
        x = self.rebin(ec, e, flux_in)
        y = np.roll(prof * mid / de, -(int(np.searchsorted(ec, 1.0, side="right")) - 1))
        c = np.fft.irfft(np.fft.rfft(x * mid / de) * np.fft.rfft(y), N_CONV) * de / mid
        c *= prof[band].sum() * x[band].sum() / c[band].sum()
        out = self.rebin(e, ec, c)
        out[(e[1:] < 0.01) | (e[:-1] > 1000.0)] = 0.0
        return out


_plain = None


def exact(case, seed):
    """Lines and convolutions in 64 bits; None for more spectra than some 20
    seconds take, and for the reflection models, whose ten zones, reflection
    tables and Comptonised continua have no short restatement."""
    global _plain
    if case["model"] not in LINE + CONV + ("mixed",) or case["rrad"] or case["requests"] > 512:
        return None
    if _plain is None:
        _plain = _Plain()
    name = {v: k for k, v in MODELS.items()}
    out = np.concatenate([_plain.spectrum(name[r["model"]], r["params"], r["energy"], r["flux_in"])
                          for r in requests_of(case, seed)])
    return torch.from_numpy(out) if case["path"] == "device" else out
