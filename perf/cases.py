"""The work that users of this library have it do, as cases to be timed and checked.

A case is a dict of plain values; `kind` says which calls of the library a pass makes:

  run       the step loop on a state in device memory: dj_set_state_device, dj_run, dj_get_state_device
  accel     one force evaluation of host arrays: PMSolverHIP.pm_acceleration
  ics       2LPT initial conditions from white noise in device memory: dj_ics_lpt_device
  gradient  the gradient of a density loss with respect to the white noise, through 2LPT and the steps
  train     one optimiser step of the learned correction at a snapshot, from fresh parameters
  spectra   the density and displacement spectra of a state over given bins

`exact` gives the same results in 64 bits from plain torch, without this repository's code.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "discodj.jl_amd"))

import discodj_amd as D  # noqa: E402

DEV = "cuda:0"
MESHES = [16, 24, 32, 48, 64, 96, 128, 192, 256, 384, 512, 768, 1024]

_RUN = dict(kind="run", L=500.0, worder=2, deconvolve=False, antialias=0, grad_order=4, lap_order=0, n_resample=1,
            resampling="fourier", precision=32, deposit="float", lean=False, net=False, stepper="bullfrog",
            a_ini=0.05, a_end=1.0, steps=10)


def _case(name=None, **kw):
    c = dict(_RUN, **kw)
    return c if name is None else dict(name=name, **c)


def listed():
    return [
        # one FP64 force of a small lattice with host arrays: unit tests, notebooks, the golden vectors' size
        _case("force_16_fp64", kind="accel", n=16, res=32, L=100.0, worder=3, antialias=1, precision=64),
        # a whole small simulation, the inner loop of parameter scans: launches and latency count
        _case("run_64", n=64, res=64, L=250.0, grad_order=2),
        # an FP64 run of a lattice that fits no power of two
        _case("run_100_192_fp64", n=100, res=192, L=200.0, worder=3, antialias=1, grad_order=4, precision=64,
              stepper="fastpm", a_ini=0.1, a_end=0.5, steps=4),
        # the lean solver with the bit-reproducible deposit on a mesh with a factor of three
        _case("run_192_384_fixed", n=192, res=384, L=400.0, worder=3, grad_order=4, lean=True, deposit="fixed64",
              stepper="fastpm", a_ini=0.2, a_end=0.6, steps=5),
        # the ordinary production run: 256^3 with interlacing
        _case("run_256", n=256, res=256, antialias=1),
        # three steps in the middle of the largest run's schedule, where the matter has clustered
        _case("run_512_1024", n=512, res=1024, L=1000.0, worder=3, antialias=1, grad_order=6, lap_order=6,
              stepper="fastpm", a_ini=0.43, a_end=0.5725, steps=3),
        # a step with the discreteness-suppressing options of the shell-crossing study
        _case("run_256_512_resampled", n=256, res=512, worder=4, deconvolve=True, antialias=1, grad_order=0,
              n_resample=2, a_ini=0.25, a_end=0.255, steps=1),
        # four steps with the learned potential correction on
        _case("run_256_net", n=256, res=256, net=True, a_ini=0.3, a_end=0.68, steps=4),
        # initial conditions of a 256^3 run
        _case("ics_256", kind="ics", n=256, res=256),
        # field-level inference: the gradient of a loss with respect to the initial white noise
        _case("gradient_256", kind="gradient", n=256, res=256),
        # training the learned correction: one optimiser step at 64^3
        _case("train_64", kind="train", n=64, res=64, L=125.0, a_ini=0.4),
        # the spectra that a study measures at every output
        _case("spectra_256_512", kind="spectra", n=256, res=512, bins=48, a_ini=0.5),
    ]


def _units(c):
    """A rough measure of a case's time, to keep drawn cases below the largest listed one."""
    T, M, P = c["precision"] // 8, c["res"] ** 3, c["n"] ** 3
    ns = 1 if c["antialias"] in (0, -1) else 2 if c["antialias"] == 1 else 8
    passes = 14 if c["grad_order"] == 0 else 5
    force = ns * (M * 2 * T * passes + P * c["n_resample"] ** 3 * (30 * T + 8 * c["worder"] ** 3))
    return force * (c["steps"] if c["kind"] == "run" else 4 * c["steps"] if c["kind"] == "gradient" else 2)


def draw(rng):
    largest = _units(next(c for c in listed() if c["name"] == "run_512_1024"))
    while True:
        kind = rng.choices(["run", "accel", "ics", "gradient", "train", "spectra"], [62, 6, 8, 8, 6, 10])[0]
        L = round(math.exp(rng.uniform(math.log(50), math.log(1500))), 1)
        worder, antialias = rng.choice([2, 3, 4]), rng.choice([0, 0, 1, 1, 1, -1, 2])
        grad = rng.choice([2, 4, 4, 6])
        lap = rng.choice([0, 0, grad])
        prec = rng.choice([32, 32, 64])
        a0 = round(rng.uniform(0.05, 0.6), 3)
        if kind in ("run", "accel"):
            res = rng.choice(MESHES[:12] if kind == "run" else MESHES[:6])
            n = max(8, round(res * math.exp(rng.uniform(math.log(0.3), 0.0))))
            c = _case(kind=kind, n=n, res=res, L=L, worder=worder, antialias=antialias, grad_order=grad, lap_order=lap,
                      precision=prec, deconvolve=rng.random() < 0.25,
                      deposit="fixed64" if rng.random() < 0.15 else "float")
            if kind == "run":
                steps = rng.randint(1, 5)
                c |= dict(stepper=rng.choice(["bullfrog", "fastpm"]), steps=steps, a_ini=a0,
                          a_end=round(a0 + 0.05 * steps, 3))
                what = rng.random()
                if what < 0.2:
                    c |= dict(grad_order=0, lap_order=0)
                elif what < 0.35:
                    nr = [m for m in MESHES if 0.3 * res <= m <= res and m <= 256]
                    if not nr:
                        continue
                    c |= dict(n=rng.choice(nr), n_resample=2, resampling=rng.choice(["fourier", "linear"]),
                              grad_order=rng.choice([0, grad]), antialias=rng.choice([0, 1]))
                elif what < 0.45:
                    c |= dict(lean=True, antialias=0)
                elif what < 0.55 and res % 64 == 0 and res <= 256:
                    c |= dict(net=True, precision=32, deposit="float", antialias=rng.choice([0, 1]))
        elif kind in ("ics", "gradient"):
            n = rng.choice([16, 32, 64, 128, 256])
            c = _case(kind=kind, n=n, res=n, L=L, precision=prec, worder=worder, grad_order=grad, lap_order=lap,
                      antialias=rng.choice([0, 0, 1]), steps=rng.randint(2, 10))
        elif kind == "train":
            n = rng.choice([64, 64, 128])
            c = _case(kind=kind, n=rng.randint(n // 2, n), res=n, L=L, worder=worder, grad_order=grad, a_ini=a0)
        else:
            res = rng.choice(MESHES[:11])
            n = rng.choice([m for m in MESHES if m <= res and 4 * m >= res and m <= 384])
            c = _case(kind=kind, n=n, res=res, L=L, precision=prec, bins=rng.randint(4, 64), a_ini=a0)
        points = (c["n"] * c["n_resample"]) ** 3 * c["precision"] // 8
        if _units(c) <= 0.8 * largest and points <= 4 * 512**3:  # in time and in memory
            return c


# ---------------------------------------------------------------------------------------- inputs
def _spectrum():
    """A CDM-like linear power spectrum with sigma_8 = 0.8, as the (k, P) table that the ICs take."""
    k = np.exp(np.linspace(math.log(1e-4), math.log(50.0), 512))
    q = k / 0.21
    t = np.log(1 + 2.34 * q) / (2.34 * q) * (1 + 3.89 * q + (16.1 * q) ** 2 + (5.46 * q) ** 3 + (6.71 * q) ** 4) ** -0.25
    p = k * t * t
    x = 8 * k
    w = 3 * (np.sin(x) - x * np.cos(x)) / x**3
    f = k**3 * p * w * w / (2 * math.pi**2)
    s8 = float(np.sum(0.5 * (f[1:] + f[:-1]) * np.diff(np.log(k))))
    return k, p * (0.64 / s8)


def _interp(x, xt, yt):
    xt, yt = (torch.as_tensor(v, dtype=torch.float64, device=x.device) for v in (xt, yt))
    i = torch.searchsorted(xt, x.clamp(xt[0], xt[-1]).contiguous()).clamp(1, len(xt) - 1)
    t = ((x - xt[i - 1]) / (xt[i] - xt[i - 1])).clamp(0, 1)
    return yt[i - 1] * (1 - t) + yt[i] * t


def _kaxes(n, L, nyquist=True):
    """Wavenumbers (kz, ky, kx) of rfftn's layout, shaped to broadcast; the Nyquist ones zeroed if asked."""
    dk = 2 * math.pi / L
    full = torch.arange(n, dtype=torch.float64, device=DEV)
    full = torch.where(full < n // 2, full, full - n) * dk
    half = torch.arange(n // 2 + 1, dtype=torch.float64, device=DEV) * dk
    if not nyquist:
        full[n // 2] = 0
        half[n // 2] = 0
    return full[:, None, None], full[None, :, None], half[None, None, :]


def _white(n, seed):
    return torch.randn((n, n, n), generator=torch.Generator(DEV).manual_seed(seed), dtype=torch.float64, device=DEV)


def _displaced(n, L, a, seed, dtype):
    """(Psi, Pi) of growing-mode matter at scale factor a: the linear displacement of a Gaussian field, its
    particles on the lattice of a grid of the next even size where n is odd."""
    m = n + n % 2
    w = torch.fft.rfftn(torch.randn((m, m, m), generator=torch.Generator(DEV).manual_seed(seed), device=DEV))
    kz, ky, kx = _kaxes(m, L, nyquist=False)
    k2 = kz**2 + ky**2 + kx**2
    amp = torch.sqrt(_interp(torch.sqrt(k2), *_spectrum()) * (m / L) ** 3) / k2.clamp_min(1e-30)
    amp[0, 0, 0] = 0
    amp = amp.float()
    psi1 = torch.stack([torch.fft.irfftn(w * (1j * k.float() * amp), s=(m, m, m))[:n, :n, :n] for k in (kx, ky, kz)])
    return (a * psi1).to(dtype).contiguous(), psi1.to(dtype).contiguous()


def _coefficients(c):
    """(dd1, alpha, beta, dd2) of the steps, uniform in the growth factor D = a of an Einstein-de Sitter universe."""
    a = np.linspace(c["a_ini"], c["a_end"], c["steps"] + 1)
    mid = 0.5 * (a[1:] + a[:-1])
    if c["stepper"] == "fastpm":
        alpha = (a[:-1] / a[1:]) ** 1.5
    else:
        d = np.diff(a)
        d2, d2p = -3 / 7 * a**2, -6 / 7 * a
        b = (d2[:-1] + d2p[:-1] * d / 2) / mid - mid
        alpha = (d2p[1:] - b) / (d2p[:-1] - b)
    return [np.ascontiguousarray(v) for v in (mid - a[:-1], alpha, (1 - alpha) / mid, a[1:] - mid)]


def _net_params(seed):
    """He-normal weights of the correction's four layers (27 taps, 2-16-16-16-1 channels), small biases."""
    rng = np.random.default_rng(seed)
    layers = []
    for i, (co, ci) in enumerate([(16, 2), (16, 16), (16, 16), (1, 16)]):
        w, b = np.zeros((27, 16, 16), np.float32), np.zeros(16, np.float32)
        w[:, :co, :ci] = rng.normal(scale=math.sqrt((2.0 if i < 3 else 0.1) / (27 * ci)), size=(27, co, ci))
        b[:co] = rng.normal(scale=0.02, size=co)
        layers += [w.reshape(-1), b]
    return np.concatenate(layers)


def _net_scale(c):
    return 0.1 * (c["L"] / c["res"]) ** 2


def _edges(c):
    kf = 2 * math.pi / c["L"]
    return np.exp(np.linspace(math.log(0.987 * kf), math.log(0.991 * kf * c["res"] / 2), c["bins"] + 1))


def _config(c):
    return D.PMConfig(res_pm=c["res"], n_part=c["n"], boxsize=c["L"], worder=c["worder"], deconvolve=c["deconvolve"],
                      antialias=c["antialias"], grad_order=c["grad_order"], lap_order=c["lap_order"],
                      n_resample=c["n_resample"], resampling=c["resampling"])


def _dtype(c):
    return torch.float64 if c["precision"] == 64 else torch.float32


class _State:
    """A solver with what its user keeps beside it: device tensors, coefficient arrays, tables."""

    def __init__(self, c):
        self.c = c
        self.S = D.PMSolverHIP(_config(c), precision=c["precision"], deposit=c["deposit"], lean=c["lean"])
        self.L, self.ctx = D.lib(), self.S._ctx

    def ok(self, rc):
        if rc:
            raise RuntimeError(self.L.dj_last_error(self.ctx).decode())


def _snapshot(c, seed):
    """A training snapshot: the displacement and the force of a mesh twice as fine, as host arrays."""
    psi, _ = _displaced(c["n"], c["L"], c["a_ini"], seed, torch.float32)
    acc = _force(dict(c, res=2 * c["res"]), psi.double())
    return psi.cpu().numpy(), acc.float().cpu().numpy()


def prepare(case, seed):
    c = case
    s = _State(c)
    if c["kind"] == "accel":
        s.psi = _displaced(c["n"], c["L"], c["a_ini"], seed, _dtype(c))[0].cpu().numpy()
    if c["kind"] in ("run", "spectra"):
        s.psi, s.pi = _displaced(c["n"], c["L"], c["a_ini"], seed, _dtype(c))
        s.psi_out, s.pi_out = torch.empty_like(s.psi), torch.empty_like(s.pi)
        if c["net"]:
            s.S.nn_set_params(_net_params(seed))
            s.S.nn_enable(True, _net_scale(c))
            a = np.linspace(c["a_ini"], c["a_end"], c["steps"] + 1)
            s.S.nn_set_schedule(0.5 * (a[1:] + a[:-1]))
    if c["kind"] in ("run", "gradient"):
        s.coef = _coefficients(c)
        s.coef_ptr = [a.ctypes.data for a in s.coef]
    if c["kind"] in ("ics", "gradient"):
        s.white = _white(c["n"], seed)
        s.k, s.p = (np.ascontiguousarray(v) for v in _spectrum())
        s.table = (s.k.ctypes.data, s.p.ctypes.data, len(s.k), c["a_ini"], 2)
        if c["kind"] == "gradient":
            s.target = 0.3 * _white(c["res"], seed + 7919)
            s.white_bar = torch.empty_like(s.white)
        else:
            s.psi_out = torch.empty((3, c["n"], c["n"], c["n"]), dtype=_dtype(c), device=DEV)
            s.pi_out = torch.empty_like(s.psi_out)
    if c["kind"] == "train":
        s.psi, s.acc = _snapshot(c, seed)
        s.weight = 1.0 / float(np.mean(s.acc.astype(np.float64) ** 2))
        s.params = _net_params(seed)
        s.S.nn_enable(False)
    if c["kind"] == "spectra":
        s.edges = _edges(c)
    torch.cuda.synchronize()
    return s


def run(state):
    s, c, L, ctx = state, state.c, state.L, state.ctx
    if c["kind"] == "accel":
        return {"acc": s.S.pm_acceleration(s.psi)}
    if c["kind"] == "run":
        s.ok(L.dj_set_state_device(ctx, s.psi.data_ptr(), s.pi.data_ptr()))
        s.ok(L.dj_run(ctx, c["steps"], *s.coef_ptr, None, D._lib.STEP_CB(), None))
        s.ok(L.dj_get_state_device(ctx, s.psi_out.data_ptr(), s.pi_out.data_ptr()))
        return {"psi": s.psi_out, "pi": s.pi_out}
    if c["kind"] == "ics":
        s.ok(L.dj_ics_lpt_device(ctx, 42, s.white.data_ptr(), *s.table))
        s.ok(L.dj_get_state_device(ctx, s.psi_out.data_ptr(), s.pi_out.data_ptr()))
        return {"psi": s.psi_out, "pi": s.pi_out}
    if c["kind"] == "gradient":
        loss = C.c_double()
        s.ok(L.dj_ics_lpt_device(ctx, 42, s.white.data_ptr(), *s.table))
        s.ok(L.dj_run_checkpointed(ctx, c["steps"], *s.coef_ptr))
        s.ok(L.dj_density_loss_device(ctx, s.target.data_ptr(), C.byref(loss)))
        s.ok(L.dj_vjp_run(ctx, None, None))
        s.ok(L.dj_vjp_ics_lpt_device(ctx, 42, s.white.data_ptr(), *s.table, s.white_bar.data_ptr()))
        # FP64 arrays that carry the accuracy of the steps' precision, and are kept in it
        return {"loss": s.S.dtype(loss.value), "white_bar": s.white_bar.to(_dtype(c))}
    if c["kind"] == "train":
        s.S.nn_set_params(s.params)
        s.S.nn_enable(True, _net_scale(c))
        loss = s.S.nn_train_step(s.psi, s.acc, c["a_ini"], 1e-3, 1, weight=s.weight)
        return {"loss": np.float32(loss), "params": s.S.nn_get_params()}
    if c["kind"] == "spectra":
        s.ok(L.dj_set_state_device(ctx, s.psi.data_ptr(), s.pi.data_ptr()))
        k, pd, pp = s.S.power_spectra_binned(s.edges)
        return {"k": k, "density": pd.astype(s.S.dtype), "displacement": pp.astype(s.S.dtype)}
    raise ValueError(c["kind"])


# ---------------------------------------------------------------------------------------- work
def work(case):
    """Bytes: the arrays that a pass takes and gives, the state once more per step, and the density and the
    potential of every force pass once.  Flops: the transforms, 3 per deposited weight, 2 per gathered
    finite-difference term, and the net's multiply-adds."""
    c = case
    T, M, P, W = c["precision"] // 8, c["res"] ** 3, c["n"] ** 3, c["worder"]
    ns = 1 if c["antialias"] in (0, -1) else 2 if c["antialias"] == 1 else 8
    fft = lambda m: 2.5 * m**3 * math.log2(m**3)  # noqa: E731
    net = 2 * 27 * (2 * 16 + 2 * 256 + 16) * M
    force_b = ns * (2 * M * T + 6 * P * T)
    force_f = ns * (fft(c["res"]) * (4 if c["grad_order"] == 0 else 2) + P * W**3 * (3 * c["n_resample"] ** 3 + 6 + 6 * c["grad_order"]))
    if c["n_resample"] > 1 and c["resampling"] == "fourier":
        force_f += ns * 3 * fft(c["n"]) * c["n_resample"] ** 3
    if c["net"]:
        force_f += ns * net
    ics_b, ics_f = P * 8 + 6 * P * T, 7 * fft(c["n"]) + 10 * fft(3 * c["n"] / 2)
    if c["kind"] == "accel":
        return {"bytes": force_b, "flops": force_f}
    if c["kind"] == "run":
        return {"bytes": 12 * P * T + c["steps"] * (12 * P * T + force_b), "flops": c["steps"] * (force_f + 12 * P)}
    if c["kind"] == "ics":
        return {"bytes": ics_b, "flops": ics_f}
    if c["kind"] == "gradient":
        return {"bytes": 2 * ics_b + c["steps"] * (36 * P * T + 4 * force_b) + 2 * M * T,
                "flops": 2 * ics_f + c["steps"] * 4 * force_f}
    if c["kind"] == "train":
        return {"bytes": 2 * force_b + 6 * P * T + 2 * 4 * 27712, "flops": 2 * force_f + 3 * net}
    return {"bytes": 12 * P * T + 2 * M * T, "flops": fft(c["res"]) + 3 * fft(c["n"]) + 3 * 8 * P}


# ---------------------------------------------------------------------------------------- 64-bit results
def _weights(W, d):
    if W == 2:
        return (1 - d).clamp_min(0)
    if W == 3:
        return torch.where(d <= 0.5, 0.75 - d * d, 0.5 * (1.5 - d).clamp_min(0) ** 2)
    return torch.where(d <= 1, (4 - 6 * d * d + 3 * d**3) / 6, (2 - d).clamp_min(0) ** 3 / 6)


def _stencil(X, W, N, L):
    """For every cell of the mass-assignment stencil of the points X (3, m): its index and its weight."""
    cells, ws = [], []
    for x in X:
        g = torch.remainder(x, L) / L * N
        b = (torch.floor(g) if W % 2 == 0 else torch.round(g)).detach()
        off = [b + (o - (0 if W == 2 else 1)) for o in range(W)]
        cells.append([torch.remainder(o, N).long() for o in off])
        ws.append([_weights(W, (g - o).abs()) for o in off])
    for i in range(W):
        for j in range(W):
            wij, cij = ws[2][i] * ws[1][j], N * (cells[1][j] + N * cells[2][i])
            for k in range(W):
                yield cij + cells[0][k], wij * ws[0][k]


_CHUNK = 1 << 24


def _deposit(X, W, N, L):
    mesh = torch.zeros(N**3, dtype=torch.float64, device=X.device)
    for at in range(0, X.shape[1], _CHUNK):
        for idx, w in _stencil(X[:, at:at + _CHUNK], W, N, L):
            mesh = mesh.index_add(0, idx, w) if w.requires_grad else mesh.index_add_(0, idx, w)
    return mesh.reshape(N, N, N)


def _gather(fields, X, W, L):
    N, out = fields[0].shape[0], []
    for at in range(0, X.shape[1], _CHUNK):
        acc = [0.0] * len(fields)
        for idx, w in _stencil(X[:, at:at + _CHUNK], W, N, L):
            for i, f in enumerate(fields):
                acc[i] = acc[i] + w * f.reshape(-1).index_select(0, idx)
        out.append(torch.stack(acc))
    return torch.cat(out, 1)


def _points(c, psi, q, shift):
    """The extra point sets of sheet resampling: the interpolated displacement at every offset of the lattice."""
    n, L, nr = c["n"], c["L"], c["n_resample"]
    wrapped = [torch.remainder(psi[a] + shift[a] + L / 2, L) - L / 2 for a in range(3)]  # [k, j, i]
    m = torch.arange(n, dtype=torch.float64, device=DEV)
    full, half = torch.where(m < n // 2, m, m - n) / n, torch.arange(n // 2 + 1, dtype=torch.float64, device=DEV) / n
    hat = [torch.fft.rfftn(w.permute(2, 1, 0)) for w in wrapped] if c["resampling"] == "fourier" else None
    for o in range(1, nr**3):
        d = [(o // nr**2) / nr, (o // nr % nr) / nr, (o % nr) / nr]
        X = []
        for a in range(3):
            if hat is not None:
                ph = [torch.exp(2j * math.pi * v * e) for v, e in zip((full, full, half), d)]
                h = torch.fft.ifftn(hat[a] * ph[0][:, None, None] * ph[1][None, :, None] * ph[2], dim=(0, 1))
                h[..., 0].imag.zero_()
                h[..., -1].imag.zero_()
                f = torch.fft.irfft(h, n=n, dim=2).permute(2, 1, 0)
            else:
                f = wrapped[a]
                for dim, e in ((2, d[0]), (1, d[1]), (0, d[2])):
                    f = (1 - e) * f + e * torch.roll(f, -1, dim)
            X.append(torch.remainder(q[a] + f + d[a] * L / n + L, L).reshape(-1))
        yield torch.stack(X)


def _net_potential(params, dens, a, rho):
    """The learned correction's potential of a density mesh: four 3x3x3 convolutions, two of them residual."""
    N = dens.shape[0]
    p = params.reshape(4, -1)
    x = torch.stack([torch.log1p((dens / rho - 1).clamp_min(-0.999)), torch.full_like(dens, a)], -1)

    def conv(x, layer, co):
        w, b = p[layer, :27 * 256].reshape(27, 16, 16), p[layer, 27 * 256:]
        ci, out = x.shape[-1], b[:co].expand(N, N, N, co)
        for t in range(27):
            out = out + torch.roll(x, (1 - t // 9, 1 - t // 3 % 3, 1 - t % 3), (0, 1, 2)) @ w[t, :co, :ci].T
        return out

    h = torch.relu(conv(x, 0, 16))
    h = h + torch.relu(conv(h, 1, 16))
    h = h + torch.relu(conv(h, 2, 16))
    return conv(h, 3, 1)[..., 0]


def _shifts(c):
    d, aa = 0.5 * c["L"] / c["res"], c["antialias"]
    if aa in (0, -1):
        return [[-aa * d] * 3]
    if aa == 1:
        return [[0.0] * 3, [d] * 3]
    return [[x, y, z] for x in (0.0, d) for y in (0.0, d) for z in (0.0, d)]


def _force(c, psi, net=None):
    """-grad phi at the particles, nabla^2 phi = delta, in 64 bits; net: (parameters, scale, a) of the correction."""
    n, N, L, W = c["n"], c["res"], c["L"], c["worder"]
    axis = torch.arange(n, dtype=torch.float64, device=psi.device) * (L / n)
    q = [axis[None, None, :], axis[None, :, None], axis[:, None, None]]
    kz, ky, kx = _kaxes(N, L)
    if c["lap_order"] == 0:
        den = -(kz**2 + ky**2 + kx**2)
    else:
        tap = {2: (2, -2), 4: (-15 / 6, 16 / 6, -1 / 6), 6: (-245 / 90, 270 / 90, -27 / 90, 2 / 90)}[c["lap_order"]]
        h = L / N
        sym = (lambda k: -4 * torch.sin(k * h / 2) ** 2 / h**2) if c["lap_order"] == 2 else (
            lambda k: sum(t * torch.cos(i * k * h) for i, t in enumerate(tap)) / h**2)
        den = sym(kz) + sym(ky) + sym(kx)
    den[0, 0, 0] = 1
    kern = 1 / den
    kern[0, 0, 0] = 0
    if c["deconvolve"]:
        for k in (kz, ky, kx):
            kern = kern * torch.sinc(k * L / (2 * math.pi * N)) ** (-2 * W)
    total, shifts = 0.0, _shifts(c)
    for s in shifts:
        X = torch.stack([(psi[a] + q[a] + s[a]).reshape(-1) for a in range(3)])
        dens = _deposit(X, W, N, L)
        if c["n_resample"] > 1:
            for P in _points(c, psi, q, s):
                dens = dens + _deposit(P, W, N, L)
        rho = n**3 * c["n_resample"] ** 3 / N**3
        spec = torch.fft.rfftn(dens) * kern / rho
        if c["grad_order"] == 0:
            acc = torch.cat([_gather([torch.fft.irfftn(spec * (-1j * k), s=(N, N, N))], X, W, L)
                             for k in reversed(_kaxes(N, L, nyquist=False))])
        else:
            phi = torch.fft.irfftn(spec, s=(N, N, N))
            del spec
            if net is not None:
                phi = phi + net[1] * _net_potential(net[0], dens, net[2], rho)
            taps = {2: (1 / 2,), 4: (8 / 12, -1 / 12), 6: (45 / 60, -9 / 60, 1 / 60)}[c["grad_order"]]
            comps = []
            for dim in (2, 1, 0):
                f = sum(t * N / L * (torch.roll(phi, i + 1, dim) - torch.roll(phi, -i - 1, dim)) for i, t in enumerate(taps))
                comps.append(_gather([f], X, W, L))
                del f
            acc = torch.cat(comps)
        total = total + acc.reshape(psi.shape) / len(shifts)
    return total


def _step(c, i, psi, pi, net=None):
    dd1, alpha, beta, dd2 = (float(v[i]) for v in _coefficients(c))
    psi = psi + dd1 * pi
    pi = alpha * pi + beta * _force(c, psi, net)
    return psi + dd2 * pi, pi


def _lpt(c, white):
    """2LPT (Psi, Pi) at growth factor a_ini of the white noise, the second order on a 3/2 grid."""
    n, L, Dg = c["n"], c["L"], c["a_ini"]
    ext, h = 3 * n // 2, n // 2
    kz, ky, kx = _kaxes(n, L)
    k2 = kz**2 + ky**2 + kx**2
    k2[0, 0, 0] = 1
    amp = -torch.sqrt(_interp(torch.sqrt(k2), *_spectrum()) * (n / L) ** 3) / k2
    amp[0, 0, 0] = 0
    phi = torch.fft.rfftn(white) * amp
    kd, ke = _kaxes(n, L, nyquist=False)[::-1], _kaxes(ext, L, nyquist=False)[::-1]
    f1 = [-1j * k * phi for k in kd]
    sides = [(slice(0, h), slice(0, h)), (slice(h + 1, n), slice(ext - h + 1, ext))]

    def pad(f):
        g = torch.zeros((ext, ext, ext // 2 + 1), dtype=f.dtype, device=f.device)
        for a, b in sides:
            for e, d in sides:
                g[b, d, :h] = f[a, e, :h] * (ext / n) ** 3
        return g

    A = [[torch.fft.irfftn(1j * ke[k] * pad(f1[i]), s=(ext,) * 3) for k in range(3)] for i in range(3)]
    mu = A[0][0] * A[1][1] + A[0][0] * A[2][2] + A[1][1] * A[2][2] - A[0][1] * A[1][0] - A[0][2] * A[2][0] - A[1][2] * A[2][1]
    g = torch.fft.rfftn(-3 / 7 * mu)
    f2 = torch.zeros_like(phi)
    for a, b in sides:
        for e, d in sides:
            f2[a, e, :h] = g[b, d, :h] * (n / ext) ** 3
    psi1 = torch.stack([torch.fft.irfftn(f, s=(n,) * 3) for f in f1])
    psi2 = torch.stack([torch.fft.irfftn(-1j * k / k2 * f2, s=(n,) * 3) for k in kd])
    return Dg * psi1 + Dg**2 * psi2, psi1 + 2 * Dg * psi2


def _binned(field, L, edges, window):
    """Sum of |f_k|^2 / window and number of the modes of every bin, over the whole spectrum."""
    N = field.shape[0]
    ks = _kaxes(N, L)
    f = torch.fft.rfftn(field)
    v = f.real**2 + f.imag**2
    if window:
        for k in ks:
            v = v / torch.sinc(k * L / (2 * math.pi * N)) ** (2 * window)
    k = torch.sqrt(ks[0] ** 2 + ks[1] ** 2 + ks[2] ** 2).reshape(-1)
    w = torch.full((N // 2 + 1,), 2.0, dtype=torch.float64, device=DEV)
    w[0] = w[-1] = 1
    w = w.expand(N, N, N // 2 + 1).reshape(-1)
    b = torch.bucketize(k, torch.as_tensor(edges, device=DEV), right=True)
    n = len(edges) + 1
    total = torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, b, w * v.reshape(-1))
    modes = torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, b, w)
    return total[1:-1], modes[1:-1]


def exact(case, seed):
    c = case
    if c["kind"] == "accel":
        return {"acc": _force(c, _displaced(c["n"], c["L"], c["a_ini"], seed, _dtype(c))[0].double())}
    if c["kind"] == "run":
        psi, pi = (v.double() for v in _displaced(c["n"], c["L"], c["a_ini"], seed, _dtype(c)))
        net = torch.as_tensor(_net_params(seed), device=DEV).double() if c["net"] else None
        a = np.linspace(c["a_ini"], c["a_end"], c["steps"] + 1)
        for i in range(c["steps"]):
            psi, pi = _step(c, i, psi, pi, None if net is None else (net, _net_scale(c), 0.5 * (a[i] + a[i + 1])))
        return {"psi": psi, "pi": pi}
    if c["kind"] == "ics":
        psi, pi = _lpt(c, _white(c["n"], seed))
        return {"psi": psi, "pi": pi}
    if c["kind"] == "gradient":
        from torch.utils.checkpoint import checkpoint

        white, target = _white(c["n"], seed).requires_grad_(True), 0.3 * _white(c["res"], seed + 7919)
        psi, pi = _lpt(c, white)
        for i in range(c["steps"]):
            psi, pi = checkpoint(lambda x, p, i=i: _step(c, i, x, p), psi, pi, use_reentrant=False)
        axis = torch.arange(c["n"], dtype=torch.float64, device=DEV) * (c["L"] / c["n"])
        X = [psi[0] + axis, psi[1] + axis[:, None], psi[2] + axis[:, None, None]]
        mesh = _deposit(torch.stack([x.reshape(-1) for x in X]), c["worder"], c["res"], c["L"])
        loss = ((mesh * (c["res"] / c["n"]) ** 3 - 1 - target) ** 2).sum()
        return {"loss": float(loss.detach()), "white_bar": torch.autograd.grad(loss, white)[0]}
    if c["kind"] == "train":
        psi, acc = _snapshot(c, seed)
        p = torch.as_tensor(_net_params(seed), device=DEV).double().requires_grad_(True)
        tgt = torch.as_tensor(acc, device=DEV).double()
        weight = 1.0 / float(np.mean(acc.astype(np.float64) ** 2))
        f = _force(c, torch.as_tensor(psi, device=DEV).double(), (p, _net_scale(c), c["a_ini"]))
        loss = weight * ((f - tgt) ** 2).mean()
        g = torch.autograd.grad(loss, p)[0]
        m, v = 0.1 * g / (1 - 0.9), 0.001 * g * g / (1 - 0.999)
        return {"loss": float(loss.detach()), "params": (p - 1e-3 * m / (torch.sqrt(v) + 1e-8)).detach()}
    psi = _displaced(c["n"], c["L"], c["a_ini"], seed, _dtype(c))[0].double()
    n, N, L, edges = c["n"], c["res"], c["L"], _edges(c)
    axis = torch.arange(n, dtype=torch.float64, device=DEV) * (L / n)
    X = torch.stack([v.reshape(-1) for v in (psi[0] + axis, psi[1] + axis[:, None], psi[2] + axis[:, None, None])])
    s, m = _binned(_deposit(X, 2, N, L), L, edges, 2)
    density = torch.where(m > 0, L**3 * s / m.clamp_min(1) / n**6, 0.0)
    s, m = map(sum, zip(*(_binned(p, L, edges, 0) for p in psi)))
    return {"k": np.sqrt(edges[1:] * edges[:-1]), "density": density,
            "displacement": torch.where(m > 0, 3 * L**3 * s / m.clamp_min(1) / n**6, 0.0)}
