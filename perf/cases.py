"""Performance cases: what a user of this framework has it do.

Each case is one call of a public entry point on a dataset that has been
preprocessed (``reconstruct()`` of the single-slice and mixed-state classes,
the batched runner) or uploaded (the differentiable loss): the sizes are those
of the package's own workloads (32 x 32 scans of 64 px frames at 0.2 A,
128 x 128 scans of 128 px frames at 0.1 A with mini-batches of 1024, 64
uneven problems side by side) and their neighbours, down to 32 px frames and
up to 256 px ones.

The datasets are simulated here with torch, seeded: a smooth random phase
object, a defocused probe of 20 mrad at 300 keV, a raster scan with a few
hundredths of an Angstrom of jitter and Poisson counts.  Reconstructions start
from a non-flat estimate of the object and a probe with the wrong defocus, as
a run that continues an earlier one does.
"""

from __future__ import annotations

import math

import numpy as np
import torch

ENERGY, SEMIANGLE, DEFOCUS = 300e3, 20.0, 200.0
WAVELENGTH = 0.0196874747  # Angstrom at 300 keV
PIXEL = {32: 0.4, 64: 0.2, 128: 0.1, 256: 0.05}   # Angstrom per pixel at each frame size
STEP = {32: 1.0, 64: 1.0, 128: 0.4, 256: 0.4}     # scan step in Angstrom
COUNTS = 1e5                                      # mean counts per pattern


def _case(name, solver, S, nx, ny, iters, batch=0, fix_probe=False, **more):
    c = dict(name=name, solver=solver, S=S, nx=nx, ny=ny, iters=iters, batch=batch,
             fix_probe=fix_probe, modes=1, sigma=0.0, q_lowpass=0.0, q_highpass=0.0, problems=1,
             object_px=0)
    c.update(more)
    return c


def listed():
    return [
        # a quick look at binned patterns: the smallest calls, where launches
        # and the host's part count
        _case("binned_32px", "gd", 32, 16, 16, 4, batch=64, object_px=128),
        # the small configuration: full batch, known probe, 8 iterations
        _case("small_64px", "gd", 64, 32, 32, 8, fix_probe=True, object_px=256),
        # the production configuration: seeded mini-batches, probe refined
        _case("production_128px", "gd", 128, 128, 128, 4, batch=1024, object_px=720),
        # an ordinary dataset as it comes off the microscope: uneven scan,
        # uneven batches, object size by the default rule
        _case("uneven_64px", "gd", 64, 61, 47, 4, batch=300),
        # large frames
        _case("large_frames_256px", "gd", 256, 24, 21, 2, batch=168),
        # scan positions refined beside object and probe
        _case("positions_128px", "positions", 128, 48, 48, 2, batch=768),
        # partially coherent illumination: three probe modes
        _case("mixed_128px", "mixed", 128, 40, 40, 2, batch=400, modes=3),
        # difference map, every position at once
        _case("difference_map_128px", "projection", 128, 56, 53, 2),
        # weak phase object as a real potential, smoothed every iteration
        _case("potential_64px", "potential", 64, 45, 45, 4, batch=512, sigma=0.3),
        # object band-limited and smoothed every iteration
        _case("filtered_128px", "gd", 128, 40, 37, 3, batch=740, sigma=0.15, q_lowpass=2.5,
              q_highpass=0.02),
        # gradients for an optimiser or a network of the user's own
        _case("loss_gradients_128px", "loss", 128, 48, 43, 1),
        # many small uneven problems side by side
        _case("many_problems", "many", 64, 30, 33, 4, problems=12),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    solver = rng.choice(["gd", "gd", "gd", "gd", "positions", "mixed", "projection", "potential",
                         "loss", "many", "filtered"])
    S = rng.choice([32, 64, 64, 128, 128, 256] if solver in ("gd", "potential")
                   else [64, 128] if solver == "many" else [32, 64, 128])
    modes = rng.randint(2, 4) if solver == "mixed" else 1
    iters = 1 if solver == "loss" else rng.randint(1, 8)
    problems = rng.randint(2, 16) if solver == "many" else 1
    # pixels of all patterns together, iterations and modes counted: below a
    # quarter of the largest listed case's
    most = (128 * 128 * 128 * 128 * 4) // 4 // (S * S * iters * modes * problems)
    edge = max(8, min(96, int(math.sqrt(most))))
    nx, ny = _log_int(rng, 8, edge), _log_int(rng, 8, edge)
    n = nx * ny
    batch = 0
    if solver in ("gd", "mixed", "positions", "potential", "filtered") and rng.random() < 0.75:
        # at most 48 mini-batches in all: the listed cases have up to 64
        batch = min(n, max(8, -(-n * iters // 48), _log_int(rng, 24, 1200)))
    c = _case("", solver, S, nx, ny, iters, batch=batch, modes=modes, problems=problems,
              fix_probe=solver in ("gd", "projection", "potential") and rng.random() < 0.25)
    if solver == "filtered":
        c.update(solver="gd", sigma=rng.choice([0.0, 1.0, 2.0]) * PIXEL[S],
                 q_lowpass=rng.uniform(0.2, 0.4) / PIXEL[S],
                 q_highpass=rng.choice([0.0, 0.02]))
    elif solver == "potential":
        c.update(sigma=rng.choice([0.0, 1.0, 1.5]) * PIXEL[S])
    del c["name"]
    return c


# -- simulated dataset ---------------------------------------------------------

def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _fidx(n):
    return np.fft.fftfreq(n, 1.0 / n).astype(np.int64)


def _smooth_field(shape, sigma_px, rng):
    """Gaussian-smoothed white noise (periodic), scaled to [0, 1]."""
    kx, ky = np.fft.fftfreq(shape[0]), np.fft.fftfreq(shape[1])
    low = np.exp(-2 * (np.pi * sigma_px) ** 2 * (kx[:, None] ** 2 + ky[None, :] ** 2))
    f = np.fft.ifft2(np.fft.fft2(rng.standard_normal(shape)) * low).real
    return (f - f.min()) / (f.max() - f.min())


def _probe(S, defocus, counts):
    """Corner-centred defocused probe, sum |fft2 P|^2 = counts (complex128)."""
    q = np.fft.fftfreq(S, PIXEL[S])
    alpha = np.hypot(q[:, None], q[None, :]) * WAVELENGTH
    edge = 2.0 * WAVELENGTH / (S * PIXEL[S])
    aperture = np.clip((SEMIANGLE * 1e-3 - alpha) / edge + 0.5, 0, 1)
    chi = math.pi / WAVELENGTH * alpha ** 2 * -defocus
    p = np.fft.ifft2(aperture * np.exp(-1j * chi))
    return p * math.sqrt(counts / np.sum(np.abs(np.fft.fft2(p)) ** 2))


def _shifted_probe(probe, frac):
    """ifft2(fft2(probe) * ramp) of complex probe (..., S, S) at frac [n, 2]."""
    S = probe.shape[-1]
    k = torch.fft.fftfreq(S, dtype=torch.float64, device=probe.device)
    f = frac.to(torch.float64)
    ramp = torch.exp(-2j * math.pi * (k[None, :, None] * f[:, 0, None, None]
                                      + k[None, None, :] * f[:, 1, None, None]))
    return torch.fft.ifft2(torch.fft.fft2(probe) * ramp.to(probe.dtype))


def _windows(pos, S, shape):
    """Flat object indices of the patches [n, S, S] and the sub-pixel parts."""
    r = torch.round(pos)
    off = torch.from_numpy(_fidx(S)).to(pos.device)
    rows = (r[:, 0].long()[:, None] + off[None, :]) % shape[0]
    cols = (r[:, 1].long()[:, None] + off[None, :]) % shape[1]
    return rows[:, :, None] * shape[1] + cols[:, None, :], pos - r


def _scene(case, seed):
    """Everything simulated for one problem: host arrays and device counts."""
    S, nx, ny = case["S"], case["nx"], case["ny"]
    px, step = PIXEL[S], STEP[S]
    rng = np.random.default_rng([seed, S, nx, ny])
    x, y = np.meshgrid(np.arange(nx) * step, np.arange(ny) * step, indexing="ij")
    ang = np.stack([x.ravel(), y.ravel()], -1) + rng.uniform(0.0, 0.1, (nx * ny, 2))
    pos = ang / px + S / 2
    if case["object_px"]:
        shape = (case["object_px"],) * 2
    else:
        shape = tuple(int(max(round(v + S / 2), S)) for v in np.round(pos.max(0)))
    pos32 = pos.astype(np.float32)
    pos32 -= pos32.mean(0) - np.array(shape) / 2

    field = _smooth_field(shape, 0.4 / px, rng)
    truth = np.exp(1j * 0.6 * field)
    probe_true = _probe(S, DEFOCUS, COUNTS)
    # the scan the microscope made differs a little from the one recorded
    moved = pos32 + (rng.normal(0, 0.3, pos32.shape).astype(np.float32)
                     if case["solver"] == "positions" else np.float32(0))
    dev = _device()
    counts = _simulate(truth, probe_true, moved, seed, dev)

    # starting values: the object at half contrast with some noise, the probe
    # at a defocus 10 A off
    noise = _smooth_field(shape, 2.0, rng) - 0.5
    guess = (0.92 + 0.06 * _smooth_field(shape, 3.0, rng)) * np.exp(1j * (0.3 * field + 0.2 * noise))
    if case["solver"] == "potential":
        guess = 0.3 * field + 0.1 * np.abs(noise)
    probe = _probe(S, DEFOCUS + 10.0, COUNTS)
    if case["solver"] == "mixed":
        k = np.fft.fftfreq(S)
        modes = [probe]
        for m in range(1, case["modes"]):
            modes.append(modes[-1] * 0.6 * np.exp(2j * np.pi * rng.uniform(-0.5, 0.5) * k)[:, None]
                         * np.exp(2j * np.pi * rng.uniform(-0.5, 0.5) * k)[None, :])
        probe = np.stack(modes)
        probe *= math.sqrt(COUNTS / np.sum(np.abs(np.fft.fft2(probe)) ** 2))
    # the region the scan covers, a quarter of a frame beyond its edge
    mask = np.zeros(shape, dtype=bool)
    lo = np.maximum(np.floor(pos32.min(0) - S / 4).astype(int), 0)
    hi = np.ceil(pos32.max(0) + S / 4).astype(int)
    mask[lo[0]:hi[0], lo[1]:hi[1]] = True
    return dict(positions_ang=ang, positions=pos32, shape=shape, counts=counts,
                object=guess.astype(np.float32 if case["solver"] == "potential" else np.complex64),
                probe=probe.astype(np.complex64), mask=mask)


def _simulate(obj, probe, pos32, seed, dev):
    """Poisson counts [N, S, S] float32 on the device, corner-centred."""
    S, n = probe.shape[0], len(pos32)
    o = torch.from_numpy(obj).to(dev).to(torch.complex64).reshape(-1)
    p = torch.from_numpy(probe).to(dev).to(torch.complex64)
    pos = torch.from_numpy(pos32).to(dev)
    gen = torch.Generator(device=dev)
    gen.manual_seed(int(seed) + 1)
    out = torch.empty((n, S, S), dtype=torch.float32, device=dev)
    for s in range(0, n, 2048):
        idx, frac = _windows(pos[s:s + 2048], S, obj.shape)
        psi = _shifted_probe(p[None], frac) * o[idx]
        out[s:s + 2048] = torch.poisson(torch.fft.fft2(psi).abs() ** 2, generator=gen)
    return out


def _parts(case, seed):
    """The single problems of a case: (case, seed) of each."""
    if case["solver"] != "many":
        return [(case, seed)]
    out = []
    for i in range(case["problems"]):
        # every second problem has the other frame size and a smaller scan;
        # scan edges differ from problem to problem
        S = case["S"] if i % 2 == 0 else (128 if case["S"] == 64 else 64)
        nx = max(8, case["nx"] - 2 * i if i % 3 else case["nx"])
        ny = max(8, case["ny"] - i)
        out.append((dict(case, solver="gd", S=S, nx=nx, ny=ny, problems=1), seed * 1000 + i))
    return out


# -- prepare and run -------------------------------------------------------------

def _reconstruction(case, seed):
    from py4dstem_amd import MixedstatePtychography, SingleslicePtychography
    from py4dstem_amd.datacube import Calibration, DataCube
    w = _scene(case, seed)
    S, px = case["S"], PIXEL[case["S"]]
    data = torch.fft.fftshift(w["counts"], dim=(-2, -1)).cpu().numpy()
    dc = DataCube(data.reshape(case["nx"], case["ny"], S, S),
                  Calibration(R_pixel_size=STEP[S], R_pixel_units="A",
                              Q_pixel_size=1.0 / (S * px), Q_pixel_units="A^-1"))
    cls = MixedstatePtychography if case["solver"] == "mixed" else SingleslicePtychography
    kind = "potential" if case["solver"] == "potential" else "complex"
    p = cls(ENERGY, datacube=dc, semiangle_cutoff=SEMIANGLE, initial_object_guess=w["object"],
            initial_probe_guess=w["probe"], initial_scan_positions=w["positions_ang"],
            object_type=kind, verbose=False)
    p.preprocess(force_com_rotation=0, force_com_transpose=False, force_com_shifts=(S / 2, S / 2),
                 object_fov_mask=w["mask"], plot_center_of_mass=False, plot_rotation=False,
                 plot_probe_overlaps=False)
    p.attach_datacube(None)  # the patterns are on the GPU now
    return p


def _options(case, seed):
    kw = dict(num_iter=case["iters"], max_batch_size=case["batch"] or None, seed_random=int(seed),
              fix_probe=case["fix_probe"], progress_bar=False, reset=True)
    if case["solver"] == "positions":
        kw.update(fix_positions=False)
    if case["solver"] == "mixed":
        kw.update(orthogonalize_probe=False)
    if case["solver"] == "projection":
        kw.update(reconstruction_method="DM_AP", reconstruction_parameter=0.5)
    if case["sigma"]:
        kw.update(gaussian_filter_sigma=case["sigma"])
    if case["q_lowpass"] or case["q_highpass"]:
        kw.update(q_lowpass=case["q_lowpass"] or None, q_highpass=case["q_highpass"] or None)
    return kw


def prepare(case, seed):
    if case["solver"] == "loss":
        from py4dstem_amd import kernels
        w = _scene(case, seed)
        dev = w["counts"].device
        return dict(kind="loss",
                    object=torch.from_numpy(w["object"]).to(dev).requires_grad_(),
                    probe=torch.from_numpy(w["probe"]).to(dev).requires_grad_(),
                    positions=torch.from_numpy(w["positions"]).to(dev),
                    amplitudes=kernels.to_kernel_layout(torch.sqrt(w["counts"])))
    if case["solver"] == "many":
        from py4dstem_amd.multi import MultiPtychography
        parts = _parts(case, seed)
        kw = [_options(c, s) for c, s in parts]
        for k in kw:
            for fixed in ("num_iter", "progress_bar"):
                del k[fixed]
        return dict(kind="many", iters=case["iters"], options=kw,
                    runner=MultiPtychography([_reconstruction(c, s) for c, s in parts]))
    return dict(kind="one", reconstruction=_reconstruction(case, seed), options=_options(case, seed),
                positions=case["solver"] == "positions")


def run(state):
    if state["kind"] == "loss":
        from py4dstem_amd.autograd import ptychographic_loss
        loss = ptychographic_loss(state["object"], state["probe"], state["positions"],
                                  state["amplitudes"])
        go, gp = torch.autograd.grad(loss, (state["object"], state["probe"]))
        # a sum of squared float32 residuals
        return {"loss": loss.detach().float(), "object": go, "probe": gp}
    if state["kind"] == "many":
        runner = state["runner"].reconstruct(state["iters"], state["options"])
        return [_results(p) for p in runner.items]
    p = state["reconstruction"].reconstruct(**state["options"])
    return _results(p, state["positions"])


def _results(p, positions=False):
    # the errors are sums of squared float32 residuals
    out = {"object": p.object, "probe": p.probe,
           "errors": np.asarray(p.error_iterations, dtype=np.float32)}
    if positions:
        out["positions"] = p.positions
    return out


def work(case):
    """Per iteration: the amplitudes of every position once, and object and
    probe read and written once per mini-batch; with projection sets the exit
    waves too.  Three 2-D transforms per position and mode (five with position
    correction), about ten operations per pixel for each of exit wave,
    projection and scatter."""
    total = {"bytes": 0.0, "flops": 0.0}
    for c, _ in _parts(case, 0):
        S, n = c["S"], c["nx"] * c["ny"]
        px, step = PIXEL[S], STEP[S]
        shape = ([c["object_px"]] * 2 if c["object_px"] else
                 [(m - 1) * step / px + S for m in (c["nx"], c["ny"])])
        opix = shape[0] * shape[1]
        batches = -(-n // c["batch"]) if c["batch"] else 1
        word = 4 if c["solver"] == "potential" else 8
        per = n * S * S * 4.0 + batches * (2 * word * opix + 16.0 * S * S * c["modes"])
        if c["solver"] == "projection":
            per += n * S * S * 16.0
        ffts = 5 if c["solver"] == "positions" else 3 * c["modes"]
        if c["solver"] == "loss":
            ffts = 4
        flops = n * S * S * (ffts * 10.0 * math.log2(S) + 30.0 * c["modes"])
        total["bytes"] += per * c["iters"]
        total["flops"] += flops * c["iters"]
    return total


# -- the same in 64 bits ---------------------------------------------------------

class _Exact:
    """One problem's reconstruction in complex128 on plain torch arrays."""

    def __init__(self, case, seed):
        w = _scene(case, seed)
        dev = w["counts"].device
        self.case, self.seed, self.S, self.shape = case, seed, case["S"], w["shape"]
        self.A = torch.sqrt(w["counts"].double())
        self.mean = w["counts"].double().sum((-2, -1)).mean()
        self.n = len(w["positions"])
        self.pos = torch.from_numpy(w["positions"]).to(dev).double()
        o = torch.from_numpy(w["object"]).to(dev)
        self.pot = case["solver"] == "potential"
        self.obj = o.double() if self.pot else o.to(torch.complex128)
        p = torch.from_numpy(w["probe"]).to(dev).to(torch.complex128)
        self.probe = p if p.dim() == 3 else p[None]
        self.outside = torch.from_numpy(~w["mask"]).to(dev)
        k = torch.from_numpy(_fidx(self.S)).to(dev).double()
        self.kx, self.ky = k[:, None], k[None, :]
        self.errors = []

    def patches(self, idx):
        flat = self.obj.reshape(-1)[idx]
        return torch.exp(1j * flat) if self.pot else flat

    def scatter(self, idx, values):
        out = torch.zeros(self.shape[0] * self.shape[1], dtype=torch.float64, device=idx.device)
        return out.index_add_(0, idx.reshape(-1), values.reshape(-1)).reshape(self.shape)

    def scatter_c(self, idx, values):
        return torch.complex(self.scatter(idx, values.real.contiguous()),
                             self.scatter(idx, values.imag.contiguous()))

    @staticmethod
    def norm(s):
        return 1.0 / torch.sqrt(1e-16 + s.max() ** 2)

    def batch(self, order):
        """One gradient-descent mini-batch; returns its summed squared error."""
        idx, frac = _windows(self.pos[order], self.S, self.shape)
        op = self.patches(idx)
        A = self.A[order]
        ps = [_shifted_probe(m[None], frac) for m in self.probe]
        far = [torch.fft.fft2(s * op) for s in ps]
        if len(far) == 1:
            mag = far[0].abs()
            unit = torch.where(mag == 0, torch.ones_like(far[0]), far[0] / mag)
            chi = [torch.fft.ifft2(A * unit - far[0])]
        else:
            mag = torch.sqrt(sum(f.abs() ** 2 for f in far))
            factor = torch.where(mag == 0, torch.zeros_like(mag), A / mag)
            chi = [torch.fft.ifft2(factor * f - f) for f in far]
        err = ((A - mag) ** 2).sum()
        step = 0.5
        s = sum(self.scatter(idx, p.abs() ** 2) for p in ps)
        terms = sum(p.conj() * x for p, x in zip(ps, chi))
        if self.pot:
            g = self.scatter(idx, (-1j * op.conj() * terms).real.contiguous())
        else:
            g = self.scatter_c(idx, terms)
        if not self.case["fix_probe"]:
            so = (op.abs() ** 2).sum(0)
            for m, x in enumerate(chi):
                self.probe[m] += step * (op.conj() * x).sum(0) * self.norm(so)
        self.obj = self.obj + step * g * self.norm(s)
        if self.case["solver"] == "positions":
            self.move(order, idx, ps[0], far[0], A)
        return err

    def move(self, order, idx, ps, far, A):
        flat = self.obj.reshape(-1)
        rows, cols = idx // self.shape[1], idx % self.shape[1]
        dx = ((rows + 1) % self.shape[0]) * self.shape[1] + cols
        dy = rows * self.shape[1] + (cols + 1) % self.shape[1]
        px = 2 * ((far - torch.fft.fft2(ps * flat[dx])) * far.conj()).real
        py = 2 * ((far - torch.fft.fft2(ps * flat[dy])) * far.conj()).real
        d = A ** 2 - far.abs() ** 2
        a, b, c = ((u * v).sum((-2, -1)) for u, v in ((px, px), (px, py), (py, py)))
        e, f = (px * d).sum((-2, -1)), (py * d).sum((-2, -1))
        det = a * c - b * b
        self.pos[order] -= 0.5 * torch.stack(((c * e - b * f) / det, (a * f - b * e) / det), -1)

    def difference_map(self, iteration):
        idx, frac = _windows(self.pos, self.S, self.shape)
        a, b, c = -0.5, 1.0, 1.5
        op = self.patches(idx)
        ps = _shifted_probe(self.probe[0][None], frac)
        psi = ps * op
        e = psi if iteration == 0 else self.exits
        far = torch.fft.fft2(c * psi + (1 - c) * e)
        mag = far.abs()
        unit = torch.where(mag == 0, torch.ones_like(far), far / mag)
        err = ((self.A - mag) ** 2).sum()
        self.exits = (1 - a - b) * e + a * psi + b * torch.fft.ifft2(self.A * unit)
        new = self.scatter_c(idx, ps.conj() * self.exits) * self.norm(
            self.scatter(idx, ps.abs() ** 2))
        if not self.case["fix_probe"]:
            self.probe[0] = ((op.conj() * self.exits).sum(0)
                             * self.norm((op.abs() ** 2).sum(0)))
        self.obj = new
        return err

    def smooth(self, x, sigma_px):
        r = int(4.0 * sigma_px + 0.5)
        t = torch.arange(-r, r + 1, device=x.device, dtype=torch.float64)
        w = torch.exp(-0.5 * t * t / sigma_px ** 2)
        w = w / w.sum()
        for axis in (0, 1):
            n = x.shape[axis]
            acc = torch.zeros_like(x)
            i = torch.arange(n, device=x.device)
            for j in range(-r, r + 1):
                m = (i + j) % (2 * n)
                m = torch.where(m < n, m, 2 * n - 1 - m)
                acc = acc + w[j + r] * x.index_select(axis, m)
            x = acc
        return x

    def constraints(self):
        c, px = self.case, PIXEL[self.S]
        if c["sigma"]:
            self.obj = self.smooth(self.obj, c["sigma"] / px)
        if c["q_lowpass"] or c["q_highpass"]:
            dev = self.obj.device
            qx = torch.fft.fftfreq(self.shape[0], px, dtype=torch.float64, device=dev)
            qy = torch.fft.fftfreq(self.shape[1], px, dtype=torch.float64, device=dev)
            q = torch.sqrt(qx[:, None] ** 2 + qy[None, :] ** 2)
            env = torch.ones_like(q)
            if c["q_highpass"]:
                env = env * (1 - 1 / (1 + (q / c["q_highpass"]) ** 4))
            if c["q_lowpass"]:
                env = env / (1 + (q / c["q_lowpass"]) ** 4)
            m = self.obj.mean()
            self.obj = torch.fft.ifft2(torch.fft.fft2(self.obj - m) * env) + m
        any_out = bool(self.outside.any())
        if self.pot:
            if any_out:
                self.obj = self.obj - self.obj[self.outside].mean()
            self.obj = self.obj.clamp_min(0.0)
        else:
            phase, amp = torch.angle(self.obj), self.obj.abs()
            if any_out:
                phase = phase - phase[self.outside].mean()
            self.obj = torch.polar(amp.clamp_max(1.0), phase)
        if not c["fix_probe"]:
            I = self.probe[0].abs() ** 2
            shift = torch.stack((-(self.kx * I).sum() / I.sum(), -(self.ky * I).sum() / I.sum()))
            self.probe = _shifted_probe(self.probe, shift[None])

    def reconstruct(self):
        c = self.case
        order = np.arange(self.n)
        b = c["batch"] or self.n
        if c["batch"]:
            np.random.seed(int(self.seed))
        count = -(-self.n // b)
        base, extra = divmod(self.n, count)
        sizes = [base + 1] * extra + [base] * (count - extra)
        for it in range(c["iters"]):
            if c["solver"] == "projection":
                err = self.difference_map(it)
            else:
                # a full batch in another order only moves its sums' rounding
                if c["batch"]:
                    np.random.shuffle(order)
                err, start = 0.0, 0
                for nb in sizes:
                    err = err + self.batch(torch.from_numpy(order[start:start + nb])
                                           .to(self.pos.device))
                    start += nb
            self.errors.append(float(err / (self.mean * self.n)))
            self.constraints()
        out = {"object": self.obj.cpu().numpy()}
        probe = np.fft.fftshift(self.probe.cpu().numpy(), axes=(-2, -1))
        out["probe"] = probe if c["solver"] == "mixed" else probe[0]
        out["errors"] = np.asarray(self.errors, dtype=np.float64)
        if c["solver"] == "positions":
            out["positions"] = self.pos.cpu().numpy() * PIXEL[self.S]
        return out


def _exact_loss(case, seed):
    w = _scene(case, seed)
    dev = w["counts"].device
    obj = torch.from_numpy(w["object"]).to(dev).to(torch.complex128)
    probe = torch.from_numpy(w["probe"]).to(dev).to(torch.complex128)
    go, gp, total = torch.zeros_like(obj), torch.zeros_like(probe), 0.0
    pos = torch.from_numpy(w["positions"]).to(dev).double()
    for s in range(0, len(pos), 256):
        o, p = obj.clone().requires_grad_(), probe.clone().requires_grad_()
        idx, frac = _windows(pos[s:s + 256], case["S"], w["shape"])
        far = torch.fft.fft2(_shifted_probe(p[None], frac) * o.reshape(-1)[idx])
        loss = ((far.abs() - torch.sqrt(w["counts"][s:s + 256].double())) ** 2).sum()
        a, b = torch.autograd.grad(loss, (o, p))
        go, gp, total = go + a, gp + b, total + loss.detach()
    return {"loss": total, "object": go, "probe": gp}


def exact(case, seed):
    if case["solver"] == "loss":
        return _exact_loss(case, seed)
    out = [_Exact(c, s).reconstruct() for c, s in _parts(case, seed)]
    return out if case["solver"] == "many" else out[0]
