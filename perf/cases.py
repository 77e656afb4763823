"""Workloads of the NUFFT operator that are timed, with their exact values.

A case is a dict of plain values; ``kind`` names the call and the sizes say
how large it is:

* ``pair``    ``op`` of an image and ``adj_op`` of measured k-space
* ``op``, ``adj``   one of the two alone (the large 3D problems)
* ``dc``      ``data_consistency``: the gradient of an iterative reconstruction
* ``grad``    ``op`` with autograd: gradients of an L2 loss for the image and
  the trajectory (one step of learning a trajectory)
* ``lsqr``    ``pinv_solver(optim="lsqr")``: a whole reconstruction
* ``gram``    ``gram_op``: the Toeplitz form of ``A^H D A``
* ``stack``   the stacked 2.5D operator, ``op`` and ``adj_op``
* ``update``  ``update_samples`` to a new trajectory, then ``op`` (motion
  correction, trajectory learning: every step pays for the new samples)
* ``frames``  ``MultiTrajectoryOperator``: frames of uneven length in one plan,
  ``op`` and ``adj_op``

``n0 n1 n2`` is the image (``n2 = 0``: 2D), ``shots x ns`` the samples
(``frames``: between half and all of ``shots`` for each frame), ``coils``
the coils, ``sense`` whether they carry sensitivity maps, ``density`` whether
k-space is density compensated, ``eps`` the requested accuracy.  Trajectories
are given in radians, so the operator takes them as they are.
"""

import math
import os
import random
import sys

import torch

_PKG = os.path.join(os.getcwd(), "mri-nufft_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

_GOLDEN = math.pi * (3.0 - math.sqrt(5.0))
# exact() is given up above this many operations of the explicit sums (64 bits)
_EXACT_FLOPS = 1.2e14


def _case(name, kind, n0, n1, n2, traj, shots, ns, coils, sense, density, eps=1e-6, **more):
    return dict(name=name, kind=kind, n0=n0, n1=n1, n2=n2, traj=traj, shots=shots, ns=ns,
                coils=coils, sense=sense, density=density, eps=eps, **more)


def listed():
    return [
        # a single-coil 2D radial slice: the smallest call, one image at a time
        _case("radial2d_256_c1", "pair", 256, 256, 0, "radial", 100, 500, 1, False, False),
        # multi-coil 2D spiral with maps and density: an ordinary 2D acquisition
        _case("spiral2d_320_c32", "pair", 320, 320, 0, "spiral", 64, 2048, 32, True, True),
        # the gradient of an unrolled or proximal 2D reconstruction
        _case("dc2d_256_c8", "dc", 256, 256, 0, "radial", 128, 512, 8, True, True),
        # one step of learning a 2D trajectory (image and trajectory gradients)
        _case("grad2d_256_c8", "grad", 256, 256, 0, "radial", 128, 1024, 8, True, False),
        # a whole 2D reconstruction with the default solver, stopped early as
        # regularisation (further on, float32 LSQR loses its orthogonality on
        # centre-out samples and its iterates say nothing about the operator)
        _case("lsqr2d_256_c16", "lsqr", 256, 256, 0, "radial", 256, 512, 16, True, False,
              iters=4),
        # dynamic imaging: frames of uneven length in one plan
        _case("frames2d_192_c8", "frames", 192, 192, 0, "radial", 55, 400, 8, True, True,
              frames=12),
        # ragged 3D: odd axes, random samples, no maps, a looser accuracy
        _case("random3d_odd_c3", "pair", 75, 90, 61, "random", 100, 1003, 3, False, False,
              eps=1e-4),
        # the 3D radial acquisition, forward and adjoint: the largest calls
        _case("radial3d_192_c16_op", "op", 192, 192, 192, "radial", 4096, 512, 16, True, False),
        _case("radial3d_192_c16_adj", "adj", 192, 192, 192, "radial", 4096, 512, 16, True, True),
        # the Toeplitz gradient of a 3D reconstruction
        _case("gram3d_128_c8", "gram", 128, 128, 128, "radial", 256, 512, 8, True, True),
        # stack of stars through the stacked operator
        _case("stack_128_c8", "stack", 128, 128, 128, "radial", 256, 256, 8, True, False),
        # a new 3D trajectory before each forward: sorting is part of the work
        _case("update3d_128_c4", "update", 128, 128, 128, "radial", 1024, 400, 4, True, False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pair", "pair", "op", "adj", "dc", "grad", "lsqr", "frames", "gram",
                       "stack", "update"])
    three = kind == "stack" or (kind not in ("grad", "lsqr", "frames") and rng.random() < 0.45)
    if kind == "gram":  # the Toeplitz form needs axes whose doubles are 2,3,5-smooth
        pick = [24, 30, 32, 36, 40, 45, 48, 50, 54, 60, 64, 72, 75, 80, 81, 90, 96, 100, 108, 120,
                125, 128] + ([] if three else [135, 144, 160, 180, 192, 200, 240, 250, 256, 320])
        n = [rng.choice(pick) for _ in range(3 if three else 2)]
    elif three:
        # odd and even axes, near-cubic
        side = _log_int(rng, 24, 144)
        n = [max(16, int(side * rng.uniform(0.7, 1.15))) for _ in range(3)]
    else:
        side = _log_int(rng, 48, 448)
        n = [max(32, int(side * rng.uniform(0.75, 1.1))) for _ in range(2)]
    ns = rng.randint(max(n), 2 * max(n) + 200)
    shots = _log_int(rng, 16, 1500) if three and kind != "stack" else _log_int(rng, 16, 320)
    coils = _log_int(rng, 1, 24 if three else 32)
    while coils > 1 and coils * math.prod(n) > 20e6:
        coils //= 2
    case = dict(kind=kind, n0=n[0], n1=n[1], n2=n[2] if three else 0,
                traj=rng.choice(["radial", "radial", "spiral", "random"]), shots=shots, ns=ns,
                coils=coils, sense=coils > 1 and rng.random() < 0.75,
                density=kind != "lsqr" and rng.random() < 0.5,
                eps=rng.choice([1e-6, 1e-6, 1e-6, 1e-5, 1e-4, 1e-3]))
    if three and case["traj"] == "spiral":
        case["traj"] = "radial"
    if kind == "lsqr":
        case["iters"] = rng.randint(3, 8) if case["traj"] == "random" else rng.randint(2, 4)
    if kind == "frames":
        case["frames"] = rng.randint(2, 12)
    return case


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _shape(case):
    return tuple(case[k] for k in ("n0", "n1", "n2") if case[k])


def _gen(seed, device):
    g = torch.Generator(device=device)
    g.manual_seed(int(seed))
    return g


def _cplx(shape, g):
    d = g.device
    return torch.complex(torch.randn(shape, generator=g, device=d),
                         torch.randn(shape, generator=g, device=d))


def _trajectory(traj, ndim, shots, ns, g):
    """(shots * ns, ndim) float32 radians, every seed another orientation."""
    d = g.device
    u = torch.rand(4, generator=g, device=d, dtype=torch.float64)
    if traj == "random":
        x = torch.rand((shots * ns, ndim), generator=g, device=d, dtype=torch.float64) - 0.5
        return (2 * math.pi * x).to(torch.float32)
    r = math.pi * torch.arange(ns, device=d, dtype=torch.float64) / max(ns - 1, 1)
    k = torch.arange(shots, device=d, dtype=torch.float64)
    if ndim == 2:
        # centre-out spokes, or interleaves of one turn, evenly rotated
        turn = 2 * math.pi * r / math.pi if traj == "spiral" else torch.zeros_like(r)
        a = (2 * math.pi * (k / shots + u[0]))[:, None] + turn[None, :]
        x = torch.stack([r * torch.cos(a), r * torch.sin(a)], -1)
    else:
        # centre-out spokes on a golden-angle spiral over the sphere, rotated
        z = (2 * k + 1) / shots - 1
        rho = torch.sqrt(torch.clamp(1 - z * z, min=0.0))
        v = torch.stack([rho * torch.cos(_GOLDEN * k), rho * torch.sin(_GOLDEN * k), z], -1)
        q = u / u.norm()
        w, i, j, l = q[0], q[1], q[2], q[3]
        rot = torch.stack([
            torch.stack([1 - 2 * (j * j + l * l), 2 * (i * j - l * w), 2 * (i * l + j * w)]),
            torch.stack([2 * (i * j + l * w), 1 - 2 * (i * i + l * l), 2 * (j * l - i * w)]),
            torch.stack([2 * (i * l - j * w), 2 * (j * l + i * w), 1 - 2 * (i * i + j * j)])])
        x = r[None, :, None] * (v @ rot.T)[:, None, :]
    return x.reshape(-1, ndim).to(torch.float32)


def _density_of(traj, ndim):
    """|k|^(d-1) compensation, the analytic weight of centre-out sampling."""
    return (0.01 + traj.norm(dim=1) / math.pi) ** (ndim - 1)


def _maps(coils, shape, g):
    """Smooth complex coil maps (Gaussian bumps) with unit root sum of squares."""
    d = g.device
    bumps = 4
    ctr = torch.rand((coils, bumps, len(shape)), generator=g, device=d) - 0.5
    amp = _cplx((coils, bumps), g)
    fac = []
    for ax, n in enumerate(shape):
        t = torch.arange(n, device=d) / n - 0.5
        fac.append(torch.exp(-((t - ctr[..., ax, None]) ** 2) / (2 * 0.3 ** 2)))
    out = torch.empty((coils, *shape), dtype=torch.complex64, device=d)
    for c in range(coils):
        a = amp[c][:, None] * fac[0][c]
        left = a if len(shape) == 2 else (a[:, :, None] * fac[1][c][:, None, :]).flatten(1)
        out[c] = (left.T @ fac[-1][c].to(torch.complex64)).reshape(shape)
    rss = sum(m.abs() ** 2 for m in out).sqrt()
    return out.div_(rss)


def _phantom(shape, g):
    """Nested and scattered ellipsoids with a little complex noise."""
    d = g.device
    grids = torch.meshgrid(*[torch.arange(n, device=d) / n - 0.5 for n in shape], indexing="ij")
    u = torch.rand((8, 2 * len(shape) + 1), generator=g, device=d)
    img = torch.zeros(shape, device=d)
    for q in range(8):
        ctr = (u[q, :len(shape)] - 0.5) * (0.1 if q == 0 else 0.5)
        ax = 0.4 if q == 0 else 0.05 + 0.15 * u[q, len(shape):2 * len(shape)]
        amp = 1.0 if q == 0 else u[q, -1] - 0.4
        ax = torch.as_tensor(ax, device=d).expand(len(shape))
        img += amp * (sum(((x - ctr[k]) / ax[k]) ** 2 for k, x in enumerate(grids)) <= 1)
    return img + 0.01 * _cplx(shape, g)


def _frame_shots(case):
    rng = random.Random(case["shots"] + 1000 * case["frames"])
    return [rng.randint(max(1, case["shots"] // 2), case["shots"]) for _ in range(case["frames"])]


def _inputs(case, seed):
    g = _gen(seed, "cuda")
    kind, shape, C = case["kind"], _shape(case), case["coils"]
    plane = shape[:2] if kind == "stack" else shape
    out = {}
    if kind == "frames":
        out["traj"] = [_trajectory(case["traj"], 2, s, case["ns"], g) for s in _frame_shots(case)]
        out["density"] = [_density_of(t, 2) for t in out["traj"]] if case["density"] else None
        M = [t.shape[0] for t in out["traj"]]
        out["maps"] = _maps(C, shape, g) if case["sense"] else None
        out["image"] = _cplx((case["frames"], *(() if case["sense"] else (C,)), *shape), g)
        out["ksp"] = [_cplx((C, m), g) for m in M]
        return out
    t = _trajectory(case["traj"], len(plane), case["shots"], case["ns"], g)
    M = t.shape[0] * (shape[2] if kind == "stack" else 1)
    out["traj"] = t
    out["density"] = _density_of(t, len(plane)) if case["density"] else None
    out["maps"] = _maps(C, shape, g) if case["sense"] else None
    if kind not in ("adj", "lsqr"):
        out["image"] = _cplx((1, 1 if case["sense"] else C, *shape), g)
    if kind == "lsqr":  # k-space measured of an object, with noise
        x = _phantom(shape, g)[None]
        x = x * out["maps"] if case["sense"] else x * _maps(C, shape, g)
        y = _Exact(t, shape).forward(x)
        noise = 0.01 * y.abs().square().mean().sqrt()
        out["ksp"] = (y + noise * _cplx((C, M), g)).to(torch.complex64)[None]
    elif kind not in ("op", "gram", "update"):
        out["ksp"] = _cplx((1, C, M), g)
    if kind == "update":  # the trajectory that the plan holds before the update
        out["old"] = _trajectory(case["traj"], len(shape), case["shots"], case["ns"], g)
    return out


def prepare(case, seed):
    import hipnufft

    st = _inputs(case, seed)
    kind, shape, C = case["kind"], _shape(case), case["coils"]
    st["kind"] = kind
    more = {} if st["density"] is None else {"density": st["density"]}
    if kind == "frames":
        from hipnufft.batched import MultiTrajectoryOperator

        st["op"] = MultiTrajectoryOperator(st["traj"], shape, n_coils=C, smaps=st["maps"],
                                           eps=case["eps"], **more)
        st["ksp"] = torch.cat([k.reshape(-1) for k in st["ksp"]])
        return st
    if kind == "stack":
        st["op"] = hipnufft.MRIStackedHipNUFFT(st["traj"].cpu().numpy(), shape, n_coils=C,
                                               smaps=st["maps"], z_index=None, eps=case["eps"],
                                               **more)
        return st
    first = st["old"] if kind == "update" else st["traj"]
    st["op"] = hipnufft.get_operator("hipnufft")(first, shape, n_coils=C, smaps=st["maps"],
                                                 eps=case["eps"], **more)
    if kind == "grad":
        st["auto"] = st["op"].make_autograd(wrt_data=True, wrt_traj=True)
    if kind == "gram":
        st["op"].compute_toeplitz_kernel()
    st["iters"] = case.get("iters", 0)
    return st


def run(state):
    kind, op = state["kind"], state["op"]
    if kind in ("pair", "stack", "frames"):
        return op.op(state["image"]), op.adj_op(state["ksp"])
    if kind == "op":
        return op.op(state["image"])
    if kind == "adj":
        return op.adj_op(state["ksp"])
    if kind == "dc":
        return op.data_consistency(state["image"], state["ksp"])
    if kind == "gram":
        return op.gram_op(state["image"])
    if kind == "update":
        op.update_samples(state["traj"])
        return op.op(state["image"])
    if kind == "lsqr":
        return op.pinv_solver(state["ksp"], optim="lsqr", max_iter=state["iters"])
    # grad: the L2 loss of the k-space, its gradients for image and trajectory
    auto = state["auto"]
    x = state["image"].detach().requires_grad_(True)
    y = auto.op(x)
    loss = 0.5 * (y - state["ksp"]).abs().square().sum()
    gx, gt = torch.autograd.grad(loss, (x, auto.samples))
    return y, gx, gt


# ---------------------------------------------------------------------------
# the work a pass cannot do without
# ---------------------------------------------------------------------------
def _samples_of(case):
    per = case["shots"] * case["ns"]
    return sum(_frame_shots(case)) * case["ns"] if case["kind"] == "frames" else per


def work(case):
    """Inputs and outputs once; fine-grid FFTs (sigma 2) and kernel footprints."""
    kind, shape, C = case["kind"], _shape(case), case["coils"]
    N, M, D = math.prod(shape), _samples_of(case), len(shape)
    w = min(max(math.ceil(-math.log10(case["eps"] / 10)), 2), 16)
    ic = 1 if case["sense"] else C
    B = case.get("frames", 1)
    fft2 = lambda n: 5.0 * 2 ** len(n) * math.prod(n) * math.log2(2 ** len(n) * math.prod(n))
    if kind == "stack":
        Z = shape[2]
        planes = Z * (fft2(shape[:2]) + 4.0 * M * w ** 2)
        one = C * (planes + 5.0 * N * math.log2(Z))
        ksp = 8.0 * C * M * Z
        pts = 8.0 * M
    else:
        one = C * (B * fft2(shape) + 4.0 * M * w ** D)
        ksp = 8.0 * C * M
        pts = 4.0 * D * M
    img = 8.0 * ic * N * B
    const = pts + (8.0 * C * N if case["sense"] else 0.0)
    dens = 4.0 * M if case["density"] else 0.0
    if kind in ("op", "update"):
        return {"bytes": const + img + ksp, "flops": one}
    if kind == "adj":
        return {"bytes": const + dens + img + ksp, "flops": one}
    if kind == "dc":
        return {"bytes": const + dens + 2 * img + ksp, "flops": 2 * one}
    if kind == "gram":
        return {"bytes": 8.0 * C * N * bool(case["sense"]) + 2 * img + 8.0 * 2 ** D * N,
                "flops": 2 * C * fft2(shape)}
    if kind == "lsqr":
        return {"bytes": const + img + ksp, "flops": 2.0 * (case["iters"] + 0.5) * one}
    if kind == "grad":  # forward, adjoint, and the derivative footprints of the forward grid
        return {"bytes": const + 2 * img + 2 * ksp + pts,
                "flops": 2 * one + 4.0 * (D + 1) * C * M * w ** D}
    return {"bytes": const + dens + 2 * img + 2 * ksp, "flops": 2 * one}


# ---------------------------------------------------------------------------
# the same in 64 bits by explicit sums
# ---------------------------------------------------------------------------
class _Exact:
    """The explicit sums of one trajectory: forward and adjoint of any batch."""

    def __init__(self, traj, shape):
        self.w = traj.to(torch.float64)
        self.shape = tuple(shape)
        self.rows = math.prod(self.shape[:-1])

    def _phase(self, d, lo, hi):
        n = torch.arange(self.shape[d], device=self.w.device, dtype=torch.float64)
        a = self.w[lo:hi, d, None] * (n - self.shape[d] // 2)
        return torch.complex(torch.cos(a), -torch.sin(a))  # (m, n)

    def _lead(self, lo, hi):
        """(rows, m): the phases of all axes but the last."""
        e = self._phase(0, lo, hi).T
        if len(self.shape) == 3:
            e = (e[:, None, :] * self._phase(1, lo, hi).T[None]).reshape(self.rows, -1)
        return e

    def _chunks(self):
        step = max(64, (1 << 25) // self.rows)
        for lo in range(0, self.w.shape[0], step):
            yield lo, min(lo + step, self.w.shape[0])

    def forward(self, x):
        """x (b, *shape) -> (b, M)"""
        x = x.to(torch.complex128).reshape(-1, self.rows, self.shape[-1])
        out = torch.empty((x.shape[0], self.w.shape[0]), dtype=torch.complex128, device=x.device)
        for lo, hi in self._chunks():
            lead, last = self._lead(lo, hi), self._phase(len(self.shape) - 1, lo, hi).T.contiguous()
            for b in range(x.shape[0]):
                out[b, lo:hi] = ((x[b] @ last) * lead).sum(0)
        return out

    def adjoint(self, y):
        """y (b, M) -> (b, *shape)"""
        y = y.to(torch.complex128)
        out = torch.zeros((y.shape[0], self.rows, self.shape[-1]), dtype=torch.complex128,
                          device=y.device)
        for lo, hi in self._chunks():
            lead = self._lead(lo, hi).conj().resolve_conj()
            last = self._phase(len(self.shape) - 1, lo, hi).conj().resolve_conj()
            for b in range(y.shape[0]):
                out[b] += (lead * y[b, lo:hi]) @ last
        return out.reshape(-1, *self.shape)


def _sense_op(e, x, maps, inv):
    return inv * e.forward(x if maps is None else x[:1] * maps)


def _sense_adj(e, y, maps, dens, inv):
    z = inv * e.adjoint(y if dens is None else y * dens)
    return z if maps is None else (z * maps.conj()).sum(0, keepdim=True)


def _lsqr(op, adj, b, iters):
    """Paige and Saunders' LSQR; None when one of its usual tests (1e-6) could stop it early."""
    norm = torch.linalg.vector_norm
    beta = norm(b)
    bnorm = float(beta)
    u = b / beta
    v = adj(u)
    alpha = norm(v)
    v = v / alpha
    w, x = v, torch.zeros_like(v)
    phibar, rhobar, anorm2 = beta, alpha, 0.0
    for _ in range(iters):
        u = op(v) - alpha * u
        beta = norm(u)
        u = u / beta
        anorm2 += float(alpha) ** 2 + float(beta) ** 2
        v = adj(u) - beta * v
        alpha = norm(v)
        v = v / alpha
        rho = torch.sqrt(rhobar ** 2 + beta ** 2)
        c, s = rhobar / rho, beta / rho
        theta, rhobar = s * alpha, -c * alpha
        phi, phibar = c * phibar, s * phibar
        x = x + (phi / rho) * w
        w = v - (theta / rho) * w
        arnorm = float(alpha) * abs(float(s * phi))
        anorm = math.sqrt(anorm2)
        if (arnorm <= 1e-4 * anorm * float(phibar.abs())
                or float(phibar.abs()) <= 1e-4 * (bnorm + anorm * float(norm(x)))):
            return None
    return x


def exact(case, seed):
    kind, shape, C = case["kind"], _shape(case), case["coils"]
    N, M = math.prod(shape), _samples_of(case)
    B = case.get("frames", 1)
    calls = {"pair": 2, "dc": 2, "gram": 2, "grad": 4, "stack": 2, "frames": 2,
             "lsqr": 2 * case.get("iters", 0) + 1}.get(kind, 1)
    if 8.0 * C * N * M * calls > _EXACT_FLOPS:
        return None
    i = _inputs(case, seed)
    maps = None if i["maps"] is None else i["maps"].to(torch.complex128)
    inv = 1.0 / math.sqrt(N * 2.0 ** len(shape))
    ic = 1 if case["sense"] else C
    if kind == "frames":
        ys, xs = [], []
        for k in range(B):
            e = _Exact(i["traj"][k], shape)
            d = None if i["density"] is None else i["density"][k].to(torch.float64)
            ys.append(_sense_op(e, i["image"][k].reshape(ic, *shape), maps, inv).reshape(-1))
            xs.append(_sense_adj(e, i["ksp"][k], maps, d, inv))
        x = torch.stack(xs)
        return torch.cat(ys), x.reshape(B, *(() if case["sense"] else (C,)), *shape)
    d = None if i["density"] is None else i["density"].to(torch.float64)
    if kind == "stack":
        X, Y, Z = shape
        e = _Exact(i["traj"], (X, Y))
        inv = 1.0 / math.sqrt(X * Y * 4.0 * 2.0 * Z)
        z = torch.arange(Z, device="cuda", dtype=torch.float64) - Z // 2
        a = 2 * math.pi / Z * (z[:, None] * z[None, :])
        f = torch.complex(torch.cos(a), -torch.sin(a))
        img = i["image"][0].to(torch.complex128)
        img = img if maps is None else img * maps
        y = torch.stack([e.forward((img[c] @ f).permute(2, 0, 1)) for c in range(C)]) * inv
        k = i["ksp"].reshape(C, Z, -1)
        out = []
        for c in range(C):
            p = e.adjoint(k[c] if d is None else k[c] * d).permute(1, 2, 0)
            out.append(p @ f.conj().resolve_conj())
        x = torch.stack(out) * inv
        x = x if maps is None else (x * maps.conj()).sum(0, keepdim=True)
        return y.reshape(1, C, -1), x.reshape(1, ic, *shape)
    e = _Exact(i["traj"], shape)
    x = None if "image" not in i else i["image"][0].to(torch.complex128)
    k = None if "ksp" not in i else i["ksp"][0].to(torch.complex128)
    op = lambda v: _sense_op(e, v, maps, inv)
    adj = lambda v, w=None: _sense_adj(e, v, maps, w, inv)
    if kind in ("op", "update"):
        return op(x)[None]
    if kind == "adj":
        return adj(k, d)[None]
    if kind == "pair":
        return op(x)[None], adj(k, d)[None]
    if kind == "dc":
        return adj(op(x) - k, d)[None]
    if kind == "gram":
        return adj(op(x), d)[None]
    if kind == "lsqr":
        v = _lsqr(op, adj, k, case["iters"])
        return None if v is None else v[None]
    y = op(x)
    r = y - k
    gt = []
    for ax, n in enumerate(shape):
        pos = torch.arange(n, device="cuda", dtype=torch.float64) - n // 2
        pos = pos.reshape([-1 if q == ax else 1 for q in range(len(shape))])
        gt.append((r.conj() * (-1j) * op(x * pos)).real.sum(0))
    w = adj(r, d)
    return y[None], w[None], torch.stack(gt, -1)
