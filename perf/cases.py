"""Timing cases: calls of the public API over the sizes, options and directions it is used with.

A case is a dict:
  kind     "project"           project_2d_forw / project_3d_to_2d_forw
           "project_step"      the same, then the gradients of the reconstruction, rotations and shifts
           "backproject"       backproject_2d_forw / backproject_2d_to_3d_forw
           "backproject_step"  the same, then the gradients of every input
           "prepare"           to_fourier of a volume, and reconstruct of a (data, weight) pair
  dim      2 or 3 (of the reconstruction)
  n        projection box ("prepare": the real-space box)
  os       oversampling; the reconstruction's box is ceil(n * os), made even
  B, P     batch items, poses of each
  cubic    cubic (True) or linear interpolation
  weights  backprojections: accumulate weights too
  cutoff   radius cutoff in Fourier pixels, 0 for none
  half     the reconstruction is stored as complex32 (forward projections)
  scale    factor on every pose matrix (1.0: rotations; else a magnification correction)
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "torch-projectors_amd"))
import torch_projectors as tp  # noqa: E402
from torch_projectors import fourier  # noqa: E402

KINDS = ("project", "project_step", "backproject", "backproject_step", "prepare")
REG = 0.1  # Wiener constant of the "prepare" cases


def _case(kind, dim, n, os_, B, P, cubic=False, weights=False, cutoff=0.0, half=False, scale=1.0, **name):
    return dict(kind=kind, dim=dim, n=n, os=os_, B=B, P=P, cubic=cubic, weights=weights, cutoff=cutoff, half=half,
                scale=scale, **name)


def listed():
    return [
        # one image scored against every in-plane angle (bench.py's c1): a call of microseconds
        _case("project", 2, 64, 2.0, 1, 256, name="p2d_64"),
        # re-projection of one reference along a tilt series: few poses, an ordinary box
        _case("project", 3, 96, 2.0, 1, 41, name="p3d_tilts_96"),
        # one minibatch of an ab-initio refinement at low resolution: forward and every gradient
        _case("project_step", 3, 64, 2.0, 1, 128, name="p3d_step_64"),
        # projection matching against one reference (c2)
        _case("project", 3, 128, 2.0, 1, 4096, name="p3d_128"),
        # the headline forward from a volume stored as complex32
        _case("project", 3, 256, 2.0, 1, 2048, half=True, name="p3d_half_256"),
        # pose and volume refinement at full resolution, cubic (c4): forward and every gradient
        _case("project_step", 3, 256, 2.0, 1, 2048, cubic=True, name="p3d_step_cubic_256"),
        # reconstruction of a particle set (c3)
        _case("backproject", 3, 128, 2.0, 1, 8192, weights=True, name="bp3d_128"),
        # the headline backprojection
        _case("backproject", 3, 256, 2.0, 1, 2048, weights=True, name="bp3d_256"),
        # a differentiable reconstruction of two half sets: ragged box, pose count and oversampling
        _case("backproject_step", 3, 90, 1.5, 2, 333, cubic=True, weights=True, cutoff=40.0, name="bp3d_step_90"),
        # alignment of several 2D classes at once with a resolution limit (c5's shape, fewer poses)
        _case("project_step", 2, 256, 2.0, 16, 512, cubic=True, cutoff=64.0, name="p2d_step_256"),
        # 2D class averages at the API's default oversampling of 1
        _case("backproject", 2, 100, 1.0, 8, 500, weights=True, name="bp2d_100"),
        # the steps around a refinement iteration: a map to Fourier space, and a reconstruction back
        _case("prepare", 3, 256, 2.0, 1, 0, name="prepare_256"),
    ]


def _box(c):
    raw = int(math.ceil(c["n"] * c["os"]))
    return raw + raw % 2


def _active(c):
    """Pixels of one projection within the cutoff."""
    n, rad = c["n"], c["cutoff"] or c["n"] / 2
    cut2, total = rad * rad, 0
    for i in range(n):
        r = i if i <= n // 2 else i - n
        if r * r <= cut2:
            total += min(n // 2, int(math.floor(math.sqrt(cut2 - r * r)))) + 1
    return total


def _vol(c):
    N = _box(c)
    return c["B"] * N ** (c["dim"] - 1) * (N // 2 + 1)


def work(c):
    if c["kind"] == "prepare":
        n, N = c["n"], _box(c)
        V, m = _vol(c), c["B"] * n ** c["dim"]
        # the map in, its spectrum out; (data, weight) in, the cropped map out; 2.5 N log2 N per real transform
        return {"bytes": 4 * m + 8 * V + 12 * V + 4 * m,
                "flops": 2 * 2.5 * c["B"] * N ** c["dim"] * c["dim"] * math.log2(N)}
    S, A, V = c["B"] * c["P"] * c["n"] * (c["n"] // 2 + 1), c["B"] * c["P"] * _active(c), _vol(c)
    K = 4 if c["cubic"] else 2
    poses = c["B"] * c["P"] * (c["dim"] ** 2 + 2) * 4
    # a tensor-product stencil reduced axis by axis (K^dim + ... + K complex multiply-adds); its transpose is
    # K^dim real scalings and additions per accumulated value; about 40 for the position and the phase
    stencil = 4 * sum(K ** k for k in range(1, c["dim"] + 1))
    rec = (4 if c["half"] else 8) * V
    taps = K ** c["dim"]
    if c["kind"] == "project":
        return {"bytes": rec + 8 * S + poses, "flops": A * (stencil + 40)}
    if c["kind"] == "project_step":
        # forward; then the upstream gradient and the volume in, the volume's and the poses' gradients out
        return {"bytes": 2 * rec + rec + 8 * S + 8 * A + 3 * poses,
                "flops": A * (stencil + 40 + 4 * taps + (1 + c["dim"]) * stencil + 60)}
    w = 1 if c["weights"] else 0
    fwd = {"bytes": (8 + 4 * w) * (A + V) + poses, "flops": A * (40 + taps * (4 + 2 * w))}
    if c["kind"] == "backproject":
        return fwd
    # backward: both upstream volumes and the projections in, gradients of projections, weights and poses out
    return {"bytes": fwd["bytes"] + (8 + 4 * w) * V + 8 * A + (8 + 4 * w) * S + 2 * poses,
            "flops": fwd["flops"] + A * ((1 + c["dim"]) * stencil + 60 + w * 2 * sum(2 ** k for k in range(1, c["dim"] + 1)))}


def tolerance(c):
    # measured against exact(): 2e-7 for the transforms; up to 1e-5 elsewhere, since fp32 sample positions of up
    # to N/2 round to about 1e-5 of a voxel (two runs, whose sums are in another order, differ by 4e-7)
    return {"rel": 1e-6 if c["kind"] == "prepare" else 4e-5}


def _cost(c):
    """Rough time, to keep drawn cases below the largest listed one."""
    if c["kind"] == "prepare":
        return 3.0 * _vol(c)
    per = (4.0 if c["dim"] == 2 else 8.0) * ((4.0 if c["dim"] == 2 else 8.0) if c["cubic"] else 1.0)
    steps = {"project": 1.0, "project_step": 5.0, "backproject": 3.0, "backproject_step": 5.0}[c["kind"]]
    return _vol(c) * 2.0 + c["B"] * c["P"] * c["n"] ** 2 / 2 * (steps * per + 4.0)


def draw(rng):
    most = 0.8 * max(_cost(c) for c in listed())

    def logint(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    while True:
        kind = rng.choice(KINDS[:4] * 3 + KINDS[4:])
        dim = 3 if kind == "prepare" else rng.choice((2, 3, 3))
        n = 2 * logint(16, 128)
        if kind == "prepare":
            c = _case(kind, dim, n, rng.choice((1.0, 1.5, 2.0)), rng.choice((1, 1, 2)), 0)
        else:
            c = _case(kind, dim, n, rng.choice((1.0, 1.5, 2.0, 2.0, 3.0)),
                      logint(1, 16) if dim == 2 else rng.choice((1, 1, 1, 2, 4)), logint(1, 4096),
                      cubic=rng.random() < 0.4, weights=kind.startswith("back") and rng.random() < 0.7,
                      cutoff=round(rng.uniform(0.25, 0.5) * n, 1) if rng.random() < 0.3 else 0.0,
                      half=kind == "project" and rng.random() < 0.15,
                      scale=1.02 if rng.random() < 0.15 else 1.0)
        if _box(c) <= 512 and _cost(c) <= most:
            return c


# ----------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _maps(c, g):
    """Real maps: noise within a soft sphere or disc, as an unfiltered reconstruction has it."""
    n, dim = c["n"], c["dim"]
    x = torch.randn(c["B"], *[n] * dim, generator=g, device="cuda")
    ax = (torch.arange(n, device="cuda", dtype=torch.float32) - n // 2) / (0.35 * n)
    rad2 = sum((ax.reshape([-1 if k == a else 1 for k in range(dim)])) ** 2 for a in range(dim))
    return x * torch.exp(-rad2 ** 4)


def _spectra(c, g):
    """The maps padded to the reconstruction's box, shifted and rfft'd with norm="forward"."""
    N, n, dim = _box(c), c["n"], c["dim"]
    lo = (N - n) // 2
    x = torch.nn.functional.pad(_maps(c, g), (lo, N - n - lo) * dim)
    axes = tuple(range(-dim, 0))
    return torch.fft.rfftn(torch.fft.fftshift(x, dim=axes), dim=axes, norm="forward").contiguous()


def _poses(c, g):
    """Uniform random orientations (in-plane angles in 2D) and shifts of a few pixels."""
    B, P = c["B"], c["P"]
    if c["dim"] == 2:
        a = torch.rand(B, P, generator=g, device="cuda", dtype=torch.float64) * 2 * math.pi
        R = torch.stack([a.cos(), -a.sin(), a.sin(), a.cos()], -1).reshape(B, P, 2, 2)
    else:
        q = torch.randn(B, P, 4, generator=g, device="cuda", dtype=torch.float64)
        w, x, y, z = (q / q.norm(dim=-1, keepdim=True)).unbind(-1)
        R = torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w),
                         2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w),
                         2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)], -1).reshape(B, P, 3, 3)
    shifts = 3 * torch.randn(B, P, 2, generator=g, device="cuda")
    return (R * c["scale"]).float().contiguous(), shifts


def _ctf2(c, g):
    """sin^2(k rho^2) weights, rho in cycles per pixel, k of each projection its own."""
    n = c["n"]
    i = torch.arange(n, device="cuda", dtype=torch.float32)
    r = torch.where(i <= n // 2, i, i - n)
    q = torch.arange(n // 2 + 1, device="cuda", dtype=torch.float32)
    rho2 = (r[:, None] ** 2 + q[None, :] ** 2) / float(n * n)
    k = 50 + 150 * torch.rand(c["B"], c["P"], 1, 1, generator=g, device="cuda")
    return torch.sin(k * rho2).square_()


def _noise(shape, g, complex_=True):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.complex64 if complex_ else torch.float32)


def prepare(c, seed):
    g, N, n = _gen(seed), _box(c), c["n"]
    rec_shape = (c["B"], *[N] * (c["dim"] - 1), N // 2 + 1)
    s = {"case": c, "cutoff": c["cutoff"] or None, "interp": "cubic" if c["cubic"] else "linear"}
    if c["kind"] == "prepare":
        s["map"] = _maps(c, g)
        s["data"] = _spectra(c, g)
        s["weight"] = torch.rand(*rec_shape, generator=g, device="cuda") * 4
        return s
    grads = c["kind"].endswith("_step")
    s["rot"], s["shift"] = (t.requires_grad_(grads) for t in _poses(c, g))
    shape = (c["B"], c["P"], n, n // 2 + 1)
    if c["kind"].startswith("project"):
        s["rec"] = _spectra(c, g)
        if c["half"]:  # the largest value at 1: within binary16's normal range
            s["rec"] = (s["rec"] / s["rec"].abs().max()).to(torch.complex32)
        s["rec"].requires_grad_(grads)
        if grads:
            s["up"] = _noise(shape, g)
    else:
        s["proj"] = _noise(shape, g).requires_grad_(grads)
        s["weights"] = _ctf2(c, g).requires_grad_(grads) if c["weights"] else None
        if grads:
            s["up"] = _noise(rec_shape, g)
            s["up_w"] = _noise(rec_shape, g, False) if c["weights"] else None
    return s


def run(s):
    c = s["case"]
    if c["kind"] == "prepare":
        return [fourier.to_fourier(s["map"], c["os"]),
                fourier.reconstruct(s["data"], s["weight"], c["os"], reg=REG)]
    if c["kind"].startswith("project"):
        op = tp.project_2d_forw if c["dim"] == 2 else tp.project_3d_to_2d_forw
        out = op(s["rec"], s["rot"], s["shift"], output_shape=(c["n"], c["n"]), interpolation=s["interp"],
                 oversampling=c["os"], fourier_radius_cutoff=s["cutoff"])
        if c["kind"] == "project":
            return out
        return [out.detach(), *torch.autograd.grad(out, [s["rec"], s["rot"], s["shift"]], s["up"])]
    op = tp.backproject_2d_forw if c["dim"] == 2 else tp.backproject_2d_to_3d_forw
    data, weight = op(s["proj"], s["rot"], weights=s["weights"], shifts=s["shift"], interpolation=s["interp"],
                      oversampling=c["os"], fourier_radius_cutoff=s["cutoff"])
    if c["kind"] == "backproject":
        return [data, weight] if c["weights"] else [data]
    if c["weights"]:
        return [data.detach(), weight.detach(),
                *torch.autograd.grad([data, weight], [s["proj"], s["weights"], s["rot"], s["shift"]],
                                     [s["up"], s["up_w"]])]
    return [data.detach(), *torch.autograd.grad([data], [s["proj"], s["rot"], s["shift"]], [s["up"]])]


# ----------------------------------------------------------------------------- the same in 64 bits
def _stencil(x, cubic):
    """Offsets, weights and their derivatives of one axis: [(floor(x) + k, w, dw)]."""
    f = torch.floor(x)
    t, i = x - f, f.long()
    if not cubic:
        one = torch.ones_like(t)
        return [(i, 1 - t, -one), (i + 1, t, one)]
    out = []
    for k in range(-1, 3):  # Catmull-Rom
        s = t - k
        a = s.abs()
        inner = k in (0, 1)
        w = 1.5 * a ** 3 - 2.5 * a ** 2 + 1 if inner else -0.5 * a ** 3 + 2.5 * a ** 2 - 4 * a + 2
        d = 4.5 * a ** 2 - 5 * a if inner else -1.5 * a ** 2 + 5 * a - 4
        out.append((i + k, w, d * torch.where(s < 0, -1.0, 1.0)))
    return out


def _flat(pos, N, H):
    """Flat index of signed positions [c, r(, d)] in the half spectrum, wrapped, and the Friedel-flipped ones;
    positions on the negative half axis are mirrored.  No range checks: `pos` is clamped or masked by the caller."""
    idx = torch.zeros_like(pos[0])
    for p in reversed(pos[1:]):
        idx = idx * N + torch.where(p < 0, p + N, p)
    return idx * H + pos[0]


def _mirror(pos):
    neg = pos[0] < 0
    return [torch.where(neg, -p, p) for p in pos], neg


def _fetch(vol, pos, N, H, cubic):
    if cubic:  # the cubic sampler clamps before the Friedel flip too
        pos = [pos[0].clamp(-(H - 1), H - 1)] + [p.clamp(-N // 2 + 1, N // 2) for p in pos[1:]]
    pos, neg = _mirror(pos)
    pos = [pos[0].clamp(max=H - 1)] + [p.clamp(-N // 2 + 1, N // 2) for p in pos[1:]]
    v = vol[_flat(pos, N, H)]
    return torch.where(neg, v.conj(), v) if v.is_complex() else v


def _in_range(pos, N, H):
    ok = pos[0] < H
    for p in pos[1:]:
        ok = ok & (p <= N // 2) & (p >= -N // 2 + 1)
    return ok


def _products(axes):
    """Taps of the tensor-product stencil: positions, the weight, and the weight with one axis' derivative."""
    import itertools
    for combo in itertools.product(*axes):
        w = combo[0][1]
        for a in combo[1:]:
            w = w * a[1]
        dws = []
        for k in range(len(combo)):
            d = combo[k][2]
            for j, a in enumerate(combo):
                if j != k:
                    d = d * a[1]
            dws.append(d)
        yield [a[0] for a in combo], w, dws


def _add(dst, idx, val):
    """dst[idx] += val, `dst` a flat real or complex tensor."""
    if val.is_complex():
        torch.view_as_real(dst).index_add_(0, idx, torch.view_as_real(val.contiguous()))
    else:
        dst.index_add_(0, idx, val)


def exact(c, seed):
    s = prepare(c, seed)
    if c["kind"] == "prepare":
        dim, n, N = c["dim"], c["n"], _box(c)
        axes, lo = tuple(range(-dim, 0)), (N - n) // 2
        x = torch.nn.functional.pad(s["map"].double(), (lo, N - n - lo) * dim)
        spec = torch.fft.rfftn(torch.fft.fftshift(x, dim=axes), dim=axes, norm="forward").contiguous()
        y = torch.fft.irfftn(s["data"].to(torch.complex128) / (s["weight"].double() + REG), s=[N] * dim, dim=axes,
                             norm="forward")
        m = int(N / c["os"])
        at = (N - m) // 2
        y = torch.fft.ifftshift(y, dim=axes)[(slice(None),) + (slice(at, at + m),) * dim]
        return [spec, y.contiguous()]
    if c["B"] * c["P"] * _active(c) * (4 if c["cubic"] else 2) ** c["dim"] > 1.5e9:
        return None
    n, dim, N, cubic = c["n"], c["dim"], _box(c), c["cubic"]
    H, hp, B, P = N // 2 + 1, n // 2 + 1, c["B"], c["P"]
    rot, shift = s["rot"].detach().double(), s["shift"].detach().double()
    i = torch.arange(n, device="cuda", dtype=torch.float64)
    freq = torch.where(i <= n // 2, i, i - n)
    R2, C2 = torch.meshgrid(freq, torch.arange(hp, device="cuda", dtype=torch.float64), indexing="ij")
    cut = c["cutoff"] or n / 2
    keep = R2 ** 2 + C2 ** 2 <= cut * cut
    once = keep & ~((C2 == 0) & (torch.arange(n, device="cuda")[:, None] >= n // 2))  # without the Friedel half
    size = N ** (dim - 1) * H
    cd, rd = torch.complex128, torch.float64
    step = max(1, int(2_000_000 // (n * hp)))

    def chunks(mask):
        """Active samples of each chunk of poses: (batch, poses, r, c, positions' stencils, phase)."""
        r, q = R2[mask], C2[mask]
        for b in range(B):
            for p0 in range(0, P, step):
                R, S = rot[b, p0:p0 + step], shift[b, p0:p0 + step]
                x = [(R[:, k, 0, None] * q + R[:, k, 1, None] * r) * c["os"] for k in range(dim)]
                ph = torch.polar(torch.ones_like(x[0]), -2 * math.pi / n * (r * S[:, 0, None] + q * S[:, 1, None]))
                yield b, slice(p0, p0 + R.shape[0]), r, q, x, ph

    def gather(vol, x, grads):
        axes, v = [_stencil(a, cubic) for a in x], 0
        d = [0] * dim
        for pos, w, dws in _products(axes):
            t = _fetch(vol, pos, N, H, cubic)
            v = v + t * w
            if grads:
                d = [d[k] + t * dws[k] for k in range(dim)]
        return v, d

    def scatter(dst, val, x, mirror, absolute=False):
        for pos, w, _ in _products([_stencil(a, cubic) for a in x]):
            pos, neg = _mirror(pos)
            t = val * (w.abs() if absolute else w)
            if t.is_complex():
                t = torch.where(neg, t.conj(), t)
            t = torch.where(_in_range(pos, N, H), t, torch.zeros_like(t))
            idx = torch.where(_in_range(pos, N, H), _flat(pos, N, H), torch.zeros_like(pos[0]))
            _add(dst, idx.reshape(-1), t.reshape(-1))
            if mirror:  # the Hermitian partner of a cell at c = 0
                other = [pos[0]] + [-p for p in pos[1:]]
                at = (pos[0] == 0) & _in_range(pos, N, H)
                for p in other[1:]:  # -N/2 and N/2 are the same row
                    p[p == -N // 2] = N // 2
                partner = _flat(other, N, H)
                at = at & (partner != idx)
                u = t.conj() if t.is_complex() else t
                if at.any():
                    _add(dst, partner[at], u[at])

    def pose_sums(g_rot, g_shift, b, at, r, q, a, da, e, m):
        """Re(a conj(dF/dx_k s)) and Re(e conj(-2 pi i k / n m)), summed over each pose's pixels."""
        for k in range(dim):
            t = (a * da[k].conj()).real
            g_rot[b, at, k, 0] = (t * q).sum(1) * c["os"]
            g_rot[b, at, k, 1] = (t * r).sum(1) * c["os"]
        t = (e.imag * m.real - e.real * m.imag) * (-2 * math.pi / n)
        g_shift[b, at, 0], g_shift[b, at, 1] = (t * r).sum(1), (t * q).sum(1)

    shape = (B, P, n, hp)
    rec_shape = (B, *[N] * (dim - 1), H)
    g_rot, g_shift = torch.zeros_like(rot), torch.zeros_like(shift)
    if c["kind"].startswith("project"):
        rec = s["rec"].detach().to(torch.complex64).to(cd).reshape(B, -1)
        out = torch.zeros(shape, dtype=cd, device="cuda")
        for b, at, r, q, x, ph in chunks(keep):
            out[b, at, keep] = gather(rec[b], x, False)[0] * ph
        if c["kind"] == "project":
            return out
        g_rec = torch.zeros(B, size, dtype=cd, device="cuda")
        for b, at, r, q, x, ph in chunks(once):
            g = s["up"][b, at][:, once].to(cd)
            scatter(g_rec[b], g * ph.conj(), x, False)
            v, d = gather(rec[b], x, True)
            pose_sums(g_rot, g_shift, b, at, r, q, g * ph.conj(), d, g, v * ph)
        return [out, g_rec.reshape(rec_shape), g_rot, g_shift]
    data = torch.zeros(B, size, dtype=cd, device="cuda")
    weight = torch.zeros(B, size, dtype=rd, device="cuda") if c["weights"] else None
    for b, at, r, q, x, ph in chunks(once):
        scatter(data[b], s["proj"].detach()[b, at][:, once].to(cd) * ph.conj(), x, True)
        if c["weights"]:
            scatter(weight[b], s["weights"].detach()[b, at][:, once].double(), x, True, absolute=True)
    res = [data.reshape(rec_shape)] + ([weight.reshape(rec_shape)] if c["weights"] else [])
    if c["kind"] == "backproject":
        return res
    g_proj = torch.zeros(shape, dtype=cd, device="cuda")
    g_w = torch.zeros(shape, dtype=rd, device="cuda") if c["weights"] else None
    up = s["up"].to(cd).reshape(B, -1)
    for b, at, r, q, x, ph in chunks(once):
        v, d = gather(up[b], x, True)
        g_proj[b, at, once] = v * ph
        a = s["proj"].detach()[b, at][:, once].to(cd) * ph.conj()
        pose_sums(g_rot, g_shift, b, at, r, q, a, d, a, v)
        if c["weights"]:  # linear whatever the data's interpolation
            uw, t = s["up_w"].double().reshape(B, -1)[b], 0
            for pos, w, _ in _products([_stencil(y, False) for y in x]):
                pos, _ = _mirror(pos)
                ok = _in_range(pos, N, H)
                t = t + torch.where(ok, uw[torch.where(ok, _flat(pos, N, H), torch.zeros_like(pos[0]))] * w,
                                    torch.zeros_like(w))
            g_w[b, at, once] = t
    return res + [g_proj] + ([g_w] if c["weights"] else []) + [g_rot, g_shift]
