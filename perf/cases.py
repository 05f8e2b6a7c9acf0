"""Measured cases: the work a user of the package has it do, over its range.

Every case goes through the public entry points (srf_amd.physics, recon,
autograd, batch, attenuation, psf, preprocess).  Kinds:

  tor_ops      projection and ratio backprojection of a fixed event set
               without plans, in the order the events came (a caller of the
               reference's two ops, model.projection / model.backprojection)
  osem         one OSEM iteration over planned, locality-ordered events
  reconstruct  the whole way from raw list-mode rows to an image: axis
               groups, event order, plans, iterations
  effmap       attenuated efficiency map of a scanner (every crystal pair)
  siddon_ops   Siddon projection and ratio backprojection without plans
  siddon_osem  one Siddon OSEM iteration over planned LORs
  psf          forward and backward PSF blur of one PSF-modelled step
  grad         differentiable projection, Poisson loss, image gradient
  batch        iterations of many independent reconstructions (HIP graph)

Inputs are synthetic: emission points in a cylinder with hot spheres,
isotropic directions within the scanner, crystal-snapped end points and a
Gaussian TOF error.  ``exact`` evaluates the same projector sums in float64
with plain torch.
"""
import math

import numpy as np
import torch

from srf_amd import attenuation, autograd, physics, preprocess
from srf_amd.batch import BatchedOSEM
from srf_amd.data import Image, ListModeData, split_from_groups
from srf_amd.psf import gaussian_psf
from srf_amd.recon import OSEM
from srf_amd.scanner import CylindricalScanner

DEV = "cuda"
CENTER = (0.0, 0.0, 0.0)
NO_TOF = 1.0e6  # tof_sigma2 at or above 405758 switches TOF off


def listed():
    return [
        # a caller that projects a handful of events at a time: launches and
        # host latency
        dict(name="tor_ops_2k", kind="tor_ops", grid="96x96x48", voxel="4.0x4.0x4.5",
             events=2000, kw=4.0, geo=False, tof_ps=530.0),
        # the two reference ops on a large event set in time order
        dict(name="tor_ops_400k", kind="tor_ops", grid="200x200x100", voxel="2.0x2.0x2.2",
             events=400_000, kw=4.0, geo=False, tof_ps=530.0),
        # quick-look reconstruction of a short frame, no TOF: many small subsets
        dict(name="osem_30k_notof", kind="osem", grid="96x96x48", voxel="4.0x4.0x4.5",
             events=30_000, subsets=8, kw=4.0, geo=False, tof_ps=0.0),
        # clinical-size TOF OSEM iteration at 200 x 200 x 100
        dict(name="osem_8m", kind="osem", grid="200x200x100", voxel="2.0x2.0x2.2",
             events=8_000_000, subsets=8, kw=4.0, geo=False, tof_ps=530.0),
        # large fine image, 400 ps
        dict(name="osem_6m_fine", kind="osem", grid="256x256x160", voxel="1.6x1.6x1.7",
             events=6_000_000, subsets=3, kw=4.0, geo=False, tof_ps=400.0),
        # raw list-mode rows to image: wide tube (8 mm, geometric width) on an
        # odd-sized 2 mm image
        dict(name="reconstruct_1m_kw8", kind="reconstruct", grid="181x175x83",
             voxel="2.0x2.0x2.2", events=1_000_000, subsets=4, iterations=1, kw=8.0, geo=True,
             tof_ps=530.0),
        # attenuated sensitivity of a small scanner (1.2M crystal pairs)
        dict(name="effmap_1m", kind="effmap", grid="160x160x64", voxel="2.5x2.5x2.5",
             rings=6, crystals=256, kw=4.0, geo=False),
        # the reference's Siddon op pair, TOF
        dict(name="siddon_ops_100k", kind="siddon_ops", grid="128x128x64",
             voxel="3.0x3.0x3.4", events=100_000, tof_ps=530.0),
        # Siddon OSEM iteration over coincidence LORs, no TOF
        dict(name="siddon_osem_500k", kind="siddon_osem", grid="128x128x64",
             voxel="3.0x3.0x3.4", events=500_000, subsets=4, tof_ps=0.0),
        # PSF blur pair of a PSF-modelled OSEM step
        dict(name="psf_200", kind="psf", grid="200x200x100", voxel="2.0x2.0x2.2",
             fwhm_xy=4.0, fwhm_z=4.4),
        # gradient of the list-mode Poisson likelihood
        dict(name="grad_1m", kind="grad", grid="128x128x64", voxel="3.0x3.0x3.4",
             events=1_000_000, kw=4.0, geo=False, tof_ps=530.0),
        # a set of small reconstructions advanced together
        dict(name="batch_12", kind="batch", grid="128x128x64", voxel="3.0x3.0x3.4",
             recons=12, events=60_000, growth=1.2, subsets=4, iterations=1, kw=4.0, geo=False,
             tof_ps=530.0),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _image(rng, lo=80, hi=200):
    nx, ny = rng.randint(lo, hi), rng.randint(lo, hi)
    nz = rng.randint(lo // 2, hi // 2)
    pitch = rng.uniform(384.0, 410.0) / max(nx, ny)
    return dict(grid=f"{nx}x{ny}x{nz}",
                voxel=f"{pitch:.4f}x{pitch:.4f}x{rng.uniform(1.0, 1.2) * pitch:.4f}")


def draw(rng):
    """One more case of the listed ones' ranges."""
    kind = rng.choice(["tor_ops", "osem", "osem", "reconstruct", "effmap", "siddon_ops",
                       "siddon_osem", "psf", "grad", "batch"])
    c = dict(kind=kind, **_image(rng))
    tof = rng.choice([0.0, 400.0, 530.0, 530.0])
    tube = dict(kw=rng.choice([3.0, 4.0, 4.0, 4.0, 6.0]), geo=rng.random() < 0.25)
    if kind == "tor_ops":
        c.update(events=_logint(rng, 1000, 400_000), tof_ps=tof, **tube)
    elif kind == "osem":
        c.update(events=_logint(rng, 10_000, 4_000_000), subsets=rng.randint(2, 10),
                 tof_ps=rng.choice([400.0, 530.0]), **tube)
    elif kind == "reconstruct":
        c.update(events=_logint(rng, 50_000, 2_000_000), subsets=rng.randint(2, 8),
                 iterations=rng.randint(1, 2), tof_ps=rng.choice([400.0, 530.0]), **tube)
    elif kind == "effmap":
        c.update(rings=rng.randint(2, 6), crystals=rng.randint(150, 256),
                 kw=rng.choice([3.0, 4.0]), geo=tube["geo"])
    elif kind in ("siddon_ops", "siddon_osem"):
        c.update(events=_logint(rng, 5000, 300_000), tof_ps=tof)
        if kind == "siddon_osem":
            c.update(subsets=rng.randint(2, 8))
    elif kind == "psf":
        c.update(fwhm_xy=rng.uniform(3.0, 6.0), fwhm_z=rng.uniform(3.0, 6.0))
    elif kind == "grad":
        c.update(events=_logint(rng, 20_000, 1_500_000), tof_ps=rng.choice([400.0, 530.0]),
                 **tube)
    else:
        c.update(recons=rng.randint(3, 12), events=_logint(rng, 10_000, 100_000),
                 growth=rng.uniform(1.0, 1.25), subsets=rng.randint(2, 6), iterations=1,
                 tof_ps=rng.choice([400.0, 530.0]), **tube)
    return c


# ------------------------------------------------------------------ inputs ---

def _parse(case):
    """The case with its grid and voxel size as lists."""
    return dict(case, grid=[int(v) for v in case["grid"].split("x")],
                voxel=[float(v) for v in case["voxel"].split("x")])


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _size(case):
    return [case["grid"][k] * case["voxel"][k] for k in range(3)]


def _axes(grid, size):
    return [CENTER[k] - size[k] / 2 + (torch.arange(grid[k], dtype=torch.float64, device=DEV) + 0.5)
            * size[k] / grid[k] for k in range(3)]


def _spheres(seed, size):
    """Hot spheres (centre, radius, activity) inside the imaged cylinder."""
    r = np.random.default_rng(seed)
    rad = 0.36 * min(size[0], size[1])
    out = []
    for _ in range(6):
        rho, ph = rad * 0.8 * math.sqrt(r.uniform()), r.uniform(0, 2 * math.pi)
        out.append(((rho * math.cos(ph), rho * math.sin(ph),
                     r.uniform(-0.3, 0.3) * min(size[2], 100.0)), r.uniform(6, 20),
                    r.uniform(2, 8)))
    return out


def _activity(seed, grid, size):
    """Voxel image (float32): cylinder with hot spheres on a low background,
    zero outside the field of view."""
    X, Y, Z = torch.meshgrid(*_axes(grid, size), indexing="ij")
    r2 = X * X + Y * Y
    img = torch.where(r2 <= (0.375 * min(size[0], size[1])) ** 2, 1.0, 0.05)
    for c, r, a in _spheres(seed, size):
        img = torch.where((X - c[0]) ** 2 + (Y - c[1]) ** 2 + (Z - c[2]) ** 2 <= r * r,
                          a + 0.0 * img, img)
    img = img * (0.9 + 0.2 * torch.rand(tuple(grid), dtype=torch.float64, device=DEV,
                                        generator=_gen(seed + 1)))
    img = torch.where(r2 <= (0.49 * min(size[0], size[1])) ** 2, img, torch.zeros_like(img))
    return img.to(torch.float32).contiguous()


def _emap(grid, size):
    """Smooth inverse efficiency, zero outside the field of view."""
    X, Y, Z = torch.meshgrid(*_axes(grid, size), indexing="ij")
    r2 = (X * X + Y * Y) / (0.5 * min(size[0], size[1])) ** 2
    z2 = (Z / (0.5 * size[2])) ** 2
    e = 1.0 / ((1.2 - 0.3 * r2) * (1.3 - z2))
    return torch.where(r2 <= 0.95 ** 2, e, torch.zeros_like(e)).to(torch.float32).contiguous()


def _start(grid, size):
    return (_emap(grid, size) > 0).to(torch.float32)


def _rows(seed, n, size, tof_ps, scanner=CylindricalScanner()):
    """n list-mode rows (x1, y1, z1, x2, y2, z2, tof), float32, in random
    (time) order."""
    gen = _gen(seed)
    R, half = scanner.radius, scanner.axial_length / 2
    sigma = (tof_ps if tof_ps > 0 else 530.0) * 0.15 / 2.35482005
    sph = _spheres(seed, size)
    rad, hz = 0.375 * min(size[0], size[1]), min(half, size[2] / 2)
    w = [math.pi * rad * rad * 2 * hz] + [4 / 3 * math.pi * r ** 3 * a for _, r, a in sph]
    w = torch.tensor(w, dtype=torch.float64, device=DEV)
    ang, ring = 2 * math.pi / scanner.nb_crystals, scanner.ring_pitch + scanner.gap
    z0 = -ring * (scanner.nb_rings - 1) / 2
    uz = min(1.0, half / math.sqrt(R * R - rad * rad))
    out, have = [], 0
    rnd = lambda *s: torch.rand(*s, dtype=torch.float64, device=DEV, generator=gen)
    while have < n:
        m = int(2.6 * (n - have)) + 1024
        comp = torch.multinomial(w, m, replacement=True, generator=gen)
        u = rnd(m, 8)
        rr, ph = rad * u[:, 0].sqrt(), 2 * math.pi * u[:, 1]
        e = torch.stack([rr * ph.cos(), rr * ph.sin(), (2 * u[:, 2] - 1) * hz], 1)
        ct, pb = 2 * u[:, 3] - 1, 2 * math.pi * u[:, 4]
        st = (1 - ct * ct).sqrt()
        b = torch.stack([st * pb.cos(), st * pb.sin(), ct], 1) * u[:, 5:6] ** (1 / 3)
        for i, (c, r, _) in enumerate(sph, 1):
            e = torch.where((comp == i)[:, None],
                            torch.tensor(c, dtype=torch.float64, device=DEV) + r * b, e)
        dz, pd = (2 * u[:, 6] - 1) * uz, 2 * math.pi * u[:, 7]
        s = (1 - dz * dz).sqrt()
        d = torch.stack([s * pd.cos(), s * pd.sin(), dz], 1)
        a = d[:, 0] ** 2 + d[:, 1] ** 2
        h = e[:, 0] * d[:, 0] + e[:, 1] * d[:, 1]
        q = (h * h - a * (e[:, 0] ** 2 + e[:, 1] ** 2 - R * R)).sqrt()
        ends = []
        for t in ((-h - q) / a, (-h + q) / a):
            p = e + t[:, None] * d
            k = torch.round((p[:, 2] - z0) / ring)
            # crystals half a pitch off the axes: none lies exactly on a voxel face
            f = (torch.floor(torch.atan2(p[:, 1], p[:, 0]) / ang) + 0.5) * ang
            ends.append((torch.stack([R * f.cos(), R * f.sin(), z0 + ring * k], 1),
                         (k >= 0) & (k < scanner.nb_rings)))
        keep = ends[0][1] & ends[1][1]
        p1, p2, e = ends[0][0][keep], ends[1][0][keep], e[keep]
        L = (p2 - p1).norm(dim=1)
        t = ((e - p1) * (p2 - p1)).sum(1) / L
        err = torch.randn(L.shape[0], dtype=torch.float64, device=DEV, generator=gen)
        row = torch.cat([p1, p2, (L / 2 - t + sigma * err)[:, None]], 1)
        out.append(row[:n - have].to(torch.float32))
        have += out[-1].shape[0]
    return torch.cat(out).contiguous()


# Columns of the group frame (on_tor_lors order): op x, y, z as world axes.
OP_AXES = {"x": (1, 2, 0), "y": (0, 2, 1), "z": (0, 1, 2)}


def _groups(rows, tof_ps, tof=True):
    """Axis groups of list-mode (or, tof False, six-column map) rows:
    {axis: ([10 or 7, N] float32, input row of each output row)}; rows with a
    negative difference along the axis are swapped and follow the others."""
    r = rows.to(torch.float64)
    p1, p2 = r[:, 0:3], r[:, 3:6]
    d = (p2 - p1).abs()
    m = {"x": (d[:, 0] >= d[:, 1]) & (d[:, 0] >= d[:, 2]),
         "y": (d[:, 1] > d[:, 0]) & (d[:, 1] >= d[:, 2])}
    m["z"] = ~(m["x"] | m["y"])
    L2 = ((p2 - p1) ** 2).sum(1)
    xy = ((p2 - p1)[:, :2] ** 2).sum(1)
    f = xy * xy / (p1[:, :2] ** 2 + p2[:, :2] ** 2).sum(1) / L2 / 2
    out = {}
    for k, a in enumerate("xyz"):
        up = (p2 - p1)[:, k] >= 0
        idx = torch.cat([torch.nonzero(m[a] & up)[:, 0], torch.nonzero(m[a] & ~up)[:, 0]])
        s = up[idx][:, None]
        q1, q2 = torch.where(s, p1[idx], p2[idx]), torch.where(s, p2[idx], p1[idx])
        ax = list(OP_AXES[a])
        cols = [q1[:, ax], q2[:, ax], f[idx][:, None]]
        if tof:
            t = torch.where(s[:, 0], r[idx, 6], -r[idx, 6])
            L = L2[idx].sqrt()
            c = q1 + (0.5 - t / L)[:, None] * (q2 - q1)
            if 0 < tof_ps < 10000:
                lim = tof_ps * 0.15 / 2.35482005 * 3
                far = ((c - q1).norm(dim=1) > lim)[:, None]
                u = (q2 - q1) / L[:, None]
                q1, q2 = torch.where(far, c - lim * u, q1), torch.where(far, c + lim * u, q2)
            cols = [q1[:, ax], q2[:, ax], c[:, ax], f[idx][:, None]]
        out[a] = (torch.cat(cols, 1).to(torch.float32).t().contiguous(), idx)
    return out


def _tof(tof_ps):
    """(tof_bin, tof_sigma2) of a time resolution."""
    if tof_ps <= 0:
        return 6.0, NO_TOF
    return 6.0, (tof_ps * 0.15 / 2.35482005) ** 2


def _model(case):
    b, s2 = _tof(case.get("tof_ps", 0.0))
    return physics.SplitLoRsModel(case["kw"], case["geo"], tof_sigma2=s2, tof_bin=b)


def _scanner(case):
    """An effmap case's scanner: 108.8 mm axially whatever its ring count."""
    return CylindricalScanner(nb_rings=case["rings"], nb_crystals=case["crystals"],
                              ring_pitch=108.8 / case["rings"])


def _mu(seed, grid, size):
    """mu-map: a water ellipse of seeded axes."""
    r = np.random.default_rng(seed)
    X, Y, _ = torch.meshgrid(*_axes(grid, size), indexing="ij")
    a, b = r.uniform(0.3, 0.42) * size[0], r.uniform(0.2, 0.35) * size[1]
    return torch.where((X / a) ** 2 + (Y / b) ** 2 <= 1.0, 0.0096, 0.0).to(
        torch.float32).contiguous()


def _batch(case):
    """The reconstructions of a batch: (index, grid, event count), every third
    one at half the image size, the event counts growing."""
    return [(i, [max(8, n // 2) for n in case["grid"]] if i % 3 == 2 else case["grid"],
             int(case["events"] * case["growth"] ** i)) for i in range(case["recons"])]


def _siddon_soa(rows):
    return rows.t().contiguous()


def prepare(case, seed):
    case = _parse(case)
    kind = case["kind"]
    grid, size = case["grid"], _size(case)
    st = {"kind": kind, "case": case}
    if kind in ("tor_ops", "osem", "grad"):
        groups = {a: g for a, (g, _) in _groups(_rows(seed, case["events"], size,
                                                      case["tof_ps"]), case["tof_ps"]).items()}
        st["model"] = _model(case)
    if kind == "tor_ops":
        st["data"] = split_from_groups(groups)
        st["image"] = Image(_activity(seed, grid, size), CENTER, size)
    elif kind == "osem":
        groups, _ = preprocess.reorder_groups(groups, case["subsets"])
        st["x0"] = _start(grid, size)
        st["osem"] = OSEM(st["model"], split_from_groups(groups),
                          Image(_emap(grid, size), CENTER, size), nb_subsets=case["subsets"],
                          tiled=True)
        st["osem"].plan(Image(st["x0"], CENTER, size))
    elif kind == "reconstruct":
        st["rows"] = _rows(seed, case["events"], size, case["tof_ps"])
        st["model"] = _model(case)
        st["x0"], st["emap"] = _start(grid, size), Image(_emap(grid, size), CENTER, size)
    elif kind == "effmap":
        st["scanner"] = _scanner(case)
        st["model"] = _model(case)
        st["mu"] = Image(_mu(seed, grid, size), CENTER, size)
    elif kind in ("siddon_ops", "siddon_osem"):
        b, s2 = _tof(case["tof_ps"])
        st["model"] = physics.CompleteLoRsModel("siddon", tof_sigma2=s2, tof_bin=b)
        rows = _rows(seed, case["events"], size, case["tof_ps"])
        st["data"] = ListModeData(_siddon_soa(rows), soa=True)
        if kind == "siddon_ops":
            st["image"] = Image(_activity(seed, grid, size), CENTER, size)
        else:
            st["x0"] = _start(grid, size)
            st["osem"] = OSEM(st["model"], st["data"], Image(_emap(grid, size), CENTER, size),
                              nb_subsets=case["subsets"], tiled=True)
            st["osem"].plan(Image(st["x0"], CENTER, size))
    elif kind == "psf":
        st["psf"] = gaussian_psf(grid, size, case["fwhm_xy"], case["fwhm_z"], DEV)
        st["image"] = Image(_activity(seed, grid, size), CENTER, size)
    elif kind == "batch":
        st["recons"], st["x0"] = [], []
        for i, g, n in _batch(case):
            rows = _rows(seed + 1000 * i, n, size, case["tof_ps"])
            groups = {a: v for a, (v, _) in _groups(rows, case["tof_ps"]).items()}
            st["x0"].append(_start(g, size))
            st["recons"].append({"image": Image(st["x0"][-1].clone(), CENTER, size),
                                 "emap": Image(_emap(g, size), CENTER, size),
                                 "data": split_from_groups(groups)})
        st["batch"] = BatchedOSEM(st["recons"], _model(case), case["subsets"])
        st["batch"].set_schedule(1, 64)
        st["batch"].iterate(1)
        st["batch"].capture()
    elif kind == "grad":
        st["data"] = split_from_groups(groups)
        st["image"] = _activity(seed, grid, size)
        st["sens"] = _start(grid, size)
        st["plans"] = st["model"].make_plans(Image(st["image"], CENTER, size), st["data"])
    return st


def run(state):
    kind, case = state["kind"], state["case"]
    size = _size(case)
    if kind == "tor_ops":
        p = state["model"].projection(state["image"], state["data"])
        bp = state["model"].backprojection(p, state["image"])
        return [torch.cat([p.x.values, p.y.values, p.z.values]), bp.data]
    if kind in ("osem", "siddon_osem"):
        img = Image(state["x0"].clone(), CENTER, size)
        state["osem"].iterate(img, 1)
        return img.data
    if kind == "reconstruct":
        groups = preprocess.recon_process(state["rows"], case["tof_ps"])
        groups, _ = preprocess.reorder_groups(groups, case["subsets"])
        osem = OSEM(state["model"], split_from_groups(groups), state["emap"],
                    nb_subsets=case["subsets"], tiled=True)
        img = Image(state["x0"].clone(), CENTER, size)
        osem.iterate(img, case["iterations"])
        osem.close()
        return img.data
    if kind == "effmap":
        return attenuation.attenuated_tor_effmap(state["scanner"], state["model"], state["mu"],
                                                 case["grid"], CENTER, size, DEV)
    if kind == "siddon_ops":
        p = state["model"].projection(state["image"], state["data"])
        bp = state["model"].backprojection(p, state["image"])
        return [p.values, bp.data]
    if kind == "psf":
        f = state["psf"].forward(state["image"])
        return [f.data, state["psf"].backward(f).data]
    if kind == "batch":
        for rc, x0 in zip(state["recons"], state["x0"]):
            rc["image"].data.copy_(x0)
        state["batch"].replay(case["iterations"])
        return [rc["image"].data for rc in state["recons"]]
    x = state["image"].clone().requires_grad_(True)
    p = autograd.project(Image(x, CENTER, size), state["data"], state["model"],
                         plans=state["plans"])
    autograd.poisson_nll(p.clamp_min(1e-7), x, state["sens"]).backward()
    return [p.detach(), x.grad]


# -------------------------------------------------------------------- work ---

def work(case):
    case = _parse(case)
    kind, grid, vox = case["kind"], case["grid"], case["voxel"]
    nvox, size = grid[0] * grid[1] * grid[2], _size(case)
    if kind == "psf":
        taps = math.pi * (3 * case["fwhm_xy"] / 2.355) ** 2 / (vox[0] * vox[1]) + \
            6 * case["fwhm_z"] / 2.355 / vox[2]
        return {"bytes": 2 * 2 * 4 * nvox, "flops": 2 * 2 * taps * nvox}
    # length of an event inside the image, mm
    tof_ps = case.get("tof_ps", 0.0)
    length = 0.6 * min(size[0], size[1])
    if tof_ps > 0:
        length = min(length, 6 * tof_ps * 0.15 / 2.355)
    if kind.startswith("siddon"):
        # per segment: step, length, multiply-add; both directions
        seg = length * (0.64 / vox[0] + 0.64 / vox[1] + 0.1 / vox[2])
        passes = case.get("subsets", 1)
        return {"bytes": 28 * case["events"] + 4 * nvox * (2 if passes == 1 else 3 * passes),
                "flops": 2 * 8 * seg * case["events"]}
    # voxels of the tube and, per voxel, distance, exponent and multiply-add
    n = case.get("events")
    if kind == "effmap":
        nc = case["rings"] * case["crystals"]
        n = nc * (nc - 1) // 2
        seg = length * (0.64 / vox[0] + 0.64 / vox[1] + 0.1 / vox[2])
        nnz = length * math.pi * (case["kw"] / 2) ** 2 / (vox[0] * vox[1] * vox[2])
        return {"bytes": 24 * n + 2 * 4 * nvox, "flops": (8 * seg + 14 * nnz) * n}
    nnz = length * math.pi * (case["kw"] / 2) ** 2 / (vox[0] * vox[1] * vox[2])
    if kind == "batch":
        n = sum(m for _, _, m in _batch(case))
        nvox = sum(g[0] * g[1] * g[2] for _, g, _ in _batch(case))
    passes = case.get("subsets", 1) * case.get("iterations", 1)
    per = 28 if kind == "reconstruct" else 40
    out = 4 * n if kind in ("tor_ops", "grad") else 0
    return {"bytes": per * n + out + 4 * nvox * (2 if passes == 1 else 3 * passes),
            "flops": 2 * 14 * nnz * n * case.get("iterations", 1)}


# ------------------------------------------------------------------- exact ---

def _tube(soa, grid, size, axis, kw, geo, tof):
    """Float64 system matrix of one axis group, in blocks: yields (event of
    each (event, slice) pair, flat world voxel [pairs, patch], weight)."""
    op = OP_AXES[axis]
    g = [grid[k] for k in op]
    h = [size[k] / grid[k] for k in op]
    lo = [CENTER[k] - size[k] / 2 for k in op]
    world = [grid[1] * grid[2], grid[2], 1]
    stride = [world[k] for k in op]
    z0 = lo[2] + h[2] / 2
    P = math.ceil((math.sqrt(2.0) * kw + h[2]) / h[0])
    r = soa.to(torch.float64)
    d = r[3:6] - r[0:3]
    a, b = torch.minimum(r[2], r[5]), torch.maximum(r[2], r[5])
    s0 = (torch.ceil((a - z0) / h[2]) - 1).clamp(0, g[2]).long()
    s1 = (torch.floor((b - z0) / h[2]) + 1).clamp(-1, g[2] - 1).long()
    cnt = (s1 - s0 + 1).clamp_min(0)
    total = torch.cumsum(cnt, 0)
    n, block = soa.shape[1], max(1, (1 << 24) // (P * P))
    ends = total.cpu().numpy()
    pos = 0
    off = torch.arange(P, device=DEV)
    while pos < n:
        base = int(ends[pos - 1]) if pos else 0
        stop = max(pos + 1, int(np.searchsorted(ends, base + block, side="right")))
        e = torch.repeat_interleave(torch.arange(pos, stop, device=DEV), cnt[pos:stop])
        first = total[pos:stop] - cnt[pos:stop] - base
        s = torch.arange(e.shape[0], device=DEV) - first[e - pos] + s0[e]
        pos = stop
        z = z0 + s.double() * h[2]
        q = (z - r[2, e]) / d[2, e]
        ok = (q > 0) & (q < 1)
        e, s, z, q = e[ok], s[ok], z[ok], q[ok]
        if e.shape[0] == 0:
            continue
        cx, cy = r[0, e] + d[0, e] * q, r[1, e] + d[1, e] * q
        L = (d[:, e] ** 2).sum(0).sqrt()
        ux, uy = d[0, e] / L, d[1, e] / L
        ix = (((cx - lo[0]) / h[0]).trunc().long() - P // 2)[:, None] + off
        iy = (((cy - lo[1]) / h[1]).trunc().long() - P // 2)[:, None] + off
        dx = cx[:, None] - (h[0] * (ix.double() + 0.5) + lo[0])
        dy = cy[:, None] - (h[1] * (iy.double() + 0.5) + lo[1])
        rc = (dx * ux[:, None])[:, None, :] + (dy * uy[:, None])[:, :, None]
        d2 = (dx * dx)[:, None, :] + (dy * dy)[:, :, None] - rc * rc
        sc = kw * kw / 36 * (r[-1, e] if geo else torch.ones_like(cx))
        inside = (d2 < 9 * sc[:, None, None]) & ((ix >= 0) & (ix < g[0]))[:, None, :] & \
            ((iy >= 0) & (iy < g[1]))[:, :, None]
        ex = -0.5 * d2 / sc[:, None, None]
        if tof is not None:
            tb, s2 = tof
            D = (r[6, e] - cx) ** 2 + (r[7, e] - cy) ** 2 + (r[8, e] - z) ** 2
            ex = ex - 0.5 * (D[:, None, None] - d2) / (s2 + tb * tb / 12)
        w = torch.where(inside, ex.exp(), torch.zeros_like(ex))
        if tof is not None:
            w = w * (tof[0] / math.sqrt(2 * math.pi * tof[1]))
        v = (ix * stride[0])[:, None, :] + (iy * stride[1])[:, :, None] + \
            (s * stride[2])[:, None, None]
        v = torch.where(inside, v, torch.zeros_like(v))
        yield e, v.reshape(e.shape[0], -1), w.reshape(e.shape[0], -1)


def _tof64(tof_ps):
    """The model's TOF parameters as the ops hold them (float32)."""
    b, s2 = _tof(tof_ps)
    return None if s2 >= 405758.0 else (float(np.float32(b)), float(np.float32(s2)))


def _frame64(case):
    """Image extent as the ops receive it (float32)."""
    return [float(np.float32(s)) for s in _size(case)]


def _project64(soa, x, case, axis, tof):
    p = torch.zeros(soa.shape[1], dtype=torch.float64, device=DEV)
    for e, v, w in _tube(soa, case["grid"], _frame64(case), axis, case["kw"], case["geo"], tof):
        p.index_add_(0, e, (w * x[v]).sum(1))
    return p


def _back64(soa, val, out, case, axis, tof):
    for e, v, w in _tube(soa, case["grid"], _frame64(case), axis, case["kw"], case["geo"], tof):
        out.index_add_(0, v.reshape(-1), (w * val[e][:, None]).reshape(-1))


def _ratio(p, floor):
    return torch.where(p > floor, 1.0 / p.clamp_min(1e-300), torch.zeros_like(p))


def _crossings(soa, grid, size, tof, step=20000):
    """Float64 Siddon segments in blocks: yields (ray slice, flat voxel, length
    factor) from the sorted crossings of each ray with every voxel face."""
    n = soa.shape[1]
    for i in range(0, n, step):
        r = soa[:, i:i + step].to(torch.float64)
        p1, d = r[0:3], r[3:6] - r[0:3]
        L = (d * d).sum(0).sqrt()
        ts = []
        tin, tout = torch.zeros_like(L), torch.ones_like(L)
        for k in range(3):
            lo, h = CENTER[k] - size[k] / 2, size[k] / grid[k]
            planes = lo + h * torch.arange(grid[k] + 1, dtype=torch.float64, device=DEV)
            dk = torch.where(d[k] == 0, torch.full_like(d[k], 1e-300), d[k])
            t = ((planes[None, :] - p1[k][:, None]) / dk[:, None]).clamp(-1.0, 2.0)
            ts.append(t)
            tin = torch.maximum(tin, torch.minimum(t[:, 0], t[:, -1]))
            tout = torch.minimum(tout, torch.maximum(t[:, 0], t[:, -1]))
        tout = torch.maximum(tin, tout)
        t = torch.cat(ts, 1)
        t = torch.minimum(torch.maximum(t, tin[:, None]), tout[:, None])
        t = torch.sort(t, 1).values
        seg = (t[:, 1:] - t[:, :-1]) * L[:, None]
        mid = 0.5 * (t[:, 1:] + t[:, :-1])
        v = torch.zeros_like(mid, dtype=torch.int64)
        for k, st in enumerate([grid[1] * grid[2], grid[2], 1]):
            q = p1[k][:, None] + mid * d[k][:, None] - (CENTER[k] - size[k] / 2)
            v += (q * (grid[k] / size[k])).floor().long().clamp(0, grid[k] - 1) * st
        f = seg / (L * L)[:, None]
        if tof is not None:
            tb, s2 = tof
            s = (L * 0.5 - r[6])[:, None] - mid * L[:, None]
            var = s2 + (seg * seg + tb * tb) / 12
            f = torch.where(s * s / var < 9, f * tb * torch.exp(-0.5 * s * s / var) /
                            torch.sqrt(2 * math.pi * var), torch.zeros_like(f))
        yield slice(i, min(n, i + step)), v, f


def _sid_project64(soa, x, case, tof):
    p = torch.empty(soa.shape[1], dtype=torch.float64, device=DEV)
    for sl, v, f in _crossings(soa, case["grid"], _frame64(case), tof):
        p[sl] = (f * x[v]).sum(1)
    return p


def _sid_back64(soa, val, out, case, tof):
    for sl, v, f in _crossings(soa, case["grid"], _frame64(case), tof):
        out.index_add_(0, v.reshape(-1), (f * val[sl][:, None]).reshape(-1))


def _parts(n, subsets):
    return [((k * n) // subsets, ((k + 1) * n) // subsets) for k in range(subsets)]


def _exact_osem(case, groups, x, tof):
    e64 = _emap(case["grid"], _size(case)).double().reshape(-1)
    K = case["subsets"]
    for _ in range(case.get("iterations", 1)):
        for k in range(K):
            bp = torch.zeros_like(x)
            for a, soa in groups.items():
                lo, hi = _parts(soa.shape[1], K)[k]
                sub = soa[:, lo:hi]
                if hi > lo:
                    _back64(sub, _ratio(_project64(sub, x, case, a, tof), 1e-7), bp, case, a, tof)
            x = x * e64 * bp
    return x


def _exact_psf(case, seed):
    (nx, ny, nz), vox = case["grid"], case["voxel"]
    size = _size(case)
    vx, vy, vz = (size[k] / case["grid"][k] for k in range(3))
    sxy, sz = case["fwhm_xy"] / 2.35482005, case["fwhm_z"] / 2.35482005
    rx, ry = math.ceil(3 * sxy / vx), math.ceil(3 * sxy / vy)
    offs = [(i, j, math.exp(-((i * vx) ** 2 + (j * vy) ** 2) / (2 * sxy * sxy)))
            for i in range(-rx, rx + 1) for j in range(-ry, ry + 1)
            if (i * vx) ** 2 + (j * vy) ** 2 <= (3 * sxy) ** 2]

    def span(n, o):  # rows whose neighbour at offset o lies inside, and the neighbours
        return slice(max(0, -o), n - max(0, o)), slice(max(0, o), n - max(0, -o))

    norm = torch.zeros(nx, ny, dtype=torch.float64, device=DEV)
    for i, j, w in offs:
        norm[span(nx, i)[0], span(ny, j)[0]] += w
    k = torch.arange(nz, dtype=torch.float64, device=DEV)
    dz = (k[:, None] - k[None, :]) * vz
    z = torch.where(dz.abs() > 3 * sz, torch.zeros_like(dz), torch.exp(-dz * dz / (2 * sz * sz)))
    z = (z / z.sum(1, keepdim=True)).float().double()
    x = _activity(seed, case["grid"], size).double()
    f, b = torch.zeros_like(x), torch.zeros_like(x)
    xz = x @ z.t()
    for i, j, w in offs:
        (r, n), (s, m) = span(nx, i), span(ny, j)
        f[r, s] += (w / norm[r, s]).float().double()[..., None] * xz[n, m]
    fz = f @ z
    for i, j, w in offs:
        (r, n), (s, m) = span(nx, i), span(ny, j)
        b[n, m] += (w / norm[r, s]).float().double()[..., None] * fz[r, s]
    return [f, b]


def exact(case, seed):
    case = _parse(case)
    kind, grid, size = case["kind"], case["grid"], _size(case)
    if kind == "psf":
        return _exact_psf(case, seed)
    tof = _tof64(case.get("tof_ps", 0.0))
    nvox = grid[0] * grid[1] * grid[2]
    if kind == "effmap":
        sc = _scanner(case)
        table = torch.from_numpy(sc.crystal_xyz(
            np.arange(sc.nb_rings * sc.nb_crystals) // sc.nb_crystals,
            np.arange(sc.nb_rings * sc.nb_crystals) % sc.nb_crystals).astype(np.float32)).to(DEV)
        ij = torch.triu_indices(table.shape[0], table.shape[0], 1, device=DEV)
        pairs = torch.cat([table[ij[0]], table[ij[1]]], 1)
        mu = _mu(seed, grid, size).double().reshape(-1)
        line = _sid_project64(pairs.t(), mu, case, None)
        d = (pairs[:, 3:6].double() - pairs[:, 0:3].double())
        att = torch.exp(-line * (d * d).sum(1))
        out = torch.zeros(nvox, dtype=torch.float64, device=DEV)
        for a, (soa, idx) in _groups(pairs, 0.0, tof=False).items():
            if soa.shape[1]:
                _back64(soa, att[idx], out, case, a, None)
        return out.reshape(grid)
    if kind == "batch":
        out = []
        for i, g, n in _batch(case):
            rows = _rows(seed + 1000 * i, n, size, case["tof_ps"])
            groups = {a: v for a, (v, _) in _groups(rows, case["tof_ps"]).items()}
            sub = dict(case, grid=g, voxel=[size[k] / g[k] for k in range(3)])
            out.append(_exact_osem(sub, groups, _start(g, size).double().reshape(-1),
                                   tof).reshape(g))
        return out
    rows = _rows(seed, case["events"], size, case["tof_ps"])
    if kind in ("siddon_ops", "siddon_osem"):
        soa = _siddon_soa(rows)
        if kind == "siddon_ops":
            p = _sid_project64(soa, _activity(seed, grid, size).double().reshape(-1), case, tof)
            bp = torch.zeros(nvox, dtype=torch.float64, device=DEV)
            _sid_back64(soa, _ratio(p, 0.0), bp, case, tof)
            return [p, bp.reshape(grid)]
        x = _start(grid, size).double().reshape(-1)
        e64 = _emap(grid, size).double().reshape(-1)
        for lo, hi in _parts(soa.shape[1], case["subsets"]):
            bp = torch.zeros_like(x)
            sub = soa[:, lo:hi]
            _sid_back64(sub, _ratio(_sid_project64(sub, x, case, tof), 0.0), bp, case, tof)
            x = x * e64 * bp
        return x.reshape(grid)
    groups = {a: g for a, (g, _) in _groups(rows, case["tof_ps"]).items()}
    if kind in ("osem", "reconstruct"):
        x = _start(grid, size).double().reshape(-1)
        return _exact_osem(case, groups, x, tof).reshape(grid)
    x = _activity(seed, grid, size).double().reshape(-1)
    ps = [_project64(groups[a], x, case, a, tof) for a in "xyz"]
    bp = torch.zeros(nvox, dtype=torch.float64, device=DEV)
    for a, p in zip("xyz", ps):
        if p.shape[0]:
            _back64(groups[a], _ratio(p, 1e-7), bp, case, a, tof)
    if kind == "tor_ops":
        return [torch.cat(ps), bp.reshape(grid)]
    return [torch.cat(ps), _start(grid, size).double() - bp.reshape(grid)]
