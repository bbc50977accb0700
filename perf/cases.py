"""Performance cases of the LCC search: the calls a fitting program makes, over the sizes it makes
them at.

Three kinds of call:

* ``scan``: ``HipCorrelator.scan()`` on a correlator that holds a target, a template, a mask and a
  rotation set: the exhaustive search itself, what the command line and the serving loop spend their
  time in.  Output: the best-LCC map.
* ``fit``: a new model on a map that stays resident: template, mask and rotations set, the search, and
  ``Analyzer``'s rows (score, Fisher z, position, rotation matrix) in order of position, in a table
  of fixed size.
* ``shapes``: the template and the mask of an atomic model on the map's grid, before a search.

The rotation index of a voxel is read where a program reads it, at the peaks (``fit``): at a voxel
whose two best rotations score the same to the last bits either index is right, so the whole index map
is no well-defined function of the inputs (the test suite compares it where the margin is decisive).

Grids run from a 32^3 first look to maps of 240 voxels a side: the cubic sizes of the benchmark's
workloads and of the serving stream, and the 2,3,5,7-smooth shapes, odd ones among them, that the
command line's trim and extend steps leave.  Inputs are synthetic: atoms packed as in a
protein, their density as the template, the density at a random pose plus noise as the target.
"""
import math

import numpy as np
import torch

from powerfit_amd import HipCorrelator, Volume, rotations_for_angle
from powerfit_amd.analyzer import Analyzer
from powerfit_amd.volume import structure_to_shape_like

# rotations in the set that each sampling angle (degrees) selects
ROTATIONS = {60.0: 24, 45.0: 60, 36.0: 216, 28.0: 360, 20.0: 648, 15.0: 1992, 12.0: 4344, 10.0: 7416}
NOISE = 0.05             # noise of the target, of its maximum
PEAK_ROWS = 1024         # rows of the table that the peaks are kept in
MASK_THRESHOLD = 0.05    # mask: template above this share of its maximum


def _case(name, kind, shape, angle, spacing, resolution, atoms, laplace=False, core=False):
    return {"name": name, "kind": kind, "nz": shape[0], "ny": shape[1], "nx": shape[2], "angle": angle,
            "spacing": spacing, "resolution": resolution, "atoms": atoms, "laplace": laplace, "core": core}


def listed():
    return [
        # a first look at a small map with the coarsest set: launches and latency count
        _case("first_look_32", "scan", (32, 32, 32), 60.0, 2.5, 7.0, 300, laplace=True, core=True),
        # the smallest map of the serving stream, 20 degrees
        _case("stream_48", "scan", (48, 48, 48), 20.0, 2.0, 8.0, 800),
        # the CPU-sized workload: 64^3 at 10 degrees
        _case("cpu64", "scan", (64, 64, 64), 10.0, 2.0, 8.0, 1500),
        # the next model on a resident map, with its peaks
        _case("fit_70x72x98", "fit", (70, 72, 98), 15.0, 1.6, 6.5, 4000),
        # Laplace pre-filter and core-weighted mask
        _case("lc96", "scan", (96, 96, 96), 10.0, 1.5, 6.0, 5000, laplace=True, core=True),
        # odd on every axis, as trimming leaves it
        _case("grid75x81x105", "scan", (75, 81, 105), 12.0, 1.5, 6.0, 5000),
        # a serving size of no power of two
        _case("grid120", "scan", (120, 120, 120), 12.0, 1.3, 5.5, 9000),
        # the headline search: 128^3 at 10 degrees
        _case("search128", "scan", (128, 128, 128), 10.0, 1.2, 5.0, 12000),
        # a large map at fine sampling of space, coarse sampling of rotations
        _case("prec192", "scan", (192, 192, 192), 20.0, 1.0, 4.0, 25000),
        # a trimmed map beyond the common sizes, core-weighted
        _case("trimmed_150x168x180", "scan", (150, 168, 180), 28.0, 1.1, 4.5, 15000, core=True),
        # the largest: an almost whole 240-voxel map
        _case("large_216x225x240", "scan", (216, 225, 240), 36.0, 1.0, 4.0, 30000),
        # template and mask of a 12,000-atom model on a 128^3 map
        _case("shapes_128", "shapes", (128, 128, 128), 10.0, 1.2, 5.0, 12000),
    ]


def _smooth(n):
    """The smallest length >= n with no prime factor above 7."""
    while True:
        m = n
        for p in (2, 3, 5, 7):
            while m % p == 0:
                m //= p
        if m == 1:
            return n
        n += 1


def draw(rng):
    kind = rng.choices(["scan", "fit", "shapes"], [7, 2, 1])[0]
    if rng.random() < 0.35:
        shape = (rng.choice([48, 64, 72, 80, 96, 120, 128, 144, 160, 192]),) * 3
    else:
        edge = math.exp(rng.uniform(math.log(32), math.log(234)))
        shape = tuple(_smooth(max(24, round(edge * rng.uniform(0.72, 1.0)))) for _ in range(3))
    voxels = shape[0] * shape[1] * shape[2]
    angle = rng.choice([a for a, k in ROTATIONS.items() if k * voxels <= 2.5e9])
    spacing = round(rng.uniform(1.0, 2.5), 2)
    # a model that fills a good part of the map: about 1.21 * 13 cubic Angstrom an atom
    radius = 0.3 * min(shape) * spacing * rng.uniform(0.6, 1.1)
    atoms = int(min(30000, max(200, 4.19 * radius ** 3 / (1.21 * 13.0))))
    case = _case("", kind, shape, angle, spacing, round(spacing * rng.uniform(3.6, 4.6), 2), atoms,
                 laplace=rng.random() < 0.3, core=rng.random() < 0.4)
    del case["name"]
    return case


# ---- inputs -----------------------------------------------------------------------------------------
def _shape(case):
    return case["nz"], case["ny"], case["nx"]


def _atoms(case, rng):
    """Atom positions (3, n) in Angstrom about the origin, and atomic numbers."""
    n = case["atoms"]
    half = min(_shape(case)) // 2 * case["spacing"]
    compact = 1.3 * (3.0 * 1.21 * 13.0 * n / (4.0 * math.pi)) ** (1.0 / 3.0)
    radius = min(compact, 0.8 * half)
    # residues packed evenly in an ellipsoid, four atoms each, 1.2-1.9 Angstrom around the first
    residues = (n + 3) // 4
    centre = rng.standard_normal((residues, 3))
    centre *= radius * np.cbrt(rng.uniform(0, 1, (residues, 1))) / np.linalg.norm(centre, axis=1, keepdims=True)
    centre *= rng.uniform(0.6, 1.0, 3)
    side = rng.standard_normal((residues, 3, 3))
    side *= rng.uniform(1.2, 1.9, (residues, 3, 1)) / np.linalg.norm(side, axis=2, keepdims=True)
    xyz = np.concatenate([centre[:, None], centre[:, None] + side], axis=1).reshape(-1, 3)[:n]
    weights = rng.choice([6.0, 7.0, 8.0, 16.0], size=n, p=[0.6, 0.19, 0.2, 0.01])
    return (xyz - xyz.mean(axis=0)).T.copy(), weights


def _density(xyz, weights, sigma, shape):
    """Atoms at xyz (3, n; x, y, z, voxels) as Gaussians of sigma voxels, periodic."""
    pos = xyz[::-1]
    base = np.floor(pos).astype(np.int64)
    frac = pos - base
    grid = np.zeros(int(np.prod(shape)))
    for corner in np.ndindex(2, 2, 2):
        at = [np.mod(base[a] + corner[a], shape[a]) for a in range(3)]
        w = weights.copy()
        for a in range(3):
            w = w * (frac[a] if corner[a] else 1.0 - frac[a])
        grid += np.bincount((at[0] * shape[1] + at[1]) * shape[2] + at[2], weights=w, minlength=grid.size)
    grid = grid.reshape(shape)
    for axis, n in enumerate(shape):
        d = np.abs(np.arange(n)[:, None] - np.arange(n)[None, :])
        d = np.minimum(d, n - d)
        blur = np.where(d <= 4.0 * sigma, np.exp(-d * d / (2.0 * sigma * sigma)), 0.0)
        if axis == 2:
            grid = grid.reshape(-1, n) @ blur
        elif axis == 1:
            grid = np.matmul(blur, grid.reshape(shape))
        else:
            grid = blur @ grid.reshape(n, -1)
        grid = grid.reshape(shape)
    return grid


def _core(mask):
    """Core weights: how many erosions by the 6-connected cross (zero border) a voxel survives."""
    live = mask > 0
    core = np.zeros(mask.shape)
    while live.any():
        core += live
        pad = np.pad(live, 1)
        live = (live & pad[:-2, 1:-1, 1:-1] & pad[2:, 1:-1, 1:-1] & pad[1:-1, :-2, 1:-1]
                & pad[1:-1, 2:, 1:-1] & pad[1:-1, 1:-1, :-2] & pad[1:-1, 1:-1, 2:])
    return core


def _inputs(case, seed):
    """Target (float32 as a map file holds it), template, mask, rotation matrices."""
    rng = np.random.default_rng(seed)
    shape = _shape(case)
    xyz, weights = _atoms(case, rng)
    xyz = xyz / case["spacing"]
    sigma = case["resolution"] / (math.sqrt(2.0) * math.pi) / case["spacing"]
    template = _density(xyz, weights, sigma, shape)
    q = rng.standard_normal(4)
    w, x, y, z = q / np.linalg.norm(q)
    pose = np.array([[1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y)],
                     [2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x)],
                     [2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)]])
    shift = rng.uniform(0, 1, 3) * np.array(shape[::-1])
    target = _density(pose @ xyz + shift[:, None], weights, sigma, shape).astype(np.float32)
    target += np.float32(NOISE * target.max()) * rng.standard_normal(shape, dtype=np.float32)
    mask = (template > MASK_THRESHOLD * template.max()).astype(np.float64)
    if case["core"]:
        mask = _core(mask)
    return target, template, mask, rotations_for_angle(case["angle"])


def _model(case, seed):
    """Atom coordinates (3, n) in Angstrom on a map at the origin, and atomic numbers."""
    return _atoms(case, np.random.default_rng(seed))


# ---- the calls --------------------------------------------------------------------------------------
def prepare(case, seed):
    if case["kind"] == "shapes":
        xyz, weights = _model(case, seed)
        grid = Volume(np.zeros(_shape(case), np.float32), case["spacing"], (0.0, 0.0, 0.0))
        return {"case": case, "grid": grid, "xyz": xyz, "weights": weights}
    target, template, mask, rotations = _inputs(case, seed)
    corr = HipCorrelator(target, laplace=case["laplace"])
    state = {"case": case, "corr": corr}
    if case["kind"] == "scan":
        corr.template = template
        corr.mask = mask
        corr.rotations = rotations
    else:
        state.update(template=template, mask=mask, rotations=rotations)
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "shapes":
        kw = {"resolution": case["resolution"]}
        template = structure_to_shape_like(state["grid"], state["xyz"], weights=state["weights"],
                                           shape="vol", **kw)
        mask = structure_to_shape_like(state["grid"], state["xyz"], shape="mask", **kw)
        return {"template": template.array, "mask": mask.array}
    corr = state["corr"]
    if case["kind"] == "scan":
        corr.scan()
        return {"lcc": corr.lcc}
    corr.template = state["template"]
    corr.mask = state["mask"]
    corr.rotations = state["rotations"]
    corr.scan()
    found = Analyzer(corr.lcc, state["rotations"], corr.rot, voxelspacing=case["spacing"]).solutions
    rows = sorted(([float(v) for v in row] for row in found), key=lambda row: row[3:6])
    table = np.zeros((PEAK_ROWS, 15), np.float32)
    table[:len(rows)] = rows
    return {"lcc": corr.lcc, "peaks": table}


def work(case):
    nz, ny, nx = _shape(case)
    voxels, half = nz * ny * nx, nz * ny * (nx // 2 + 1)
    if case["kind"] == "shapes":
        # the 64-bit grids that come back, and the atoms' boxes
        box = (2.0 * 4.0 * case["resolution"] / (math.sqrt(2.0) * math.pi) / case["spacing"]) ** 3
        return {"bytes": 16 * voxels + 32 * case["atoms"], "flops": case["atoms"] * box * 12}
    # per rotation: two samplings (about 40 operations a voxel of the sphere), the spectra of the
    # template and the mask (and of its square where it is weighted), three products and inverse
    # transforms, the score; template, mask, target spectra and result once
    forward = 3 if case["core"] else 2
    sphere = 4.19 * (min(nz, ny, nx) // 2) ** 3
    fft = 2.5 * voxels * math.log2(voxels)
    flops = ROTATIONS[case["angle"]] * ((forward + 3) * fft + 40 * sphere + 18 * half + 6 * voxels)
    return {"bytes": 8 * voxels + 16 * half + voxels + 8 * voxels, "flops": flops}


# ---- the same in 64 bits ----------------------------------------------------------------------------
def _laplace(a):
    return sum(np.roll(a, s, axis) for axis in range(3) for s in (1, -1)) - 6.0 * a


def _exact_lcc(case, seed, device):
    target, template, mask, rotations = _inputs(case, seed)
    shape = _shape(case)
    target = target.astype(np.float64)
    target = target / target.max()
    where = target > 0.05 * target.max()
    inside = mask != 0
    if case["laplace"]:
        target, template = _laplace(target), _laplace(template)
    template = template * mask
    template[inside] -= template[inside].mean()
    template[inside] /= template[inside].std()
    template = template * mask
    count = float(inside.sum())

    def put(a):
        return torch.from_numpy(np.ascontiguousarray(a)).to(device)

    radius = min(shape) // 2
    t, m, target = put(template).reshape(-1), put(mask).reshape(-1), put(target)
    spectrum, spectrum2 = torch.fft.rfftn(target), torch.fft.rfftn(target * target)
    # voxels of the rotation sphere, by signed coordinates
    signed = [torch.arange(n, device=device) for n in shape]
    signed = [torch.where(s <= radius, s, s - n) for s, n in zip(signed, shape)]
    near = (signed[0][:, None, None] ** 2 + signed[1][None, :, None] ** 2
            + signed[2][None, None, :] ** 2) <= radius * radius
    iz, iy, ix = torch.nonzero(near, as_tuple=True)
    flat = (iz * shape[1] + iy) * shape[2] + ix
    z, y, x = (signed[a][i].double() for a, i in enumerate((iz, iy, ix)))
    rotated, weight = torch.zeros_like(t), torch.zeros_like(m)
    best = torch.zeros(shape, dtype=torch.float64, device=device)
    live = put(where)
    nz, ny, nx = shape

    def at(values, a, b, c):
        return values[(torch.remainder(a, nz) * ny + torch.remainder(b, ny)) * nx + torch.remainder(c, nx)]

    def nearest(v):
        whole = torch.trunc(v)
        part = v - whole
        return (whole + (part >= 0.5).double() - (part <= -0.5).double()).long()

    for rot in rotations.tolist():
        xs, ys, zs = ((z * rot[2][k] + y * rot[1][k]) + x * rot[0][k] for k in range(3))
        x0, y0, z0 = (torch.floor(v) for v in (xs, ys, zs))
        dx, dy, dz = xs - x0, ys - y0, zs - z0
        i, j, k = z0.long(), y0.long(), x0.long()
        value = torch.zeros_like(xs)
        for a in (0, 1):
            for b in (0, 1):
                for c in (0, 1):
                    value += (at(t, i + a, j + b, k + c) * (dz if a else 1 - dz) * (dy if b else 1 - dy)
                              * (dx if c else 1 - dx))
        rotated[flat] = value
        weight[flat] = at(m, nearest(zs), nearest(ys), nearest(xs))
        p = torch.fft.rfftn(rotated.view(shape)).conj()
        w = torch.fft.rfftn(weight.view(shape)).conj()
        w2 = torch.fft.rfftn((weight * weight).view(shape)).conj() if case["core"] else w
        g, a, b = (torch.fft.irfftn(s, s=shape) for s in (p * spectrum, w * spectrum, w2 * spectrum2))
        score = g / torch.sqrt(b * count - a * a)
        best = torch.where(live & (score > best), score, best)
    return best.cpu().numpy()


def _exact_shapes(case, seed, device):
    xyz, weights = _model(case, seed)
    shape = _shape(case)
    spacing = case["spacing"]
    # a Gaussian of the resolution's sigma an atom, cut at 4 sigma, one periodic wrap
    sigma = case["resolution"] / (math.sqrt(2.0) * math.pi) / spacing
    points = torch.from_numpy(xyz / spacing).to(device)
    weights = torch.from_numpy(weights).to(device)
    reach = math.ceil(4.0 * sigma)
    off = torch.arange(-reach, reach + 1, device=device)
    oz, oy, ox = (o.reshape(-1) for o in torch.meshgrid(off, off, off, indexing="ij"))
    grid = torch.zeros(int(np.prod(shape)), dtype=torch.float64, device=device)
    for part in torch.split(torch.arange(points.shape[1], device=device), 2048):
        p = points[:, part]
        v = [torch.round(p[a])[:, None] + o[None, :] for a, o in enumerate((ox, oy, oz))]
        d2 = sum((v[a] - p[a][:, None]) ** 2 for a in range(3))
        keep = d2 <= (4.0 * sigma) ** 2
        for a in range(3):
            keep &= (v[a] > -shape[2 - a]) & (v[a] < shape[2 - a])
        val = weights[part][:, None] * torch.exp(-d2 / (2.0 * sigma * sigma))
        vx, vy, vz = (torch.remainder(v[a], shape[2 - a]).long() for a in range(3))
        grid.index_add_(0, ((vz * shape[1] + vy) * shape[2] + vx)[keep], val[keep])
    return grid.view(shape).cpu().numpy()


def exact(case, seed):
    device = "cuda" if torch.cuda.is_available() else "cpu"
    if case["kind"] == "shapes":
        return {"template": _exact_shapes(case, seed, device), "mask": None}
    lcc = _exact_lcc(case, seed, device)
    return {"lcc": lcc} if case["kind"] == "scan" else {"lcc": lcc, "peaks": None}
