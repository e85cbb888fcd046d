"""Performance cases: the projections and reconstructions that programs make with this framework.

Every case is a scan (a volume of cubic voxels, a circular or helical,
parallel or cone-beam trajectory, a detector) and one pass over it through a
public entry point:

* ``pair``      ``A(x)`` and ``A.T(y)`` of one operator;
* ``slices``    the autograd operator on a batch of 2D slices (``is_2d``);
* ``autograd``  gradient of ``|A x - y|^2`` for a batch of volumes;
* ``gradient64``  the same in float64 (finite-difference checks);
* ``sirt``      a whole SIRT reconstruction;
* ``fdk``       a whole FDK reconstruction;
* ``normal``    ``fused_normal`` over several instances;
* ``requests``  one fused launch each way over a mix of small requests.

Volumes are sums of seeded balls plus 1 % noise; projections are the exact
line integrals of such balls, so that both hold what a scan holds.
"""
import math
import random

import numpy as np
import torch

import tomosipo_amd as ts
from tomosipo_amd.fused import fused_backward, fused_forward, fused_normal
from tomosipo_amd.sirt import sirt
from tomosipo_amd.torch_support import to_autograd

DEVICE = "cuda"
BALLS = 6
EPSILON = 1e-8          # the clip of SIRT's weights: at most 1 / EPSILON
EXACT_SAMPLES = 2.4e10  # ray samples that the float64 values are computed for


def _case(name, path, beam, shape, angles, det, **more):
    nz, ny, nx = shape
    case = {"name": name, "path": path, "beam": beam, "nz": nz, "ny": ny, "nx": nx, "angles": angles,
            "rows": det[0], "cols": det[1], "pitch": 1.0 if beam == "parallel" else math.sqrt(2.0),
            "magnification": 1.0, "tilt": 0.0, "ss": 1, "batch": 1, "iterations": 0}
    case.update(more)
    return case


def listed():
    return [
        # a quick look or a unit test: one small parallel scan each way, where launches count
        _case("pair_parallel_64", "pair", "parallel", (64, 64, 64), 96, (64, 96)),
        # the ordinary cone-beam scan of a laboratory instrument, each way
        _case("pair_cone_256", "pair", "cone", (256, 256, 256), 360, (256, 384)),
        # a short stack of synchrotron slices, odd everywhere
        _case("pair_parallel_slab", "pair", "parallel", (75, 441, 441), 361, (75, 623)),
        # a scan around an axis that is tilted against the volume's
        _case("pair_tilted_192", "pair", "cone", (192, 192, 192), 240, (192, 288), tilt=0.2),
        # coarse detector pixels, 2 x 2 rays in each
        _case("pair_supersampled_128", "pair", "cone", (128, 128, 128), 180, (96, 144), ss=2,
              pitch=math.sqrt(2.0) * 4.0 / 3.0),
        # learned 2D reconstruction: a batch of slices, forward and gradient
        _case("slices_256_batch16", "slices", "parallel", (1, 256, 256), 180, (1, 384), batch=16),
        # learned 3D reconstruction: a batch of volumes, forward and gradient
        _case("autograd_parallel_128_batch8", "autograd", "parallel", (128, 128, 128), 180, (128, 192), batch=8),
        # gradient check in double precision
        _case("gradient64_32", "gradient64", "parallel", (32, 32, 32), 48, (32, 48)),
        # iterative reconstruction of the ordinary scan
        _case("sirt_cone_256", "sirt", "cone", (256, 256, 256), 360, (256, 384), iterations=10),
        # direct reconstruction of a large scan
        _case("fdk_cone_512", "fdk", "cone", (512, 512, 512), 720, (512, 768)),
        # throughput: large helical instances, each forward and back
        _case("normal_helix_512", "normal", "helix", (512, 512, 512), 720, (512, 768), batch=2),
        # a server's batch of small requests of both beams, each way
        _case("requests_128", "requests", "mixed", (128, 128, 128), 180, (128, 192), batch=8),
    ]


def draw(rng):
    path = rng.choice(["pair_parallel", "pair_cone", "pair_slab", "pair_tilted", "pair_supersampled", "slices",
                       "autograd", "gradient64", "sirt", "fdk", "normal", "requests"])

    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def cube(lo, hi):
        # near-cubic volumes: equal sides half of the time
        n = size(lo, hi)
        if rng.random() < 0.5:
            return n, n, n
        return tuple(max(lo // 2, int(n * rng.uniform(0.75, 1.1))) for _ in range(3))

    def detector(shape):
        return int(shape[0] * rng.uniform(0.85, 1.15)), int(max(shape[1:]) * rng.uniform(1.1, 1.55))

    def angles(lo, hi):
        return size(lo, hi)

    if path == "pair_parallel":
        s = cube(48, 256)
        return _case("", "pair", "parallel", s, angles(48, 360), detector(s), pitch=rng.choice([1.0, math.sqrt(2.0)]))
    if path == "pair_cone":
        s = cube(48, 320)
        return _case("", "pair", rng.choice(["cone", "helix"]), s, angles(48, 400), detector(s),
                     magnification=rng.choice([1.0, 1.6]))
    if path == "pair_slab":
        n = size(128, 640)
        s = (size(8, 96), n, n + rng.randrange(-16, 17))
        return _case("", "pair", rng.choice(["parallel", "cone"]), s, angles(64, 400), detector(s))
    if path == "pair_tilted":
        s = cube(32, 200)
        return _case("", "pair", rng.choice(["parallel", "cone"]), s, angles(32, 260), detector(s),
                     tilt=round(rng.uniform(0.05, 0.4), 3))
    if path == "pair_supersampled":
        s = cube(32, 160)
        ss = rng.choice([2, 3])
        det = tuple(max(8, d * 3 // 4) for d in detector(s))
        return _case("", "pair", rng.choice(["parallel", "cone"]), s, angles(32, 200), det, ss=ss,
                     pitch=math.sqrt(2.0) * 4.0 / 3.0)
    if path == "slices":
        n = size(64, 512)
        s = (1, n, n)
        return _case("", "slices", "parallel", s, angles(45, 360), (1, detector(s)[1]), batch=size(1, 32))
    if path == "autograd":
        s = cube(48, 144)
        return _case("", "autograd", rng.choice(["parallel", "cone"]), s, angles(48, 200), detector(s),
                     batch=rng.randrange(2, 9))
    if path == "gradient64":
        s = cube(12, 40)
        return _case("", "gradient64", rng.choice(["parallel", "cone"]), s, angles(16, 64), detector(s))
    if path == "sirt":
        s = cube(64, 224)
        return _case("", "sirt", rng.choice(["parallel", "cone"]), s, angles(60, 300), detector(s),
                     iterations=rng.randrange(3, 16))
    if path == "fdk":
        s = cube(96, 400)
        return _case("", "fdk", "cone", s, angles(120, 720), detector(s))
    if path == "normal":
        s = cube(128, 288)
        return _case("", "normal", "helix", s, angles(120, 400), detector(s), batch=rng.randrange(2, 5))
    n = size(64, 144)
    return _case("", "requests", "mixed", (n, n, n), angles(60, 200), (n, n + n // 2), batch=rng.randrange(4, 13))


# ---------------------------------------------------------------------------
# geometry
# ---------------------------------------------------------------------------

def _parts(case):
    """The scans of a case: itself, or the requests of a mix (sides from half of
    the case's to all of it, other angle counts, the beams in turn)."""
    if case["path"] != "requests":
        return [case]
    rng = random.Random(9)
    parts = []
    for k in range(case["batch"]):
        n = int(case["nx"] * rng.choice([0.5, 0.75, 1.0]))
        part = dict(case, path="pair", beam=("cone", "parallel")[k % 2], nz=n, ny=n, nx=n, rows=n, cols=n + n // 2,
                    angles=max(8, int(case["angles"] * rng.uniform(0.35, 1.0))), pitch=math.sqrt(2.0), batch=1)
        parts.append(part)
    return parts


def _voxel(case):
    return 1.0 / max(case["nx"], case["ny"])


def _vectors(case, instance=0):
    """(ray directions or sources, detector positions, v, u), each (angles, 3) in (z, y, x)."""
    n = case["angles"]
    turn = math.pi if case["beam"] == "parallel" else 2 * math.pi
    # (the first angle is off the axes: no ray family lies exactly between two of them)
    theta = (np.arange(n) + 0.3) * turn / n
    zero, one = np.zeros(n), np.ones(n)
    along = np.stack([zero, np.cos(theta), np.sin(theta)], axis=1)
    u = np.stack([zero, -np.sin(theta), np.cos(theta)], axis=1)
    v = np.stack([one, zero, zero], axis=1)
    pixel = case["pitch"] * _voxel(case) * case["magnification"]
    if case["beam"] == "parallel":
        first, det = along, 0.0 * along
    else:
        distance = 2.0 * math.sqrt(2.0)
        first, det = -distance * along, (case["magnification"] - 1.0) * distance * along
    if case["beam"] == "helix":
        rng = np.random.default_rng(1000 + instance)
        first = first + rng.normal(0.0, 1e-3, size=first.shape)
        first[:, 0] += np.linspace(-0.25, 0.25, n)
    if case["tilt"]:
        c, s = math.cos(case["tilt"]), math.sin(case["tilt"])
        turned = np.array([[c, 0.0, s], [0.0, 1.0, 0.0], [-s, 0.0, c]])
        first, det, u, v = (w @ turned.T for w in (first, det, u, v))
    return first, det, pixel * v, pixel * u


def _operator(case, instance=0):
    first, det, v, u = _vectors(case, instance)
    h = _voxel(case)
    vg = ts.volume(shape=(case["nz"], case["ny"], case["nx"]), size=(case["nz"] * h, case["ny"] * h, case["nx"] * h))
    shape = (case["rows"], case["cols"])
    if case["beam"] == "parallel":
        pg = ts.parallel_vec(shape=shape, ray_dir=first, det_pos=det, det_v=v, det_u=u)
    else:
        pg = ts.cone_vec(shape=shape, src_pos=first, det_pos=det, det_v=v, det_u=u)
    return ts.operator(vg, pg, detector_supersampling=case["ss"])


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _balls(case, seed):
    """Centres, radii and densities of seeded balls within the scanned region."""
    rng = np.random.default_rng([7, seed])
    h = _voxel(case)
    half = 0.5 * h * np.array([case["nz"], case["ny"], case["nx"]])
    reach = float(min(half[1], half[2]))
    radius = rng.uniform(0.1, 0.4, BALLS) * reach
    at = rng.uniform(-0.55, 0.55, (BALLS, 3)) * np.array([half[0], reach, reach])
    return at, radius, rng.uniform(0.3, 1.5, BALLS)


def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _volume(case, seed, dtype=torch.float32):
    h = _voxel(case)
    shape = (case["nz"], case["ny"], case["nx"])
    z, y, x = ((torch.arange(n, device=DEVICE, dtype=torch.float32) + 0.5 - 0.5 * n) * h for n in shape)
    vol = torch.randn(shape, generator=_generator(seed), device=DEVICE) * 0.01
    for (cz, cy, cx), r, d in zip(*_balls(case, seed)):
        inside = ((z - cz) ** 2)[:, None, None] + ((y - cy) ** 2)[:, None] + (x - cx) ** 2 < r * r
        vol += d * inside
    return vol.to(dtype)


def _projections(case, seed, instance=0, dtype=torch.float32):
    """Line integrals of the balls along the rays through the pixel centres, with 1 % noise."""
    first, det, v, u = (torch.from_numpy(w).to(DEVICE) for w in _vectors(case, instance))
    rows, cols, n = case["rows"], case["cols"], case["angles"]
    at, radius, density = _balls(case, seed)
    i = torch.arange(rows, device=DEVICE, dtype=torch.float64) - 0.5 * (rows - 1)
    j = torch.arange(cols, device=DEVICE, dtype=torch.float64) - 0.5 * (cols - 1)
    out = torch.randn((rows, n, cols), generator=_generator(seed), device=DEVICE) * 0.01
    step = max(1, int(2 ** 24 // (rows * cols)))
    for a in range(0, n, step):
        part = slice(a, min(n, a + step))
        p = [det[part, k, None] + j * u[part, k, None] + i[:, None, None] * v[part, k, None] for k in range(3)]
        if case["beam"] == "parallel":
            w = [first[part, k, None] for k in range(3)]
        else:
            w = [p[k] - first[part, k, None] for k in range(3)]
        ww = w[0] ** 2 + w[1] ** 2 + w[2] ** 2
        for k in range(len(radius)):
            c = [at[k][e] - p[e] for e in range(3)]
            cw = c[0] * w[0] + c[1] * w[1] + c[2] * w[2]
            apart = c[0] ** 2 + c[1] ** 2 + c[2] ** 2 - cw ** 2 / ww
            out[:, part] += (2 * density[k] * torch.sqrt(torch.clamp(radius[k] ** 2 - apart, min=0.0))).float()
    return out.to(dtype)


def _one(case, seed):
    """A case's volume and projections of one instance (other balls in the two)."""
    return _volume(case, 2 * seed), _projections(case, 2 * seed + 1)


def prepare(case, seed):
    path, batch = case["path"], case["batch"]
    if path == "requests":
        parts = _parts(case)
        ops = [_operator(p) for p in parts]
        for op in ops:
            op.projector.plan(torch.cuda.current_device())
        data = [_one(p, 1000 * seed + k) for k, p in enumerate(parts)]
        return {"path": path, "ops": ops, "xs": [d[0] for d in data], "ys": [d[1] for d in data]}
    if path == "normal":
        ops = [_operator(case, k) for k in range(batch)]
        for op in ops:
            op.projector.plan(torch.cuda.current_device())
        return {"path": path, "ops": ops, "xs": [_volume(case, 1000 * seed + k) for k in range(batch)],
                "ys": [torch.empty(op.range_shape, device=DEVICE) for op in ops],
                "bs": [torch.empty(op.domain_shape, device=DEVICE) for op in ops]}
    A = _operator(case)
    A.projector.plan(torch.cuda.current_device())
    if path == "pair":
        x, y = _one(case, seed)
        return {"path": path, "A": A, "x": x, "y": y, "out_y": torch.empty(A.range_shape, device=DEVICE),
                "out_x": torch.empty(A.domain_shape, device=DEVICE)}
    if path == "sirt":
        return {"path": path, "A": A, "y": _projections(case, seed), "iterations": case["iterations"]}
    if path == "fdk":
        return {"path": path, "A": A, "y": _projections(case, seed),
                "out": torch.empty(A.domain_shape, device=DEVICE)}
    if path == "gradient64":
        return {"path": "autograd", "f": to_autograd(A, dtype=torch.float64),
                "x": _volume(case, 2 * seed, torch.float64).requires_grad_(),
                "y": _projections(case, 2 * seed + 1, dtype=torch.float64)}
    data = [_one(case, 1000 * seed + k) for k in range(batch)]
    x, y = torch.stack([d[0] for d in data]), torch.stack([d[1] for d in data])
    if path == "slices":  # (batch, channel, rows, columns) images
        f = to_autograd(A, num_extra_dims=2, is_2d=True)
        x, y = x, y.transpose(1, 2).reshape(batch, 1, case["angles"], case["cols"]).contiguous()
    else:
        f = to_autograd(A, num_extra_dims=1)
    return {"path": "autograd", "f": f, "x": x.contiguous().requires_grad_(), "y": y}


def run(state):
    path = state["path"]
    if path == "pair":
        A = state["A"]
        A(state["x"], out=state["out_y"])
        A.T(state["y"], out=state["out_x"])
        return [state["out_y"], state["out_x"]]
    if path == "autograd":
        x = state["x"]
        x.grad = None
        projected = state["f"](x)
        loss = torch.sum((projected - state["y"]) ** 2)
        loss.backward()
        return [projected.detach(), x.grad]
    if path == "sirt":
        return sirt(state["A"], state["y"], state["iterations"])
    if path == "fdk":
        return ts.fdk(state["A"], state["y"], out=state["out"])
    if path == "normal":
        ys, bs = fused_normal(state["ops"], state["xs"], state["ys"], state["bs"], groups=len(state["ops"]))
        return [ys, bs]
    return [fused_forward(state["ops"], state["xs"]), fused_backward(state["ops"], state["ys"])]


# ---------------------------------------------------------------------------
# the work of a pass
# ---------------------------------------------------------------------------

def _sizes(case):
    volume = case["nz"] * case["ny"] * case["nx"]
    pixels = case["rows"] * case["angles"] * case["cols"]
    # samples of the rays that meet the volume: one for each slice that a ray crosses, about one
    # ray for each pixel of the volume's shadow (or, where it is smaller, of the detector)
    side = max(case["nx"], case["ny"])
    rows = min(case["rows"], case["nz"] / case["pitch"]) * case["ss"]
    cols = min(case["cols"], 1.2 * side / case["pitch"]) * case["ss"]
    return volume, pixels, rows * cols * case["angles"] * side * 0.8


def work(case):
    if case["path"] == "requests":
        parts = [work(p) for p in _parts(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    volume, pixels, samples = _sizes(case)
    each = 4.0 * (volume + pixels)
    # 14 operations for a bilinear sample, in each direction
    if case["path"] == "pair":
        return {"bytes": 2 * each, "flops": 28 * samples}
    if case["path"] in ("slices", "autograd", "gradient64"):
        # x and y in, the projections and the gradient out
        size = 2.0 if case["path"] == "gradient64" else 1.0
        return {"bytes": 2 * each * case["batch"] * size, "flops": 28 * samples * case["batch"]}
    if case["path"] == "normal":
        # x in, its projections and their backprojection out
        return {"bytes": (2 * 4.0 * volume + 4.0 * pixels) * case["batch"], "flops": 28 * samples * case["batch"]}
    if case["path"] == "sirt":
        return {"bytes": each, "flops": 28 * samples * (case["iterations"] + 1)}
    # fdk: the ramp filter (two multiply-adds for each output and tap pair) and 11 operations for a voxel and angle
    return {"bytes": each, "flops": 11.0 * volume * case["angles"] + 2.0 * pixels * 20}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

def _grid(case, instance=0):
    """Ray family in grid units (voxel centres on the integers), (z, y, x)."""
    h = _voxel(case)
    lo = -0.5 * h * np.array([case["nz"], case["ny"], case["nx"]])
    first, det, v, u = _vectors(case, instance)
    s = first / h if case["beam"] == "parallel" else (first - lo) / h - 0.5
    ray = s if case["beam"] == "parallel" else (det - first) / h
    return s, (det - lo) / h - 0.5, v / h, u / h, ray


def _samples(case, instance, a, grid):
    """The slices of angle a in chunks: (axes, slices, flat index and weight of each sample's lower
    corner in a volume with one zero voxel below and two above, length of a step)."""
    s, det, v, u, ray = (w[a] for w in grid)
    size = [case["nz"], case["ny"], case["nx"]]
    m = max(range(3), key=lambda k: (abs(ray[k]), k))  # (z, y, x): x before y before z where equal
    p, q = [k for k in range(3) if k != m]
    ss, rows, cols = case["ss"], case["rows"] * case["ss"], case["cols"] * case["ss"]
    i = (torch.arange(rows, device=DEVICE, dtype=torch.float64) + 0.5) / ss - 0.5 * case["rows"]
    j = (torch.arange(cols, device=DEVICE, dtype=torch.float64) + 0.5) / ss - 0.5 * case["cols"]
    point = [det[k] + i[:, None] * v[k] + j * u[k] for k in range(3)]
    if case["beam"] == "parallel":
        step = [torch.full_like(point[0], s[k] / s[m]) for k in (p, q)]
    else:
        step = [(point[k] - s[k]) / (point[m] - s[m]) for k in (p, q)]
    h = _voxel(case)
    length = h * torch.sqrt(1.0 + step[0] ** 2 + step[1] ** 2)
    many = max(1, int(2 ** 24 // (rows * cols)))
    for n0 in range(0, size[m], many):
        n = torch.arange(n0, min(size[m], n0 + many), device=DEVICE, dtype=torch.float64)[:, None, None]
        index, weight = n.long(), []
        for k, d in ((p, step[0]), (q, step[1])):
            at = torch.clamp(point[k] + (n - point[m]) * d, -1.0, float(size[k]))
            low = torch.floor(at)
            weight.append(at - low)
            index = index * (size[k] + 3) + (low.long() + 1)
        yield (m, p, q), index, weight, length, size[q] + 3


def _turned(volume, axes):
    return torch.nn.functional.pad(volume.permute(*axes), (1, 2, 1, 2)).contiguous()


def _forward64(case, volume, instance=0):
    grid = _grid(case, instance)
    ss = case["ss"]
    out = torch.zeros((case["rows"], case["angles"], case["cols"]), device=DEVICE, dtype=torch.float64)
    layouts = {}
    for a in range(case["angles"]):
        total = 0.0
        for axes, index, (wp, wq), length, row in _samples(case, instance, a, grid):
            if axes not in layouts:
                layouts[axes] = _turned(volume.double(), axes)
            flat = layouts[axes].view(-1)
            near = torch.lerp(flat[index], flat[index + 1], wq)
            far = torch.lerp(flat[index + row], flat[index + row + 1], wq)
            total = total + torch.lerp(near, far, wp).sum(0)
        line = length * total
        out[:, a] = line.view(case["rows"], ss, case["cols"], ss).mean(dim=(1, 3))
    return out


def _backward64(case, projections, instance=0):
    grid = _grid(case, instance)
    ss = case["ss"]
    sums = {}
    size = (case["nz"], case["ny"], case["nx"])
    for a in range(case["angles"]):
        y = projections[:, a].double().repeat_interleave(ss, 0).repeat_interleave(ss, 1) / ss ** 2
        for axes, index, (wp, wq), length, row in _samples(case, instance, a, grid):
            if axes not in sums:
                m, p, q = axes
                sums[axes] = torch.zeros((size[m], size[p] + 3, size[q] + 3), device=DEVICE, dtype=torch.float64)
            flat = sums[axes].view(-1)
            ly = length * y
            for offset, w in ((0, (1 - wp) * (1 - wq)), (1, (1 - wp) * wq), (row, wp * (1 - wq)), (row + 1, wp * wq)):
                flat.index_add_(0, (index + offset).reshape(-1), (w * ly).reshape(-1))
    out = torch.zeros(size, device=DEVICE, dtype=torch.float64)
    for axes, padded in sums.items():
        inner = padded[:, 1:-2, 1:-2]
        out += inner.permute(*[axes.index(k) for k in range(3)])
    return out


def _sirt64(case, y, iterations):
    ones_x = torch.ones((case["nz"], case["ny"], case["nx"]), device=DEVICE, dtype=torch.float64)
    r = torch.clamp(1.0 / _forward64(case, ones_x), max=1.0 / EPSILON)
    c = torch.clamp(1.0 / _backward64(case, torch.ones_like(y, dtype=torch.float64)), max=1.0 / EPSILON)
    x = torch.zeros_like(ones_x)
    for _ in range(iterations):
        x = x + c * _backward64(case, r * (y.double() - _forward64(case, x)))
    return x


def _fdk64(case, y):
    """Feldkamp reconstruction: cosine weights, sampled Ram-Lak filter along the rows, bilinear
    backprojection with weight (step / 2) (D / U)^2, on the detector plane through the origin."""
    first, det, v, u = _vectors(case)
    n, rows, cols, h = case["angles"], case["rows"], case["cols"], _voxel(case)
    lag = np.arange(-(cols - 1), cols)
    kernel = np.where(lag == 0, 0.25, 0.0)
    odd = lag % 2 != 0
    kernel[odd] = -1.0 / (math.pi ** 2 * lag[odd].astype(np.float64) ** 2)
    length = 1 << (3 * cols - 2).bit_length()
    response = torch.fft.rfft(torch.from_numpy(kernel).to(DEVICE), n=length)
    z, yy, x = ((torch.arange(k, device=DEVICE, dtype=torch.float64) + 0.5 - 0.5 * k) * h
                for k in (case["nz"], case["ny"], case["nx"]))
    i = torch.arange(rows, device=DEVICE, dtype=torch.float64) - 0.5 * (rows - 1)
    j = torch.arange(cols, device=DEVICE, dtype=torch.float64) - 0.5 * (cols - 1)
    out = torch.zeros((case["nz"], case["ny"], case["nx"]), device=DEVICE, dtype=torch.float64)
    for a in range(n):
        distance = float(np.linalg.norm(first[a]))
        normal = -first[a] / distance
        scale = distance / float((det[a] - first[a]) @ normal)  # to the plane through the origin
        pixel = scale * float(np.linalg.norm(u[a]))
        weight = distance / torch.sqrt(distance ** 2 + (i[:, None] * pixel) ** 2 + (j * pixel) ** 2)
        line = torch.fft.irfft(torch.fft.rfft(weight * y[:, a].double(), n=length) * response, n=length)
        filtered = torch.nn.functional.pad(line[:, cols - 1:2 * cols - 1] / pixel, (1, 1, 1, 1)).contiguous()
        unit = u[a] / np.linalg.norm(u[a])
        depth = distance + yy[:, None] * normal[1] + x * normal[2]
        near = distance / depth
        column = (near * (yy[:, None] * unit[1] + x * unit[2]) / pixel + 0.5 * (cols - 1)).clamp(-1.0, float(cols))
        jl = torch.floor(column).clamp(max=float(cols - 1))
        wj = column - jl
        row = (near * (z / pixel)[:, None, None] + 0.5 * (rows - 1)).clamp(-1.0, float(rows))
        il = torch.floor(row).clamp(max=float(rows - 1))
        flat = filtered.view(-1)
        index = (il.long() + 1) * (cols + 2) + (jl.long() + 1)
        row -= il
        low = torch.lerp(flat[index], flat[index + 1], wj)
        index += cols + 2
        value = torch.lerp(low, torch.lerp(flat[index], flat[index + 1], wj), row)
        value *= (math.pi / n) * near ** 2
        out += value
    return out


def exact(case, seed):
    path, batch = case["path"], case["batch"]
    samples = sum(_sizes(p)[2] for p in _parts(case))
    many = {"pair": 2, "slices": 2 * batch, "autograd": 2 * batch, "gradient64": 2, "normal": 2 * batch,
            "sirt": 2 * (case["iterations"] + 1), "requests": 2, "fdk": 0}[path]
    if samples * many > EXACT_SAMPLES:
        return None
    if path == "pair":
        x, y = _one(case, seed)
        return [_forward64(case, x), _backward64(case, y)]
    if path == "sirt":
        return _sirt64(case, _projections(case, seed), case["iterations"])
    if path == "fdk":
        return _fdk64(case, _projections(case, seed))
    if path == "normal":
        ys = [_forward64(case, _volume(case, 1000 * seed + k), k) for k in range(batch)]
        return [ys, [_backward64(case, y, k) for k, y in enumerate(ys)]]
    if path == "requests":
        parts = _parts(case)
        data = [_one(p, 1000 * seed + k) for k, p in enumerate(parts)]
        return [[_forward64(p, d[0]) for p, d in zip(parts, data)],
                [_backward64(p, d[1]) for p, d in zip(parts, data)]]
    if path == "gradient64":
        x, y = _volume(case, 2 * seed, torch.float64), _projections(case, 2 * seed + 1, dtype=torch.float64)
        projected = _forward64(case, x)
        return [projected, _backward64(case, 2 * (projected - y))]
    data = [_one(case, 1000 * seed + k) for k in range(batch)]
    projected = [_forward64(case, x) for x, _ in data]
    gradient = [_backward64(case, 2 * (p - y)) for p, (_, y) in zip(projected, data)]
    projected, gradient = torch.stack(projected), torch.stack(gradient)
    if path == "slices":
        projected = projected.transpose(1, 2).reshape(batch, 1, case["angles"], case["cols"])
    return [projected, gradient]
