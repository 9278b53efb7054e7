"""What the speed of this library is measured on.

Each case is one thing that a program using lj_gpu_amd has it do, through the
Python mirror of the C ABI (Context and DeviceArray), with positions, momenta
and neighbour lists resident on the GPU as such a program keeps them. The sizes
are those of the benchmark, the tests and the reference's own problem, and
odd, ragged ones between them (lattices with vacancies, particles in a shuffled
order).

Five uses:

force     p += F(q) dt repeated over an installed list (the reference's
          measure() loop): list kinds, layouts, precisions, open and periodic
          boxes, one step as an integrator of its own calls it or many
kernel    one launch over the caller's own, unvalidated CSR arrays with the
          reference kernels' argument list
refresh   what an integrator does when its list has gone stale: build the list
          from the positions on the device, then evaluate the force once
replicas  independent boxes of uneven size in one launch
md        the velocity-Verlet driver with its list rebuilds and energy samples
"""
import ctypes
import math

import numpy as np
import torch

import lj_gpu_amd as lj

CUTOFF = 3.0
SEARCH = 3.3
CL2 = CUTOFF * CUTOFF


def listed():
    return [
        # The smallest periodic system of the tests: one evaluation per call, so
        # launch and latency are everything (unit-cell studies, unit tests).
        _force("force_smallest", cells=6, density=1.0, steps=1),
        # The reference's own benchmark: open box, density 0.5, 100 calls.
        _force("force_reference_open", cells=25, density=0.5, box="open", steps=100, dt=0.001,
               jitter="reference"),
        # The headline benchmark: 119,164 particles at density 1, full list.
        _force("force_headline", cells=31, density=1.0, steps=100),
        # The mixed-precision kernels, on SoA arrays.
        _force("force_mixed_soa", cells=31, density=1.0, steps=100, layout="soa", prec="mixed"),
        # The largest single system of the benchmark, 1,048,576 particles.
        _force("force_large", cells=64, density=1.0, steps=10),
        # A half list evaluated by scattering to both particles (the
        # reference's action-reaction kernels), a fluid with vacancies.
        _force("force_half_atomic", cells=25, density=0.8, vacancies=37, steps=4,
               list="half_atomic"),
        # The drop-in launch: the reference kernels' argument list over the
        # caller's CSR arrays, on the reference's problem.
        {"name": "kernel_csr_open", "use": "kernel", "cells": 25, "density": 0.5, "vacancies": 0,
         "shuffled": False, "list": "full", "dt": 0.001, "jitter": "reference"},
        # An integrator's list refresh at the headline size; its particles have
        # long left the lattice order, and there is no round number of them.
        {"name": "refresh_headline", "use": "refresh", "cells": 31, "density": 1.0,
         "vacancies": 101, "shuffled": True, "dt": 0.01, "jitter": "periodic"},
        # The same for a small system, where its many short steps count.
        {"name": "refresh_small", "use": "refresh", "cells": 8, "density": 0.8, "vacancies": 5,
         "shuffled": True, "dt": 0.01, "jitter": "periodic"},
        # The batched replica workload of the benchmark.
        {"name": "replicas_256", "use": "replicas", "replicas": 256, "cells_lo": 6,
         "cells_hi": 20, "steps": 10, "dt": 0.01},
        # Molecular dynamics of a small fluid: thousands of short launches.
        _md("md_small", cells=10, density=0.8, steps=100, rebuild_every=20, skin=0.3),
        # Molecular dynamics where the kicks and the list rebuilds are the work.
        _md("md_large", cells=64, density=0.8, steps=40, rebuild_every=20, skin=0.3),
    ]


def _force(name, **kw):
    c = {"use": "force", "vacancies": 0, "shuffled": False, "box": "periodic", "list": "full",
         "layout": "aos", "prec": "f64", "dt": 0.01, "jitter": "periodic"}
    c.update(kw)
    if name:
        c["name"] = name
    return c


def _md(name, **kw):
    c = {"use": "md", "vacancies": 0, "shuffled": False, "temperature": 1.0, "dt": 0.005,
         "sample_every": 20, "jitter": "periodic"}
    c.update(kw)
    if name:
        c["name"] = name
    return c


def _cells(rng, lo, hi):
    """FCC cells per side, spread evenly over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _holes(rng, cells):
    """Vacancies: none, or a ragged number up to a fiftieth of the particles."""
    return rng.choice([0, rng.randint(1, max(1, 4 * cells ** 3 // 50))])


def draw(rng):
    use = rng.choice(["force", "force", "force", "kernel", "refresh", "replicas", "md"])
    density = round(rng.uniform(0.5, 1.0), 3)
    shuffled = rng.random() < 0.5
    if use == "force":
        kind = rng.choice(["full", "full", "full", "half_expand", "half_atomic"])
        cells = _cells(rng, 6, 25 if kind == "half_atomic" else 60)
        entries = 4 * cells ** 3 * 4.18879 * SEARCH ** 3 * density
        steps = rng.choice([1, 1, 4, 10, 20, 50, 100])
        while steps > 1 and steps * entries > 1.4e9:  # no more than the largest listed one
            steps = max(1, steps // 4)
        box = rng.choice(["periodic", "periodic", "open"])
        return _force("", cells=cells, density=density, vacancies=_holes(rng, cells),
                      shuffled=shuffled, box=box, list=kind,
                      layout=rng.choice(["aos", "aos", "soa", "aos3"]),
                      prec=rng.choice(["f64", "f64", "mixed", "kahan"]), steps=steps,
                      dt=round(rng.uniform(0.001, 0.01), 4))
    if use == "kernel":
        cells = _cells(rng, 6, 40)
        return {"use": use, "cells": cells, "density": density, "vacancies": _holes(rng, cells),
                "shuffled": shuffled, "list": rng.choice(["full", "full", "half_atomic"]),
                "dt": round(rng.uniform(0.001, 0.01), 4), "jitter": "reference"}
    if use == "refresh":
        cells = _cells(rng, 6, 50)
        return {"use": use, "cells": cells, "density": density, "vacancies": _holes(rng, cells),
                "shuffled": shuffled, "dt": round(rng.uniform(0.001, 0.01), 4),
                "jitter": "periodic"}
    if use == "replicas":
        lo = rng.randint(5, 9)
        return {"use": use, "replicas": int(round(math.exp(rng.uniform(math.log(3),
                                                                      math.log(200))))),
                "cells_lo": lo, "cells_hi": rng.randint(lo, 16),
                "steps": rng.choice([1, 10, 20]), "dt": round(rng.uniform(0.001, 0.01), 4)}
    cells = _cells(rng, 6, 50)
    return _md("", cells=cells, density=round(rng.uniform(0.6, 0.9), 3),
               vacancies=_holes(rng, cells), shuffled=shuffled,
               steps=rng.choice([10, 23, 40, 60]), rebuild_every=rng.choice([5, 10, 20]),
               skin=rng.choice([0.3, 0.5]), sample_every=rng.choice([0, 10, 20]))


# ---------------------------------------------------------------------------
# Inputs, in plain numpy
# ---------------------------------------------------------------------------
def _fcc(cells, density, rng, jitter):
    """FCC lattice of 4 cells^3 particles with a uniform jitter: (N, 4), side."""
    a = (4.0 / density) ** (1.0 / 3.0)
    ix = np.arange(cells)
    z, y, x = np.meshgrid(ix, ix, ix, indexing="ij")
    base = np.stack([x, y, z], -1).reshape(-1, 1, 3).astype(np.float64)
    corner = np.array([[0, 0, 0], [.5, 0, 0], [0, .5, 0], [0, 0, .5]])
    corner[1:] = 0.5 - corner[1:]  # the three face centres
    r = ((base + corner) * a).reshape(-1, 3)
    lo, hi = (0.0, 0.1) if jitter == "reference" else (-0.05, 0.05)
    r += rng.uniform(lo, hi, size=r.shape)
    return r, cells * a


def _system(case, seed):
    """Positions (N, 4) with a zero fourth column, and the box (0: open)."""
    rng = np.random.default_rng(seed)
    r, side = _fcc(case["cells"], case["density"], rng, case["jitter"])
    if case["vacancies"]:
        keep = np.ones(len(r), bool)
        keep[rng.choice(len(r), case["vacancies"], replace=False)] = False
        r = r[keep]
    if case["shuffled"]:
        r = r[rng.permutation(len(r))]
    box = 0.0
    if case["use"] in ("refresh", "md") or (case["use"] == "force" and case["box"] == "periodic"):
        box = side
        r -= box * np.floor(r / box)
        r[r >= box] = 0.0
    q = np.zeros((len(r), 4))
    q[:, :3] = r
    return q, box


def _momenta(n, temperature, seed):
    rng = np.random.default_rng(seed + 77)
    p = np.zeros((n, 4))
    p[:, :3] = rng.normal(0.0, math.sqrt(temperature), size=(n, 3))
    p[:, :3] -= p[:, :3].mean(0)
    return p


def _replica_systems(case, seed):
    """The boxes of a batch: cells per side and densities drawn per replica
    (the batch's shape belongs to the case, so from a generator of its own)."""
    shape = np.random.default_rng(4)
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(case["replicas"]):
        k = int(shape.integers(case["cells_lo"], case["cells_hi"] + 1))
        r, side = _fcc(k, float(shape.uniform(0.5, 1.0)), rng, "periodic")
        r -= side * np.floor(r / side)
        r[r >= side] = 0.0
        out.append((r, side))
    return out


# ---------------------------------------------------------------------------
# Measured passes
# ---------------------------------------------------------------------------
class _View:
    """A DeviceArray as torch sees it."""

    def __init__(self, a):
        self.a = a
        self.__cuda_array_interface__ = {"shape": a.shape, "typestr": "<f8", "strides": None,
                                         "data": (a.ptr, False), "version": 2}


def _tensor(a):
    return torch.as_tensor(_View(a), device="cuda")


def _columns(ctx, q, layout):
    """Positions and momenta in a layout: device arrays and p's tensors."""
    n = q.shape[0]
    if layout == "soa":
        qd = [ctx.array(np.ascontiguousarray(q[:, c])) for c in range(3)]
        pd = [ctx.zeros((n,)) for _ in range(3)]
        return qd, pd, [_tensor(a) for a in pd]
    w = 3 if layout == "aos3" else 4
    qd, pd = ctx.array(np.ascontiguousarray(q[:, :w])), ctx.zeros((n, w))
    return qd, pd, [_tensor(pd)]


def prepare(case, seed):
    ctx = lj.Context(0)
    s = {"case": case, "ctx": ctx}
    if case["use"] == "replicas":
        systems = _replica_systems(case, seed)
        n = sum(len(r) for r, _ in systems)
        q = np.zeros((n, 4))
        q[:, :3] = np.concatenate([r for r, _ in systems])
        offsets = np.cumsum([0] + [len(r) for r, _ in systems]).astype(np.int32)
        s["q"], s["p"], s["out"] = _columns(ctx, q, "aos")
        ctx.set_replicas(offsets, np.array([b for _, b in systems]))
        ctx.build_list(s["q"], n, 0.0, lj.LIST_FULL, SEARCH)
        return s
    q, s["box"] = _system(case, seed)
    n = s["n"] = q.shape[0]
    if case["use"] == "md":
        s["q0"], s["p0"] = ctx.array(q), ctx.array(_momenta(n, case["temperature"], seed))
        s["q"], s["p"] = ctx.empty((n, 4)), ctx.empty((n, 4))
        s["out"] = [_tensor(s["q"]), _tensor(s["p"])]
        return s
    s["q"], s["p"], s["out"] = _columns(ctx, q, case.get("layout", "aos"))
    if case["use"] == "kernel":
        half = case["list"] == "half_atomic"
        ctx.set_half_mode(lj.HALF_ATOMIC)
        ctx.set_tiling(0)
        ctx.build_list(s["q"], n, 0.0, lj.LIST_HALF if half else lj.LIST_FULL, SEARCH)
        csr = ctx.get_list()
        s["kind"], s["entries"] = csr.kind, csr.n_entries
        s["csr"] = [ctx.array(a) for a in (csr.sorted_list, csr.number_of_partners, csr.pointer)]
    elif case["use"] == "force":
        half = case["list"] != "full"
        ctx.set_half_mode(lj.HALF_ATOMIC if case["list"] == "half_atomic" else lj.HALF_EXPAND)
        build = {"aos": ctx.build_list, "soa": ctx.build_list_soa,
                 "aos3": ctx.build_list_aos3}[case["layout"]]
        build(s["q"], n, s["box"], lj.LIST_HALF if half else lj.LIST_FULL, SEARCH)
    return s


def run(s):
    case, ctx, q, p = s["case"], s["ctx"], s["q"], s["p"]
    use = case["use"]
    if use == "md":
        for dst, src in ((q, s["q0"]), (p, s["p0"])):
            lj._check(lj.lib().ljgpu_memcpy_dtod(ctx.handle, dst.ptr, src.ptr,
                                                 ctypes.c_size_t(src.nbytes)))
        _, samples = ctx.md_run(q, p, s["box"], case["steps"], dt=case["dt"], cutoff=CUTOFF,
                                skin=case["skin"], rebuild_every=case["rebuild_every"],
                                sample_every=case["sample_every"])
        return {"q": s["out"][0], "p": s["out"][1], "samples": samples}
    # Fresh momenta, as the reference's measure() starts from.
    for a in p if isinstance(p, list) else [p]:
        a.zero()
    if use == "refresh":
        ctx.build_list(q, s["n"], s["box"], lj.LIST_FULL, SEARCH)
        ctx.force_aos_f64(q, p, case["dt"], CL2, s["box"], 1)
    elif use == "replicas":
        ctx.force_aos_f64(q, p, case["dt"], CL2, 0.0, case["steps"])
    elif use == "kernel":
        lst, nop, ptr = s["csr"]
        ctx.force_kernel_csr_f64(q, p, s["n"], case["dt"], CL2, lst, nop, ptr, s["entries"],
                                 s["kind"])
    else:
        args = (q, p, case["dt"], CL2, s["box"], case["steps"])
        name = "force_" + case["layout"] + ("_f64" if case["prec"] == "f64" else "_mixed")
        if case["prec"] != "f64":
            args += (lj.ACCUM_KAHAN_F32 if case["prec"] == "kahan" else lj.ACCUM_F64,)
        getattr(ctx, name)(*args)
    return s["out"]


def work(case):
    """Per force evaluation: the list once (4-byte entries), positions once,
    momenta read and written; 22 operations per evaluated entry of the search
    sphere, a half list's each serving two particles. A list build reads the
    positions and writes the list once."""
    def evaluation(n, density, half=False, width=32, open_box_side=0.0):
        partners = 4.0 / 3.0 * math.pi * SEARCH ** 3 * density
        if open_box_side > 0.0:  # particles near the faces have fewer partners
            partners *= max(0.3, 1.0 - 3.0 * 3.0 / 8.0 * SEARCH / open_box_side)
        e = n * partners * (0.5 if half else 1.0)
        return 4.0 * e + n * (8.0 + 3.0 * width), 22.0 * e + 6.0 * n, 4.0 * e + 40.0 * n

    if case["use"] == "replicas":
        shape = np.random.default_rng(4)
        b = f = 0.0
        for _ in range(case["replicas"]):
            k = int(shape.integers(case["cells_lo"], case["cells_hi"] + 1))
            eb, ef, _ = evaluation(4 * k ** 3, float(shape.uniform(0.5, 1.0)))
            b, f = b + eb, f + ef
        return {"bytes": b * case["steps"], "flops": f * case["steps"]}
    n = 4 * case["cells"] ** 3 - case["vacancies"]
    side = case["cells"] * (4.0 / case["density"]) ** (1.0 / 3.0)
    density = case["density"] * n / (4 * case["cells"] ** 3)
    is_open = case["use"] == "kernel" or case.get("box") == "open"
    width = {"soa": 24, "aos3": 24}.get(case.get("layout"), 32)
    b, f, lb = evaluation(n, density, case.get("list", "full") == "half_atomic", width,
                          side if is_open else 0.0)
    if case["use"] == "refresh":
        return {"bytes": b + lb, "flops": f}
    if case["use"] == "md":
        rebuilds = 1 + case["steps"] // case["rebuild_every"]
        steps = case["steps"]
        return {"bytes": steps * (b + 96.0 * n) + rebuilds * lb, "flops": steps * (f + 12.0 * n)}
    steps = case.get("steps", 1)
    return {"bytes": steps * b, "flops": steps * f}


# ---------------------------------------------------------------------------
# The same results from plain torch in 64 bits
# ---------------------------------------------------------------------------
def _plain_force(r, box, energy=False):
    """F (N, 3) of every pair inside the cutoff, and the shifted potential
    energy. Particles sorted along x; a block of them meets those within the
    cutoff along x, in their periodic images."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    r = torch.as_tensor(np.ascontiguousarray(r), device=dev, dtype=torch.float64)
    n = r.shape[0]
    order = torch.argsort(r[:, 0])
    s = r[order]
    src = s
    if box > 0.0:
        low, high = s[s[:, 0] <= CUTOFF], s[s[:, 0] >= box - CUTOFF]
        shift = torch.tensor([box, 0.0, 0.0], device=dev, dtype=torch.float64)
        src = torch.cat([high - shift, s, low + shift])
    xs = src[:, 0].contiguous()
    f = torch.zeros_like(s)
    u = 0.0
    s6 = 1.0 / CL2 ** 3
    shift_u = 4.0 * s6 * (s6 - 1.0)
    a = 0
    while a < n:
        b = min(n, a + 1024)
        lo = int(torch.searchsorted(xs, s[a, 0] - CUTOFF - 1e-9))
        hi = int(torch.searchsorted(xs, s[b - 1, 0] + CUTOFF + 1e-9))
        d = [src[lo:hi, c][None, :] - s[a:b, c][:, None] for c in range(3)]
        if box > 0.0:
            for c in (1, 2):
                d[c] -= box * torch.round(d[c] / box)
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
        i, j = torch.nonzero((r2 <= CL2) & (r2 > 0.0), as_tuple=True)
        w = r2[i, j]
        i6 = 1.0 / (w * w * w)
        g = (24.0 * i6 - 48.0 * i6 * i6) / w
        for c in range(3):
            f[a:b, c].index_add_(0, i, g * d[c][i, j])
        if energy:
            u += float((4.0 * i6 * (i6 - 1.0) - shift_u).sum()) / 2.0
        a = b
    out = torch.empty_like(f)
    out[order] = f
    return out.cpu().numpy(), u


def exact(case, seed):
    if case["use"] == "replicas":
        f = np.concatenate([_plain_force(r, box)[0] for r, box in _replica_systems(case, seed)])
        p = np.zeros((len(f), 4))
        p[:, :3] = f * (case["dt"] * case["steps"])
        return [p]
    q, box = _system(case, seed)
    if case["use"] == "md":
        if len(q) * case["steps"] > 2e6:
            return None
        return _plain_md(case, q, _momenta(len(q), case["temperature"], seed), box)
    f, _ = _plain_force(q[:, :3], box)
    f = f * (case["dt"] * case.get("steps", 1))
    layout = case.get("layout", "aos")
    if layout == "soa":
        return [np.ascontiguousarray(f[:, c]) for c in range(3)]
    if layout == "aos3":
        return [f]
    p = np.zeros((len(f), 4))
    p[:, :3] = f
    return [p]


def _plain_md(case, q, p, box):
    """Velocity Verlet over every pair inside the cutoff."""
    q, p, dt = q.copy(), p.copy(), case["dt"]
    every, rows = case["sample_every"], []

    def sample(step, u):
        k = 0.5 * float((p[:, :3] ** 2).sum())
        rows.append([step, u, k, u + k])

    f, u = _plain_force(q[:, :3], box, True)
    sample(0, u)
    for s in range(1, case["steps"] + 1):
        p[:, :3] += f * (0.5 * dt)
        q[:, :3] += p[:, :3] * dt
        q[:, :3] -= box * np.floor(q[:, :3] / box)
        f, u = _plain_force(q[:, :3], box, True)
        p[:, :3] += f * (0.5 * dt)
        if (every and s % every == 0) or s == case["steps"]:
            sample(s, u)
    return {"q": q, "p": p, "samples": np.array(rows)}
