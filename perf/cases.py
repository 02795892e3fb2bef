"""Measured work of the sparse-voxel library: the calls a decoder's program makes, through the
package's entry points, over the sizes it meets.

The voxel sets are thickness-2 surface bands of rotated ellipsoid and box shells, sorted with x
slowest: what the decoders and the benchmark of this repository run on. A case names its exact
voxel count: the shells are scaled to give somewhat more and the set is cut off by an x plane.
Weights are random with variance 1 / fan-in, features standard normal.

Kinds of cases, each one or two public calls:

  table     rulebook_build_planned: the neighbour table and the conv plan of a new voxel set, made
            once per level and decode. It returns the table; the plan is an opaque handle whose
            worth the convs below show (theirs come from the same call).
  level     the step from one level to the next: subdivide, then the table and plan of the children
  conv      subm_conv3x3_planned on a plan and packed weights that the program keeps
  conv_f32  subm_conv3x3 in fp32: the cast-to-f32 mode
  thin      subm_conv3x3 with a few channels (f16 or bf16): the memory-bound layers
  convnext  the ConvNeXt block on its plan, weights packed once
  c2s       the features of the 2x subdivision block, on plans of both levels
  head      the decoders' output: layer_norm without affine, then the output linear
"""
from __future__ import annotations

import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
SIZE = {"f32": 4, "f16": 2, "bf16": 2}
# active taps per voxel of a thickness-2 band, and children per parent when it is subdivided to the
# next level's band (both vary by a few per cent with the shapes)
TAPS = 18.5
CHILDREN = 4.1


def _package():
    """The package directory's name holds a dot, so it is loaded by path."""
    if "trellis_cpp_amd" not in sys.modules:
        pkg_dir = os.path.join(ROOT, "trellis.cpp_amd")
        spec = importlib.util.spec_from_file_location("trellis_cpp_amd", os.path.join(pkg_dir, "__init__.py"),
                                                      submodule_search_locations=[pkg_dir])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["trellis_cpp_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["trellis_cpp_amd"]


# ---- cases ------------------------------------------------------------------------------------
def listed():
    return [
        # a 64^3 latent's level: some ten thousand voxels, made anew for every object (launches count)
        {"name": "table_15k", "kind": "table", "n": 14_487, "grid": 64},
        # from a 256^3 level to its ~1.2M children at 512^3
        {"name": "level_290k", "kind": "level", "n": 290_011, "grid": 256},
        # the smallest calls: a 32^3 latent of a small object in a narrow layer
        {"name": "conv_2k_c64", "kind": "conv", "n": 2_606, "grid": 32, "ci": 64, "co": 64, "dtype": "f16"},
        # the benchmark's 128^3 set at 256 channels
        {"name": "conv_117k_c256", "kind": "conv", "n": 117_343, "grid": 128, "ci": 256, "co": 256, "dtype": "bf16"},
        # the 256^3 target: ~600K voxels at 128 channels
        {"name": "conv_643k_c128", "kind": "conv", "n": 643_361, "grid": 256, "ci": 128, "co": 128, "dtype": "bf16"},
        # the precision check's fp32 mode on the 64^3 shell
        {"name": "conv_f32_15k_c64", "kind": "conv_f32", "n": 14_487, "grid": 64, "ci": 64, "co": 64},
        # a thin layer over the 256^3 set
        {"name": "thin_1m7_c8", "kind": "thin", "n": 1_694_162, "grid": 256, "ci": 8, "co": 8, "dtype": "bf16"},
        # the decoders' widest ConvNeXt block on a 32^3 latent (the 512^3 pipeline's first level)
        {"name": "convnext_4k_c1024", "kind": "convnext", "n": 4_099, "grid": 32, "c": 1024, "dtype": "f16"},
        # the second level's block: most of the decoders' blocks (16 of 32) run at this width
        {"name": "convnext_35k_c512", "kind": "convnext", "n": 35_001, "grid": 64, "c": 512, "dtype": "bf16"},
        # the last stage's block at 512^3
        {"name": "convnext_600k_c128", "kind": "convnext", "n": 599_577, "grid": 512, "c": 128, "dtype": "bf16"},
        # the third stage's up-block, 256 -> 128 channels
        {"name": "c2s_60k_c256", "kind": "c2s", "n": 60_013, "grid": 128, "cin": 256, "cout": 128, "dtype": "bf16"},
        # the shape decoder's output layer over a 512^3 level: 7 channels a voxel
        {"name": "head_1m2_c64", "kind": "head", "n": 1_200_007, "ci": 64, "co": 7, "dtype": "f16"},
    ]


def _child_count(n):
    return int(CHILDREN * n)


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid_for(n):
    """The grid (a power of two) whose shells have about n voxels."""
    return 32 if n < 6_000 else 64 if n < 40_000 else 128 if n < 180_000 else 256 if n < 700_000 else 512


def draw(rng):
    kind = rng.choice(["table", "level", "conv", "conv", "conv_f32", "thin", "convnext", "c2s", "head"])
    dtype = rng.choice(["f16", "bf16"])
    # N C^2 up to about the 256^3 target's (a level's voxel count times its channels squared stays
    # about the same down a decoder)
    if kind == "table":
        n = _log_int(rng, 1_000, 1_600_000)
        return {"kind": kind, "n": n, "grid": _grid_for(n)}
    if kind == "level":
        n = _log_int(rng, 1_000, 400_000)
        return {"kind": kind, "n": n, "grid": _grid_for(n)}
    if kind == "conv":
        c = rng.choice([64, 128, 256, 512, 1024])
        n = _log_int(rng, 500, min(1_500_000, 10_000_000_000 // (c * c)))
        return {"kind": kind, "n": n, "grid": _grid_for(n), "ci": c, "co": rng.choice([c, max(64, c // 2)]), "dtype": dtype}
    if kind == "conv_f32":
        c = rng.choice([32, 64, 128])
        n = _log_int(rng, 500, 200_000_000 // (c * c))
        return {"kind": kind, "n": n, "grid": _grid_for(n), "ci": c, "co": c}
    if kind == "thin":
        n = _log_int(rng, 20_000, 1_700_000)
        return {"kind": kind, "n": n, "grid": _grid_for(n), "ci": rng.choice([8, 16, 32]), "co": rng.choice([8, 16]),
                "dtype": dtype}
    if kind == "convnext":
        # at the width whose MLP is this library's kernel (wider ones are the library GEMM's)
        n = _log_int(rng, 1_000, 550_000)
        return {"kind": kind, "n": n, "grid": _grid_for(n), "c": 128, "dtype": dtype}
    if kind == "c2s":
        cin = rng.choice([128, 256])
        n = _log_int(rng, 1_000, 4_000_000_000 // (cin * cin))
        return {"kind": kind, "n": n, "grid": _grid_for(n), "cin": cin, "cout": cin // 2, "dtype": dtype}
    return {"kind": kind, "n": _log_int(rng, 10_000, 2_000_000), "ci": 64, "co": rng.choice([6, 7]), "dtype": dtype}


# ---- voxel sets -------------------------------------------------------------------------------
class _Shells:
    """Rotated ellipsoid and box shells drawn in a grid; distance estimates on the GPU."""

    def __init__(self, rng, grid, n, count):
        self.parts = []
        shape = rng.uniform(0.6, 1.0, (count, 3))
        # the shells' areas (an ellipsoid's by its mean radius, a box's exactly) times the thickness
        area = 0.0
        for k in range(count):
            a, b, c = shape[k]
            area += 8 * (a * b + b * c + a * c) if k % 2 else 4 * math.pi * ((a * b) ** 1.6 / 3 + (a * c) ** 1.6 / 3 + (b * c) ** 1.6 / 3) ** (1 / 1.6)
        scale = math.sqrt(1.15 * n / (2.0 * area))
        for k in range(count):
            semi = shape[k] * scale
            m = semi.max() + 2
            lo, hi = min(m, grid / 2), max(grid - m, grid / 2)
            q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
            self.parts.append((k % 2 == 1, rng.uniform(lo, hi, 3), semi, q))

    def scaled(self, f):
        other = object.__new__(_Shells)
        other.parts = [(box, center * f, semi * f, rot) for box, center, semi, rot in self.parts]
        return other

    def grown(self, f):
        other = object.__new__(_Shells)
        other.parts = [(box, center, semi * f, rot) for box, center, semi, rot in self.parts]
        return other

    def distance(self, p):
        """|distance| of points p [K, 3] to the nearest surface."""
        best = None
        for box, center, semi, rot in self.parts:
            c = torch.tensor(center, dtype=torch.float32, device=p.device)
            r = torch.tensor(rot, dtype=torch.float32, device=p.device)
            s = torch.tensor(semi, dtype=torch.float32, device=p.device)
            q = p - c
            q = torch.stack([(q * r[:, j]).sum(1) for j in range(3)], 1)
            if box:
                e = q.abs() - s
                d = e.clamp_min(0).square().sum(1).sqrt() + e.max(1).values.clamp_max(0)
            else:
                u = q / s
                f = u.square().sum(1).sqrt().clamp_min(1e-6)
                d = (f - 1) * f / (u / s).square().sum(1).sqrt().clamp_min(1e-12)
            d = d.abs()
            best = d if best is None else torch.minimum(best, d)
        return best

    def band(self, grid):
        """int32 [N, 3], sorted: the voxels whose centre is within 1 of a surface."""
        ax = torch.arange(grid, device="cuda", dtype=torch.int32)
        if grid > 64:   # cells of 8 voxels that a surface can cross, then their voxels
            cells = grid // 8
            ca = torch.arange(cells, device="cuda", dtype=torch.int32)
            cc = torch.cartesian_prod(ca, ca, ca)
            # the ellipsoid distance is a first-order estimate: a generous margin around the cell
            near = cc[self.distance((cc * 8 + 4).float()) < 14.0]
            off = torch.cartesian_prod(ax[:8], ax[:8], ax[:8])
            v = (near[:, None, :] * 8 + off[None, :, :]).reshape(-1, 3)
        else:
            v = torch.cartesian_prod(ax, ax, ax)
        v = v[self.distance(v.float() + 0.5) < 1.0]
        key = (v[:, 0].long() * grid + v[:, 1]) * grid + v[:, 2]
        return v[key.argsort()].contiguous()

    def mask(self, coords, m):
        """uint8 [N, 8]: the m children of coords nearest to a surface of the next level (whose shells
        these are, at twice the resolution): a band of about thickness 2 with an exact count."""
        d = []
        for o in range(8):
            off = torch.tensor([o & 1, (o >> 1) & 1, (o >> 2) & 1], device=coords.device, dtype=torch.int32)
            d.append(self.distance((coords * 2 + off).float() + 0.5))
        mask = torch.zeros(len(coords) * 8, dtype=torch.uint8, device=coords.device)
        mask[torch.stack(d, 1).reshape(-1).sort(stable=True).indices[:m]] = 1
        return mask.reshape(-1, 8)



def _voxels(n, grid, seed):
    """(int32 [n, 3] coordinates on the GPU, the shells they come from)"""
    rng = np.random.default_rng(seed)
    sh = _Shells(rng, grid, n, 3 if grid <= 64 else 6)
    for _ in range(40):
        v = sh.band(grid)
        if len(v) >= n:
            return v[:n].contiguous(), sh
        sh = sh.grown(1.08)
    raise ValueError(f"a {grid}^3 grid holds no such set of {n} voxels")


# ---- inputs -----------------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 7919 + 17)
    return g


def _normal(g, shape, std=1.0, dtype=torch.float32, mean=0.0):
    return (torch.randn(shape, generator=g, device="cuda") * std + mean).to(dtype)


def _convnext_weights(g, c, dt):
    return {"conv.weight": _normal(g, (c, 27, c), 1 / math.sqrt(TAPS * c), dt), "conv.bias": _normal(g, (c,), 0.1),
            "norm.weight": _normal(g, (c,), 0.1, mean=1.0), "norm.bias": _normal(g, (c,), 0.1),
            "mlp.0.weight": _normal(g, (4 * c, c), 1 / math.sqrt(c), dt), "mlp.0.bias": _normal(g, (4 * c,), 0.1),
            "mlp.2.weight": _normal(g, (c, 4 * c), 1 / math.sqrt(4 * c), dt), "mlp.2.bias": _normal(g, (c,), 0.1)}


def _c2s_weights(g, cin, cout, dt):
    return {"norm1.weight": _normal(g, (cin,), 0.1, mean=1.0), "norm1.bias": _normal(g, (cin,), 0.1),
            "conv1.weight": _normal(g, (8 * cout, 27, cin), 1 / math.sqrt(TAPS * cin), dt),
            "conv1.bias": _normal(g, (8 * cout,), 0.1),
            "conv2.weight": _normal(g, (cout, 27, cout), 1 / math.sqrt(TAPS * cout), dt),
            "conv2.bias": _normal(g, (cout,), 0.1)}


def _inputs(case, seed):
    """The case's inputs from the seed alone, before anything of the library is used."""
    kind, g, n = case["kind"], _gen(seed), case["n"]
    if kind == "head":
        dt = DTYPES[case["dtype"]]
        return {"case": case, "x": _normal(g, (n, case["ci"])), "b": _normal(g, (case["co"],), 0.1),
                "w": _normal(g, (case["co"], case["ci"]), 1 / math.sqrt(case["ci"]), dt)}
    coords, sh = _voxels(n, case["grid"], seed)
    s = {"case": case, "coords": coords}
    if kind in ("conv", "thin", "conv_f32"):
        dt, ci, co = DTYPES[case.get("dtype", "f32")], case["ci"], case["co"]
        s["x"] = _normal(g, (n, ci), 1.0, dt)
        s["w"] = _normal(g, (co, 27, ci), 1 / math.sqrt(TAPS * ci), dt)
        s["b"] = _normal(g, (co,), 0.1)
    elif kind == "convnext":
        s["x"] = _normal(g, (n, case["c"]))
        s["p"] = _convnext_weights(g, case["c"], DTYPES[case["dtype"]])
    elif kind == "c2s":
        s["x"] = _normal(g, (n, case["cin"]))
        s["p"] = _c2s_weights(g, case["cin"], case["cout"], DTYPES[case["dtype"]])
        s["mask"] = sh.scaled(2.0).mask(coords, _child_count(n))
    elif kind == "level":
        s["mask"] = sh.scaled(2.0).mask(coords, _child_count(n))
    return s


def _children(mask, coords):
    parent, octant = mask.nonzero(as_tuple=True)
    off = torch.stack([octant & 1, (octant >> 1) & 1, (octant >> 2) & 1], 1).to(torch.int32)
    return (2 * coords[parent] + off).contiguous()


def prepare(case, seed):
    tsp = _package()
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("table", "level", "head"):
        return s
    s["nbr"], s["plan"] = tsp.rulebook_build_planned(s["coords"])
    if kind == "conv":
        s["packed"] = tsp.conv_weight_pack(s["w"])
    elif kind == "convnext":
        s["p"]["conv.packed"] = tsp.conv_weight_pack(s["p"]["conv.weight"])
        if case["c"] == 128:
            s["p"]["mlp.packed"] = tsp.convnext_mlp_pack(s["p"]["mlp.0.weight"], s["p"]["mlp.2.weight"])
    elif kind == "c2s":
        s["p"]["conv1.packed"] = tsp.conv_weight_pack(s["p"]["conv1.weight"])
        s["p"]["conv2.packed"] = tsp.conv_weight_pack(s["p"]["conv2.weight"])
        s["child"], s["gidx"], s["mstart"] = tsp.subdivide(s["mask"], s["coords"])
        s["child_nbr"], s["child_plan"] = tsp.rulebook_build_planned(s["child"])
    return s


def run(state):
    tsp, s = _package(), state
    case = s["case"]
    kind = case["kind"]
    if kind == "table":
        nbr, s["plan"] = tsp.rulebook_build_planned(s["coords"], check=False)
        return nbr
    if kind == "level":
        child, gidx, mstart = tsp.subdivide(s["mask"], s["coords"])
        nbr, s["plan"] = tsp.rulebook_build_planned(child, check=False)
        return {"coords": child, "gidx": gidx, "mstart": mstart, "nbr": nbr}
    if kind == "conv":
        return tsp.subm_conv3x3_planned(s["x"], s["nbr"], s["plan"], s["packed"], s["b"], case["co"])
    if kind in ("conv_f32", "thin"):
        return tsp.subm_conv3x3(s["x"], s["nbr"], s["w"], s["b"])
    if kind == "convnext":
        return tsp.convnext(s["x"], s["nbr"], s["p"], plan=s["plan"])
    if kind == "head":
        h = tsp.layer_norm(s["x"], eps=1e-5, out_dtype=s["w"].dtype)
        return tsp.linear(h, s["w"], s["b"], out_dtype=torch.float32)
    return tsp.c2s(s["x"], s["nbr"], s["mask"], s["mstart"], s["gidx"], len(s["gidx"]), case["cout"], s["child_nbr"],
                   s["p"], plan=s["plan"], child_plan=s["child_plan"])

# ---- what a pass cannot do without ------------------------------------------------------------
def _level(n):
    """The table of n voxels and the plan that goes with it, as inputs: 27 words a voxel."""
    return 108.0 * n


def _convnext_work(n, c, es):
    return (n * c * 4 * 2 + _level(n) + (27 * c * c + 8 * c * c) * es, 2.0 * TAPS * n * c * c + 16.0 * n * c * c)


def _c2s_work(n, m, cin, cout, es):
    """conv1's outputs are the kept children's alone."""
    return (n * cin * 4 + m * cout * 4 + _level(n) + _level(m) + 8 * n + 8 * m + (27 * 8 * cout * cin + 27 * cout * cout) * es,
            2.0 * TAPS * m * cin * cout + 2.0 * TAPS * m * cout * cout)


def work(case):
    kind, n = case["kind"], case["n"]
    if kind == "table":
        return {"bytes": 12.0 * n + _level(n), "flops": 0.0}
    if kind == "level":
        m = _child_count(n)
        return {"bytes": 12.0 * n + 8 * n + 4 * n + (12 + 4) * m + _level(m), "flops": 0.0}
    es = SIZE[case.get("dtype", "f32")]
    if kind == "head":
        return {"bytes": n * (case["ci"] + case["co"]) * 4.0, "flops": 2.0 * n * case["ci"] * case["co"]}
    if kind in ("conv", "conv_f32", "thin"):
        ci, co = case["ci"], case["co"]
        return {"bytes": n * (ci + co) * es + _level(n) + 27.0 * ci * co * es, "flops": 2.0 * TAPS * n * ci * co}
    if kind == "convnext":
        b, f = _convnext_work(n, case["c"], es)
        return {"bytes": b, "flops": f}
    b, f = _c2s_work(n, _child_count(n), case["cin"], case["cout"], es)
    return {"bytes": b, "flops": f}


def tolerance(case):
    kind = case["kind"]
    if kind in ("table", "level"):
        return "exact"
    if kind == "conv_f32":
        return {"rel": 2e-6}
    if kind in ("conv", "thin"):
        # one rounding of the result to 16 bits
        return {"rel": 8e-3 if case["dtype"] == "bf16" else 1e-3}
    # a block (or the norm before the output layer): its products' inputs are rounded to 16 bits inside
    return {"rel": 6e-3 if case["dtype"] == "bf16" else 1e-3}


# ---- the same in 64 bits ----------------------------------------------------------------------
def _table64(coords):
    """int64 [27, N] neighbour rows, N where there is none (coordinates distinct)."""
    n, g = len(coords), int(coords.max()) + 3
    grid = torch.full((g * g * g,), n, dtype=torch.int32, device=coords.device)
    c = coords.long() + 1
    key = (c[:, 0] * g + c[:, 1]) * g + c[:, 2]
    grid[key] = torch.arange(n, dtype=torch.int32, device=coords.device)
    return torch.stack([grid[key + (kd * g + kh) * g + kw] for kd in (-1, 0, 1) for kh in (-1, 0, 1) for kw in (-1, 0, 1)])


def _conv64(x, table, w, b):
    """x [N, Ci] f64; rows in pieces so that the gathered copies stay small."""
    n, co = x.shape[0], w.shape[0]
    out = b.double().repeat(n, 1)
    wt = [w[:, t].double().t().contiguous() for t in range(27)]
    for r0 in range(0, n, 1 << 18):
        for t in range(27):
            row = table[t, r0:r0 + (1 << 18)].long()
            at = (row < n).nonzero().squeeze(1)
            out[r0 + at] += x[row[at]] @ wt[t]
    return out


def _norm64(x, eps, w=None, b=None):
    x = x - x.mean(1, keepdim=True)
    x = x / (x.square().mean(1, keepdim=True) + eps).sqrt()
    return x if w is None else x * w.double() + b.double()


def _silu64(x):
    return x / (1 + torch.exp(-x))


def _convnext64(x, table, p):
    h = _norm64(_conv64(x, table, p["conv.weight"], p["conv.bias"]), 1e-6, p["norm.weight"], p["norm.bias"])
    h = _silu64(h @ p["mlp.0.weight"].double().t() + p["mlp.0.bias"].double())
    return h @ p["mlp.2.weight"].double().t() + p["mlp.2.bias"].double() + x


def _c2s64(x, table, mask, child_table, p):
    n, cin = x.shape
    cout = p["conv2.bias"].numel()
    parent, octant = mask.nonzero(as_tuple=True)
    h = _silu64(_norm64(x, 1e-6, p["norm1.weight"], p["norm1.bias"]))
    h = _conv64(h, table, p["conv1.weight"], p["conv1.bias"]).reshape(n, 8, cout)[parent, octant]
    h = _conv64(_silu64(_norm64(h, 1e-6)), child_table, p["conv2.weight"], p["conv2.bias"])
    return h + x.reshape(n, 8, cin // 8)[parent, octant].repeat_interleave(cout // (cin // 8), 1)


def exact(case, seed):
    kind = case["kind"]
    s = _inputs(case, seed)
    if kind in ("table", "level"):
        return None
    if kind == "head":
        return _norm64(s["x"].double(), 1e-5) @ s["w"].double().t() + s["b"].double()
    table = _table64(s["coords"])
    if kind in ("conv", "conv_f32", "thin"):
        return _conv64(s["x"].double(), table, s["w"], s["b"])
    if kind == "convnext":
        return _convnext64(s["x"].double(), table, s["p"])
    return _c2s64(s["x"].double(), table, s["mask"], _table64(_children(s["mask"], s["coords"])), s["p"])
