"""The edge cases of the planned conv on both of its kernels (csrc/conv_halo_kernel.hpp for large
grids, csrc/conv_split_kernel.hpp for small ones) and in each kind of stores: a padding row that is
not finite, weights that are not, an exact zero padding row, tiles that read their rows from memory, an
odd number of 16-channel slices. Which kernel a size takes is asked of the library's own rule."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL_16 = 1e-3
TOL_16_OUT = 4e-3
# kind of stores -> channels, 64-channel groups of a small-grid unit, voxels for the small and the large
# grid (on 256 compute units)
KINDS = {"f32": (1024, 1, 3001, 9001), "16-bit": (1024, 1, 5001, 9001), "64": (64, 1, 3001, 66001),
         "octants": (1024, 1, 4001, 9001), "c2s 64": (512, 1, 3001, 17001), "c2s 128": (1024, 2, 5001, 9001),
         "norm 64": (64, 1, 3001, 66001), "norm 128": (128, 2, 40001, 66001), "skip": (512, 1, 4001, 17001)}


def _large(tsp, n, ci, co, ncg):
    rule = tsp.lib()["_ZN3tsp15conv_split_pickEliii"]
    rule.argtypes, rule.restype = [ctypes.c_int64, ctypes.c_int, ctypes.c_int, ctypes.c_int], ctypes.c_int
    return rule(n, ci, co, ncg) == 0


def _case(tsp, kind, kernel, ci):
    import torch
    co, ncg, small, large = KINDS[kind]
    n = large if kernel == "large" else small
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert _large(tsp, n, ci, co, ncg) == (kernel == "large")
    return n, co


def _shell(shells, n):
    """n voxels of a shell four voxels thick (a few have all 27 taps), and its table's device tensors."""
    r = 14.0
    while True:
        g = int(2 * r) + 8
        c = shells.sphere_shell(g, g / 2, r - 2.0, r + 2.0)
        if len(c) >= n:
            return np.ascontiguousarray(c[:n], np.int32)
        r *= 1.15


class Run:
    """A conv of one kind of stores: out() on a plan, and which of its rows read an absent tap."""

    def __init__(self, tsp, shells, kind, kernel, ci, key="bf16", order=None):
        import torch
        self.tsp, self.kind, self.ci = tsp, kind, ci
        self.n, self.co = _case(tsp, kind, kernel, ci)
        print(f"[conv kernels] {kind} {kernel} n={self.n} ci={ci} co={self.co} {key}", flush=True)
        self.dt = torch.bfloat16 if key == "bf16" else torch.float16
        coords = _shell(shells, self.n)
        if order is not None:
            coords = np.concatenate([coords[:1], coords[1:][order.permutation(self.n - 1)]])
        g = torch.Generator(device="cuda").manual_seed(self.n + ci)
        rand = lambda shape, std: torch.randn(shape, generator=g, device="cuda") * std
        self.x = rand((self.n, ci), 1.0)
        self.w = rand((self.co, 27, ci), (27 * ci) ** -0.5).to(self.dt)
        self.b = rand((self.co,), 0.1)
        self.c = torch.from_numpy(np.ascontiguousarray(coords)).cuda()
        self.nbr, self.plan = tsp.rulebook_build_planned(self.c)
        t = self.nbr.reshape(27, self.n)
        self.absent = (t == self.n).any(0)
        self.near0 = (t == 0).any(0)
        if kind in ("octants", "c2s 64", "c2s 128"):
            self.mask = (torch.rand((self.n, 8), generator=g, device="cuda") < 0.4).to(torch.uint8)
            self.child, self.gidx, self.mstart = tsp.subdivide(self.mask, self.c)
        if kind in ("c2s 64", "c2s 128"):
            cout = self.co // 8
            self.cnbr, self.cplan = tsp.rulebook_build_planned(self.child)
            self.w2, self.b2 = rand((cout, 27, cout), (27 * cout) ** -0.5).to(self.dt), rand((cout,), 0.1)
        if kind == "skip":
            self.sx = rand((self.n // 4, 128), 1.0)
            self.sg = torch.randint(0, 8 * (self.n // 4), (self.n,), generator=g, device="cuda", dtype=torch.int32)
        if kind.startswith("norm"):
            self.nw, self.nb = 1 + rand((self.co,), 0.1), rand((self.co,), 0.1)

    def conv(self, f, out_dtype, plan=None, zero_pad=False):
        """The plain planned conv."""
        return self.tsp.subm_conv3x3_planned(f, self.nbr, self.plan if plan is None else plan,
                                             self.tsp.conv_weight_pack(self.w), self.b, self.co, out_dtype=out_dtype,
                                             zero_pad=zero_pad)

    def out(self, plan=None):
        import torch
        tsp, f, plan = self.tsp, self.x.to(self.dt), self.plan if plan is None else plan
        pw = tsp.conv_weight_pack(self.w)
        if self.kind in ("f32", "16-bit", "64"):
            return self.conv(f, self.dt if self.kind == "16-bit" else torch.float32, plan)
        if self.kind == "octants":
            return tsp.subm_conv3x3_planned_octants(f, self.nbr, plan, pw, self.b, self.co // 8, self.mask, self.mstart,
                                                    len(self.gidx))
        if self.kind == "skip":
            return tsp.subm_conv3x3_planned_skip(f, self.nbr, plan, pw, self.b, self.co, self.sx, self.sg)
        if self.kind.startswith("norm"):
            return tsp.subm_conv3x3_planned_ln(f, self.nbr, plan, pw, self.b, self.co, self.nw, self.nb)
        return tsp.c2s(self.x, self.nbr, self.mask, self.mstart, self.gidx, len(self.gidx), self.co // 8, self.cnbr,
                       {"norm1.weight": torch.ones(self.ci, device="cuda"), "norm1.bias": torch.zeros(self.ci, device="cuda"),
                        "conv1.weight": self.w, "conv1.bias": self.b, "conv2.weight": self.w2, "conv2.bias": self.b2},
                       plan=plan, child_plan=self.cplan)

    def reference(self):
        """The same by a kernel that gathers each row (its f32 conv) and separate passes."""
        import torch
        tsp, f = self.tsp, self.x.to(self.dt)
        if self.kind.startswith("c2s"):
            f = tsp.layer_norm(self.x, torch.ones(self.ci, device="cuda"), torch.zeros(self.ci, device="cuda"), 1e-6,
                               silu=True, out_dtype=self.dt)
        h = tsp.subm_conv3x3(f, self.nbr, self.w, self.b, out_dtype=torch.float32,
                             algo="narrow" if self.ci % 32 else "mfma_gather", zero_pad=self.kind == "skip")
        if self.kind in ("octants", "c2s 64", "c2s 128"):
            h = tsp.c2s_gather(h, self.gidx, self.co // 8)
        if self.kind.startswith("c2s"):
            h = tsp.layer_norm(h, None, None, 1e-6, silu=True, out_dtype=self.dt)
            h = tsp.subm_conv3x3(h, self.cnbr, self.w2, self.b2, out_dtype=torch.float32, algo="mfma_gather", zero_pad=True)
            tsp.c2s_skip_add(self.x, self.gidx, h)
        if self.kind == "skip":
            tsp.c2s_skip_add(self.sx, self.sg, h)
        if self.kind.startswith("norm"):
            h = tsp.layer_norm(h, self.nw, self.nb, 1e-6)
        return h


def _same(out, ref, tol):
    """The same values that are not finite, and the rest within tol of the largest."""
    import torch
    out, ref = out.float(), ref.float()
    assert torch.equal(out.isnan(), ref.isnan())
    inf = ref.isinf()
    assert torch.equal(out.isinf(), inf) and torch.equal(out[inf], ref[inf])
    ok = ref.isfinite()
    if not bool(ok.any()):   # (a weight that is not finite, then a norm: no row is)
        return
    assert float((out[ok] - ref[ok]).abs().max() / ref[ok].abs().max()) < tol


# f32 sums in two orders; a rounding of the result to 16 bits; the C2S block also rounds conv2's input,
# where a value that rounds the other way is one 16-bit step off
TOL = {"16-bit": TOL_16_OUT, "norm 64": TOL_16_OUT, "norm 128": TOL_16_OUT, "c2s 64": TOL_16_OUT, "c2s 128": TOL_16_OUT}


@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("kernel", ["small", "large"])
@pytest.mark.parametrize("bad", ["none", "row 0 inf", "row 0 nan", "weight inf", "weight nan"])
def test_edge_values(gpu_lib, shells, kind, kernel, bad):
    """Against the gather kernel and separate passes. Row 0 not finite: every row with an
    absent tap is NaN (with the skip stores, whose padding row is an exact zero, only row 0's
    neighbours); a weight that is not: every tap runs, 0 W being NaN."""
    import torch
    r = Run(gpu_lib, shells, kind, kernel, 32)
    value = float("nan") if bad.endswith("nan") else float("inf")
    if bad.startswith("row 0"):
        r.x[0, 7] = value
    if bad.startswith("weight"):
        r.w[5, 3, 9] = value
    out = r.out()
    assert bool(out.isfinite().any()) or (bad.startswith("weight") and kind.startswith("norm"))
    _same(out, r.reference(), TOL.get(kind, TOL_16))
    if bad.startswith("row 0") and kind in ("f32", "16-bit", "64", "norm 64", "norm 128"):
        assert bool(r.absent.any()) and bool((~r.absent & ~r.near0).any())
        assert bool(out[r.absent].isnan().all()) and bool(out[~r.absent & ~r.near0].isfinite().all())


@pytest.mark.parametrize("kernel", ["small", "large"])
@pytest.mark.parametrize("kind", ["f32", "octants", "norm 64", "skip"])
@pytest.mark.parametrize("key", ["bf16", "f16"])
def test_rows_from_memory(gpu_lib, shells, kind, kernel, key):
    """Voxels in random order and tiles of consecutive rows: more distinct rows than are staged, so the
    tiles gather them from memory -- to the bits of the Morton plan's tiles."""
    import torch
    r = Run(gpu_lib, shells, kind, kernel, 48, key, order=np.random.default_rng(1))
    rows = gpu_lib.conv_plan_build(r.nbr, r.n)
    head = rows[:16 * (r.n // 512)].view(torch.int32).reshape(-1, 4)
    assert bool((head[:, 1] == 1).any())
    out = r.out(rows)
    assert torch.equal(out, r.out())
    _same(out, r.reference(), TOL.get(kind, TOL_16))


@pytest.mark.parametrize("kernel", ["small", "large"])
@pytest.mark.parametrize("ci", [16, 48, 80])
def test_odd_slices_and_zero_padding(gpu_lib, orc, shells, kernel, ci):
    """An odd number of 16-channel slices (no pipelining over tiles), with the padding row an exact zero
    though row 0 is not finite, against the oracle on sampled rows."""
    import torch
    r = Run(gpu_lib, shells, "f32", kernel, ci)
    r.x[0, 3] = float("inf")
    out = r.conv(r.x.to(r.dt), torch.float32, zero_pad=True)
    far = (~r.near0).nonzero().squeeze(1).cpu().numpy()
    assert bool(out[~r.near0].isfinite().all())
    pick = np.random.default_rng(ci).choice(far, 200, replace=False)
    feats = r.x.to(r.dt).float().cpu().numpy()
    feats[0] = 0
    ref = orc.subm_conv_f64_rows(feats, r.nbr.cpu().numpy(), r.w.float().cpu().numpy(), r.b.cpu().numpy(), pick)
    assert orc.rel_err(out.cpu().numpy()[pick], ref) < TOL_16
