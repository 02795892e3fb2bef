"""GPU parity of the C2S block with an octant plan (csrc/plan.hip octant_plan_build): conv1 over each
octant's kept parents only, where the device finds that it pays.

The cases sit where the plan can go wrong: octants kept by half, a quarter (tiles of fewer than 512
parents) and three quarters of the parents; both conv kernels (large grid, small grid); and where it
is built and not run: octants with very different totals, one with none; plan tiles of consecutive
rows and scattered voxels, whose octant tiles exceed the staged rows; a single round of units.
test_gpu_octant_plan_corners.py reads which of the two plans was run."""
from __future__ import annotations

import numpy as np
import pytest

from host_cases import rounding_noise_floor

pytestmark = pytest.mark.gpu


def _coords(shells, n, kind):
    if kind == "scattered":
        return np.ascontiguousarray(shells.random_distinct_voxels(n, 200, n), np.int32)
    c = shells.sphere_shell(96, 48.0, 34.0, 36.4 if n > 12000 else 35.6)
    assert len(c) >= n
    return np.ascontiguousarray(c[:n], np.int32)


def _mask(rng, n, keep):
    p = {"half": [0.5] * 8, "quarter": [0.27] * 8, "most": [0.75] * 8,
         "uneven": [1.0, 0.9, 0.05, 0.0, 0.6, 0.5, 0.3, 0.001]}[keep]
    return np.where(rng.random((n, 8)) < p, rng.integers(1, 256, (n, 8)), 0).astype(np.uint8)


@pytest.mark.parametrize("n,cin,cout,keep,kind,key", [
    (12001, 512, 256, "half", "morton", "bf16"), (8001, 512, 256, "uneven", "morton", "f16"),
    (8000, 512, 256, "quarter", "rows", "bf16"), (6000, 512, 256, "half", "morton", "f16"),
    (9000, 512, 256, "half", "scattered", "bf16"),
    (3500, 1024, 512, "most", "morton", "bf16"), (14001, 256, 128, "half", "morton", "f16"),
    (24001, 256, 128, "uneven", "morton", "bf16")])
def test_c2s_on_octant_plan(gpu_lib, orc, shells, n, cin, cout, keep, kind, key):
    """Against the block composed of the single entry points (norm1 + SiLU, the octant conv on the
    parents' plan, norm2 + SiLU, the skip conv): the same bits where conv1's stores do not normalise
    (Cout >= 256); at Cout = 128, whose stores do, against the oracle's block on sampled rows at the
    bar of test_gpu_composite.py."""
    import torch
    print(f"[octant plan] n={n} {cin}->{cout} {keep} {kind} {key}", flush=True)
    dt = torch.bfloat16 if key == "bf16" else torch.float16
    rng = np.random.default_rng(n + cin)
    coords = _coords(shells, n, kind)
    mask = _mask(rng, n, keep)
    x = rng.standard_normal((n, cin)).astype(np.float32)
    p = {"norm1.weight": (1 + 0.1 * rng.standard_normal(cin)).astype(np.float32),
         "norm1.bias": (0.1 * rng.standard_normal(cin)).astype(np.float32),
         "conv1.weight": shells.round_to((rng.standard_normal((8 * cout, 27, cin), dtype=np.float32) / np.sqrt(27 * cin)).astype(np.float32), key),
         "conv1.bias": (0.1 * rng.standard_normal(8 * cout)).astype(np.float32),
         "conv2.weight": shells.round_to((rng.standard_normal((cout, 27, cout), dtype=np.float32) / np.sqrt(27 * cout)).astype(np.float32), key),
         "conv2.bias": (0.1 * rng.standard_normal(cout)).astype(np.float32)}
    pd = {k: torch.from_numpy(v).cuda().to(dt if v.ndim == 3 else torch.float32) for k, v in p.items()}
    c = torch.from_numpy(coords).cuda()
    mt = torch.from_numpy(mask.reshape(-1)).cuda()
    nbr, plan = gpu_lib.rulebook_build_planned(c)
    if kind == "rows":
        plan = gpu_lib.conv_plan_build(nbr, n)
    child, gidx, mstart = gpu_lib.subdivide(mt, c)
    m = len(gidx)
    cnbr, cplan = gpu_lib.rulebook_build_planned(child)
    xd = torch.from_numpy(x).cuda()
    out = gpu_lib.c2s(xd, nbr, mt, mstart, gidx, m, cout, cnbr, pd, plan=plan, child_plan=cplan)
    if cout > 128:
        h0 = gpu_lib.layer_norm(xd, pd["norm1.weight"], pd["norm1.bias"], 1e-6, silu=True, out_dtype=dt)
        g = gpu_lib.subm_conv3x3_planned_octants(h0, nbr, plan, gpu_lib.conv_weight_pack(pd["conv1.weight"]),
                                                 pd["conv1.bias"], cout, mt, mstart, m)
        h2 = gpu_lib.layer_norm(g, None, None, 1e-6, silu=True, out_dtype=dt)
        ref = gpu_lib.subm_conv3x3_planned_skip(h2, cnbr, cplan, gpu_lib.conv_weight_pack(pd["conv2.weight"]),
                                                pd["conv2.bias"], cout, xd, gidx)
        assert torch.equal(out, ref)
        return
    pick = np.unique(np.concatenate([np.arange(20), np.arange(m - 20, m), rng.integers(0, m, 60)]))
    q, wt = {"b." + k: v for k, v in p.items()}, {"b." + k: (key if v.ndim == 3 else "f32") for k, v in p.items()}
    (ref, _), floor = rounding_noise_floor(
        orc, lambda: orc.c2s_block_rows(x, coords, q, "b", cout, mask, pick, wt), runs=2)
    assert orc.rel_err(out.cpu().numpy()[pick], ref) < max(2e-4, 1.5 * floor)
