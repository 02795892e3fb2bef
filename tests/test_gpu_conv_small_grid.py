"""GPU parity of the small-grid planned conv (csrc/conv_split_kernel.hpp): a tile's row groups, its
channels and a slice's taps spread over several workgroups and waves.

The cases sit where its pieces can go wrong: each number of row groups a unit (1, 2, 4 -- by the
voxel count and the channels, on 256 compute units), a last tile of one voxel and of one past a
row group, an odd number of 16-channel slices, tiles staged 32 and (more than 1024 distinct rows,
as tiles of consecutive rows of a shell have) 16 channels at a time, and each kind of stores.

The sums of an output are in one order with and without a plan and whatever its tile order, so the
convs are compared bit for bit; against the fp64 oracle, sampled rows at the bars of
test_gpu_conv.py (fp32 accumulation; one rounding where the output is 16-bit)."""
from __future__ import annotations

import numpy as np
import pytest

from host_cases import rounding_noise_floor

pytestmark = pytest.mark.gpu

TOL_16 = 1e-3
TOL_16_OUT = 4e-3


def _shell(shells, n):
    """n voxels of a shell, sorted (consecutive rows: 1.0-1.9 K distinct neighbour rows a tile)."""
    r = 10.0
    while True:
        g = int(2 * r) + 8
        c = shells.sphere_shell(g, g / 2, r - 1.0, r + 1.0)
        if len(c) >= n:
            return np.ascontiguousarray(c[:n], np.int32)
        r *= 1.25


def _inputs(shells, n, ci, co, key, seed):
    import torch
    dt = torch.bfloat16 if key == "bf16" else torch.float16
    rng = np.random.default_rng(seed)
    feats = shells.round_to(rng.standard_normal((n, ci)).astype(np.float32), key)
    weight = shells.round_to((rng.standard_normal((co, 27, ci)) / np.sqrt(27 * ci)).astype(np.float32), key)
    bias = (rng.standard_normal(co) * 0.1).astype(np.float32)
    dev = [torch.from_numpy(feats).to(dt).cuda(), torch.from_numpy(weight).to(dt).cuda(), torch.from_numpy(bias).cuda()]
    return rng, dt, feats, weight, bias, dev


# (n, ci, co): units of 1 row group (the first five), of 2, of 4
SIZES = [(1, 64, 64), (513, 64, 128), (1153, 48, 64), (2606, 16, 192), (15000, 128, 128),
         (33001, 64, 64), (20000, 64, 128), (40001, 32, 128), (35003, 128, 128)]


@pytest.mark.parametrize("n,ci,co", SIZES)
@pytest.mark.parametrize("key", ["bf16", "f16"])
def test_small_grid_plain(gpu_lib, orc, shells, n, ci, co, key):
    """The conv on a Morton plan, on a plan of consecutive rows and without a plan: the same bits, and
    the oracle's values on the first, last and random rows; 16-bit output: the f32 one rounded."""
    import torch
    print(f"[small grid] n={n} ci={ci} co={co} {key}", flush=True)
    rng, dt, feats, weight, bias, (f, w, b) = _inputs(shells, n, ci, co, key, n + ci)
    coords = _shell(shells, n)
    c = torch.from_numpy(coords).cuda()
    nbr, plan = gpu_lib.rulebook_build_planned(c)
    pw = gpu_lib.conv_weight_pack(w)
    out = gpu_lib.subm_conv3x3_planned(f, nbr, plan, pw, b, co, out_dtype=torch.float32)
    rows = gpu_lib.subm_conv3x3_planned(f, nbr, gpu_lib.conv_plan_build(nbr, n), pw, b, co, out_dtype=torch.float32)
    out16 = gpu_lib.subm_conv3x3_planned(f, nbr, plan, pw, b, co)
    assert torch.equal(out, rows)
    assert torch.equal(out16, out.to(dt))
    if ci % 32 == 0:
        assert torch.equal(out, gpu_lib.subm_conv3x3(f, nbr, w, b, out_dtype=torch.float32, algo="mfma"))
    pick = np.unique(np.concatenate([np.arange(min(n, 40)), np.arange(max(0, n - 200), n), rng.integers(0, n, 300)]))
    ref = orc.subm_conv_f64_rows(feats, nbr.cpu().numpy(), weight, bias, pick)
    assert orc.rel_err(out.cpu().numpy()[pick], ref) < TOL_16


@pytest.mark.parametrize("n,ci,cout", [(700, 64, 64), (6000, 128, 64), (3001, 256, 128), (9000, 64, 128),
                                       (2100, 512, 256)])
@pytest.mark.parametrize("key", ["bf16", "f16"])
def test_small_grid_c2s_stores(gpu_lib, orc, shells, n, ci, cout, key):
    """The octant stores (bit for bit the conv, then the gather), the skip stores (the conv, then the
    skip pass), and the C2S block, whose conv1 stores normalise at Cout = 64 and 128, against the
    oracle's block on sampled rows at the bar of test_gpu_composite.py (1.5 x the case's rounding
    noise floor)."""
    import torch
    print(f"[small grid] c2s n={n} ci={ci} cout={cout} {key}", flush=True)
    co = 8 * cout
    rng, dt, feats, weight, bias, (f, w, b) = _inputs(shells, n, ci, co, key, n + cout)
    coords = _shell(shells, n)
    c = torch.from_numpy(coords).cuda()
    nbr, plan = gpu_lib.rulebook_build_planned(c)
    mask = (rng.random((n, 8)) < 0.5).astype(np.uint8)
    mask[::9] = 0
    mt = torch.from_numpy(mask.reshape(-1)).cuda()
    child, gidx, mstart = gpu_lib.subdivide(mt, c)
    m = len(gidx)
    pw = gpu_lib.conv_weight_pack(w)
    full = gpu_lib.subm_conv3x3_planned(f, nbr, plan, pw, b, co, out_dtype=torch.float32)
    fused = gpu_lib.subm_conv3x3_planned_octants(f, nbr, plan, pw, b, cout, mt, mstart, m)
    assert torch.equal(fused, gpu_lib.c2s_gather(full, gidx, cout))
    cnbr, cplan = gpu_lib.rulebook_build_planned(child)
    _, _, _, w2, b2, (f2, w2d, b2d) = _inputs(shells, m, cout, cout, key, n)
    cin = 2 * cout
    x = torch.from_numpy(rng.standard_normal((n, cin)).astype(np.float32)).cuda()
    pw2 = gpu_lib.conv_weight_pack(w2d)
    two = gpu_lib.subm_conv3x3_planned(f2, cnbr, cplan, pw2, b2d, cout, out_dtype=torch.float32)
    gpu_lib.c2s_skip_add(x, gidx, two)
    assert torch.equal(gpu_lib.subm_conv3x3_planned_skip(f2, cnbr, cplan, pw2, b2d, cout, x, gidx), two)
    if cout > 128:
        return
    w1 = shells.round_to((rng.standard_normal((co, 27, cin)) / np.sqrt(27 * cin)).astype(np.float32), key)
    p = {"norm1.weight": np.ones(cin, np.float32), "norm1.bias": np.zeros(cin, np.float32), "conv1.weight": w1,
         "conv1.bias": bias, "conv2.weight": w2, "conv2.bias": b2}
    pd = {k: torch.from_numpy(v).cuda().to(dt if v.ndim == 3 else torch.float32) for k, v in p.items()}
    blk = gpu_lib.c2s(x, nbr, mt, mstart, gidx, m, cout, cnbr, pd, plan=plan, child_plan=cplan)
    pick = np.unique(np.concatenate([np.arange(20), np.arange(m - 20, m), rng.integers(0, m, 60)]))
    q, wt = {"b." + k: v for k, v in p.items()}, {"b." + k: (key if v.ndim == 3 else "f32") for k, v in p.items()}
    (ref, _), floor = rounding_noise_floor(
        orc, lambda: orc.c2s_block_rows(x.cpu().numpy(), coords, q, "b", cout, mask, pick, wt), runs=2)
    assert orc.rel_err(blk.cpu().numpy()[pick], ref) < max(2e-4, 1.5 * floor)


@pytest.mark.parametrize("n,ci,co", [(1, 128, 128), (5001, 128, 128), (35001, 128, 128), (2049, 48, 64), (34000, 64, 64)])
@pytest.mark.parametrize("key", ["bf16", "f16"])
def test_small_grid_row_norm(gpu_lib, orc, shells, n, ci, co, key):
    """The conv with its LayerNorm in the stores against the oracle's conv and norm on sampled rows."""
    import torch
    print(f"[small grid] row norm n={n} ci={ci} co={co} {key}", flush=True)
    rng, dt, feats, weight, bias, (f, w, b) = _inputs(shells, n, ci, co, key, n + co)
    c = torch.from_numpy(_shell(shells, n)).cuda()
    nbr, plan = gpu_lib.rulebook_build_planned(c)
    nw = (1 + 0.1 * rng.standard_normal(co)).astype(np.float32)
    nb = (0.1 * rng.standard_normal(co)).astype(np.float32)
    out = gpu_lib.subm_conv3x3_planned_ln(f, nbr, plan, gpu_lib.conv_weight_pack(w), b, co,
                                          torch.from_numpy(nw).cuda(), torch.from_numpy(nb).cuda())
    pick = np.unique(np.concatenate([np.arange(min(n, 40)), np.arange(max(0, n - 200), n), rng.integers(0, n, 300)]))
    ref = orc.layer_norm(orc.subm_conv_f64_rows(feats, nbr.cpu().numpy(), weight, bias, pick), nw, nb, 1e-6)
    assert orc.rel_err(out.float().cpu().numpy()[pick], ref) < TOL_16_OUT
