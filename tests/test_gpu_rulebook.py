"""GPU parity of the coordinate hash / neighbour table: bit-exact against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _gpu_table(pkg, coords):
    import torch
    c = torch.from_numpy(np.ascontiguousarray(coords, np.int32)).cuda()
    nbr = pkg.rulebook_build(c)
    torch.cuda.synchronize()
    return nbr.cpu().numpy()


def _case(name):
    print(f"[rulebook] {name}", flush=True)


@pytest.mark.parametrize("fixture", ["rulebook_rand800.npz", "rulebook_edges.npz"])
def test_golden(gpu_lib, golden, fixture):
    _case(fixture)
    g = golden(fixture)
    assert np.array_equal(_gpu_table(gpu_lib, g["coords"]), g["nbr"])


def test_edge_cases(gpu_lib, orc, shells):
    rng = np.random.default_rng(21)
    big = (1 << 21) - 3
    cases = {
        "single": np.array([[0, 0, 0]], np.int32),
        "duplicates": rng.integers(0, 12, size=(3000, 3)).astype(np.int32),
        "corners": np.array([[0, 0, 0], [big, big, big], [big, 0, big], [1, 0, 0],
                             [big - 1, big, big]], np.int32),
        "sparse-huge": rng.integers(0, big + 1, size=(5000, 3)).astype(np.int32),
        "dense-cube": np.array([(x, y, z) for x in range(10) for y in range(10)
                                for z in range(10)], np.int32),
        "shell-255": shells.sphere_shell(40, 20.0, 10.0, 11.0)[:255],
        "shell-257": shells.sphere_shell(40, 20.0, 10.0, 11.0)[:257],
        "unsorted": rng.permutation(shells.sphere_shell(40, 20.0, 12.0, 14.0)),
        # a cell directory fits the workspace but the occupied cells' blocks do not: the hash
        "scattered-box": rng.integers(0, 400, size=(20000, 3)).astype(np.int32),
        # duplicates spread over many cells of the grid
        "shell-duplicates": np.concatenate([shells.sphere_shell(40, 20.0, 12.0, 14.0)] * 2)[::-1].copy(),
        # rows in (x, y, z) order with repeats next to each other (the grid's duplicate fix is
        # skipped only for strictly ascending rows): every row twice, and one repeat whose two rows
        # fall in different workgroups of the ascending check
        "sorted-repeats": np.repeat(shells.sphere_shell(40, 20.0, 12.0, 14.0), 2, axis=0),
        "sorted-one-repeat": np.insert(shells.sphere_shell(40, 20.0, 12.0, 14.0), 256,
                                       shells.sphere_shell(40, 20.0, 12.0, 14.0)[255], axis=0),
    }
    import torch
    for name, c in cases.items():
        _case(name)
        ref = orc.neighbor_table_sorted(c)
        assert np.array_equal(_gpu_table(gpu_lib, c), ref), name
        # pair count, also of a copy of the table that starts 1-3 elements past a 16-byte boundary
        n, want = len(c), int((ref != len(c)).sum())
        for off in range(4):
            buf = torch.zeros(27 * n + off, dtype=torch.int32, device="cuda")
            buf[off:] = torch.from_numpy(ref).cuda()
            view = buf[off:]
            assert view.data_ptr() % 16 == 4 * off
            assert gpu_lib.count_pairs(view, n) == want, (name, off)


def test_empty(gpu_lib):
    import torch
    nbr = gpu_lib.rulebook_build(torch.zeros((0, 3), dtype=torch.int32, device="cuda"))
    assert nbr.numel() == 0


def test_out_of_range_reported(gpu_lib):
    import torch
    for bad in ([-1, 0, 0], [0, (1 << 21) - 2, 0]):
        c = torch.tensor([[1, 1, 1], bad], dtype=torch.int32, device="cuda")
        with pytest.raises(gpu_lib.TspError):
            gpu_lib.rulebook_build(c)


@pytest.mark.parametrize("name", ["shell64-c64-f32", "shells256-c128-bf16"])
def test_workload_bit_exact(gpu_lib, orc, shells, name):
    _case(name)
    import torch
    w = shells.workload(name)
    c = torch.from_numpy(w.coords).cuda()
    nbr = gpu_lib.rulebook_build(c)
    again = gpu_lib.rulebook_build(c)
    got = nbr.cpu().numpy()
    ref = orc.neighbor_table(w.coords)
    assert np.array_equal(got, ref)
    assert torch.equal(nbr, again)                                   # deterministic
    assert gpu_lib.count_pairs(nbr, w.n) == orc.count_pairs(ref, w.n)


def test_one_voxel_per_brick_bit_exact(gpu_lib, orc):
    """Every voxel in a 2x2x2 brick of its own: the table holds N bricks in 1.5 N + 1024 buckets,
    the fullest it gets, so probe sequences run longest. 10^6 voxels on a 100^3 brick grid, each
    at a random octant, so neighbouring bricks still give neighbours."""
    _case("one-voxel-per-brick 100^3")
    rng = np.random.default_rng(5)
    a = np.stack(np.meshgrid(*(np.arange(100, dtype=np.int32),) * 3, indexing="ij"), -1)
    # voxel x lies in brick (x + 1) >> 1: x = 2a + 1 + e with e in {0, 1} gives brick a + 1
    c = (2 * a.reshape(-1, 3) + rng.integers(0, 2, size=(a.size // 3, 3)) + 1).astype(np.int32)
    c = c[rng.permutation(len(c))]
    ref = orc.neighbor_table(c)
    assert np.array_equal(_gpu_table(gpu_lib, c), ref)
    assert (ref[13 * len(c):14 * len(c)] == np.arange(len(c))).all()   # centre tap: itself


def _spread(n, ext, seed=5):
    rng = np.random.default_rng(seed)
    return np.unique(rng.integers(0, ext, (n, 3)).astype(np.int32), axis=0)


@pytest.mark.parametrize("n,ext", [(1, 1), (600, 40), (2000, 120), (2000, 1000), (700, 1020), (70000, 300)])
def test_wide_boxes(gpu_lib, orc, n, ext):
    """Tables and ordered plans where the directory and the blocks outnumber the voxels' scans: one
    word, rounds of four words a thread over several workgroups, several rounds a workgroup."""
    import torch
    _case(f"wide box {n} {ext}")
    coords = _spread(n, ext)
    n = len(coords)
    c = torch.from_numpy(coords).cuda()
    ref = orc.neighbor_table_sorted(coords)
    assert np.array_equal(_gpu_table(gpu_lib, coords), ref)
    nbr, joint = gpu_lib.rulebook_build_planned(c)
    assert np.array_equal(nbr.cpu().numpy(), ref)
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn((n, 32), generator=g, device="cuda").to(torch.bfloat16)
    w = torch.randn((64, 27, 32), generator=g, device="cuda").to(torch.bfloat16)
    b = torch.randn(64, generator=g, device="cuda")
    want = gpu_lib.subm_conv3x3(x, nbr, w, b, out_dtype=torch.float32, algo="mfma")
    pw = gpu_lib.conv_weight_pack(w)
    for plan in (joint, gpu_lib.conv_plan_build(nbr, n, coords=c)):
        out = torch.full((n, 64), float("nan"), device="cuda")
        gpu_lib.subm_conv3x3_planned(x, nbr, plan, pw, b, 64, out=out, out_dtype=torch.float32)
        assert torch.equal(out, want)


def test_wide_box_time(gpu_lib):
    """The ordered plan of a few voxels takes about the same time in a box with 8 times the directory
    (2^21 words): 1.02 times as long; 1.5 with workgroups for the voxels alone."""
    import torch
    us = []
    for ext in (500, 1000):
        _case(f"wide box time {ext}")
        c = torch.from_numpy(_spread(2000, ext)).cuda()
        nbr = gpu_lib.rulebook_build(c)
        plan = gpu_lib.conv_plan_build(nbr, len(c), coords=c)
        best = float("inf")
        for _ in range(5):
            t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            t0.record()
            for _ in range(20):
                gpu_lib.conv_plan_build(nbr, len(c), coords=c, plan=plan)
            t1.record()
            torch.cuda.synchronize()
            best = min(best, t0.elapsed_time(t1))
        us.append(best)
    assert us[1] < 1.3 * us[0]
