"""The C2S block's octant plan (csrc/plan.hip) where it is not the usual call: a workspace without
room for it, or not aligned; masks that keep some octants far more often than others; the
block in parts; weights and a row 0 that are not finite."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _al(b):
    return (b + 255) // 256 * 256


def _without_plan(n, m, cin, cout):
    """The C2S workspace without the octant plan (both plans given, packed 16-bit weights): norm1's
    output, conv1's rows in f32 where its stores do not normalise, conv2's input, the block words."""
    return (_al(2 * n * cin) + (0 if cout in (64, 128) else _al(4 * m * cout)) + _al(2 * m * cout)
            + _al(16 * -(-n // 512)))


def _block(tsp, shells, n, cin, cout, keep, key="bf16", seed=0, counts=None):
    """A C2S block with device tensors: n parents of a shell, octant o kept with probability keep[o], or by
    exactly counts[o] of them."""
    import torch
    dt = torch.bfloat16 if key == "bf16" else torch.float16
    rng = np.random.default_rng(n + cin + seed)
    coords = shells.sphere_shell(96, 48.0, 34.0, 36.4 if n > 12000 else 35.6)
    assert len(coords) >= n
    c = torch.from_numpy(np.ascontiguousarray(coords[:n], np.int32)).cuda()
    mask = (rng.random((n, 8)) < np.asarray(keep)).astype(np.uint8)
    if counts is not None:
        mask = np.stack([rng.permutation(n) < k for k in counts], 1).astype(np.uint8)
    mask = torch.from_numpy(mask.reshape(-1)).cuda()
    g = torch.Generator(device="cuda")
    g.manual_seed(n + seed)
    rand = lambda shape, std, d: (torch.randn(shape, generator=g, device="cuda") * std).to(d)
    p = {"norm1.weight": 1 + rand((cin,), 0.1, torch.float32), "norm1.bias": rand((cin,), 0.1, torch.float32),
         "conv1.weight": rand((8 * cout, 27, cin), (27 * cin) ** -0.5, dt), "conv1.bias": rand((8 * cout,), 0.1, torch.float32),
         "conv2.weight": rand((cout, 27, cout), (27 * cout) ** -0.5, dt), "conv2.bias": rand((cout,), 0.1, torch.float32)}
    p["conv1.packed"], p["conv2.packed"] = tsp.conv_weight_pack(p["conv1.weight"]), tsp.conv_weight_pack(p["conv2.weight"])
    nbr, plan = tsp.rulebook_build_planned(c)
    child, gidx, mstart = tsp.subdivide(mask, c)
    cnbr, cplan = tsp.rulebook_build_planned(child)
    x = rand((n, cin), 1.0, torch.float32)
    return {"n": n, "m": len(gidx), "cin": cin, "cout": cout, "x": x, "nbr": nbr, "plan": plan, "mask": mask,
            "gidx": gidx, "mstart": mstart, "cnbr": cnbr, "cplan": cplan, "p": p}


def _weights(tsp, p):
    from trellis_cpp_amd import C2SWeights
    ptr, code = (lambda t: ctypes.c_void_p(t.data_ptr())), tsp.dtype_code
    return C2SWeights(ptr(p["norm1.weight"]), ptr(p["norm1.bias"]), ptr(p["conv1.weight"]), code(p["conv1.weight"].dtype),
                      ptr(p["conv1.bias"]), ptr(p["conv1.packed"]), ptr(p["conv2.weight"]), code(p["conv2.weight"].dtype),
                      ptr(p["conv2.bias"]), ptr(p["conv2.packed"]))


def _run(tsp, b, ws, ws_bytes):
    """tsp_c2s on the workspace's first ws_bytes -> (status, out)."""
    import torch
    ptr = lambda t: ctypes.c_void_p(t.data_ptr()) if t is not None else None
    out = torch.full((b["m"], b["cout"]), float("nan"), device="cuda")
    st = tsp.lib().tsp_c2s(ptr(b["x"]), b["n"], b["cin"], ptr(b["nbr"]), ptr(b["plan"]), ptr(b["mask"]), ptr(b["mstart"]),
                           ptr(b["gidx"]), b["m"], b["cout"], ptr(b["cnbr"]), ptr(b["cplan"]),
                           ctypes.byref(_weights(tsp, b["p"])), ptr(out), ptr(ws), ws_bytes, 0,
                           ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    return st, out


def _bytes(tsp, b, m=None):
    return tsp.lib().tsp_c2s_workspace_bytes(b["n"], b["m"] if m is None else m, b["cin"], b["cout"],
                                             ctypes.byref(_weights(tsp, b["p"])), 1, 1, 0)


@pytest.mark.parametrize("n,cin,cout", [(14001, 256, 128), (8001, 512, 256)])
def test_workspace_without_the_plan(gpu_lib, shells, n, cin, cout):
    """A workspace of the size without the octant plan -- what callers asked for before there was one,
    or sized for more children than there are -- is accepted, gives the same bits and is not written
    past its end; a byte less is refused."""
    import torch
    print(f"[octant plan] small workspace n={n} {cin}->{cout}", flush=True)
    b = _block(gpu_lib, shells, n, cin, cout, [0.5] * 8)
    full, less = _bytes(gpu_lib, b), _without_plan(n, b["m"], cin, cout)
    assert less < full, "the case is meant to take an octant plan"
    ws = torch.full((full,), 0xA5, dtype=torch.uint8, device="cuda")
    st, want = _run(gpu_lib, b, ws, full)
    assert st == 0
    ws.fill_(0xA5)
    for size in (less, full - 1):
        st, got = _run(gpu_lib, b, ws, size)
        assert st == 0 and torch.equal(got, want)
    assert bool((ws[less:] == 0xA5).all())
    assert _run(gpu_lib, b, ws, less - 1)[0] == 5
    # sized for every octant kept, where conv1 takes no plan
    assert _bytes(gpu_lib, b, 8 * n) == _without_plan(n, 8 * n, cin, cout)
    st, got = _run(gpu_lib, b, ws, min(full, _bytes(gpu_lib, b, 8 * n)))
    assert st == 0 and torch.equal(got, want)


@pytest.mark.parametrize("n,cin,cout", [(14001, 256, 128), (24000, 256, 128)])
def test_workspace_not_aligned(gpu_lib, shells, n, cin, cout):
    """A workspace 8 bytes off 16 runs conv1 without an octant plan: with no child plan the block is the
    aligned one's up to the order of conv2's sums (at most 2 K eps sum|w h|, |h| of rms about 0.6 after
    LN + SiLU and |w_o| about 1); with one it is refused, as conv2 on the matrix cores needs 16 bytes."""
    import torch
    print(f"[octant plan] unaligned workspace n={n} {cin}->{cout}", flush=True)
    b = _block(gpu_lib, shells, n, cin, cout, [0.5] * 8)
    size = _bytes(gpu_lib, b)
    assert _without_plan(n, b["m"], cin, cout) < size, "the case is meant to take an octant plan"
    ws = torch.full((size + 16,), 0xA5, dtype=torch.uint8, device="cuda")
    assert _run(gpu_lib, b, ws[8:], size)[0] == 1
    b = {**b, "cplan": None}
    st, want = _run(gpu_lib, b, ws, size)
    assert st == 0
    ws.fill_(0xA5)
    st, got = _run(gpu_lib, b, ws[8:], size)
    k = 27 * cout
    assert st == 0
    torch.testing.assert_close(got, want, rtol=0, atol=2 * k * 2.0 ** -24 * k ** 0.5)
    assert bool((ws[:8] == 0xA5).all()) and bool((ws[8 + size:] == 0xA5).all())


# keep probabilities of the octants, and whether the plan then pays: only where its fullest octant has
# clearly fewer tiles than the parents (large grid) or all octants together do (small grid)
MASKS = {"half": [0.5] * 8, "rare": [0.3] * 8, "two rates": [0.4, 0.6] * 4, "one full": [1.0] + [0.05] * 7,
         "half full": [0.9] * 4 + [0.1] * 4, "none": [0.0, 0.001] + [0.5] * 6}


def _front_us(tsp, b, ws, ws_bytes):
    """The shortest of five runs of the block's front part (conv1 and its norms), us."""
    import torch
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    out = torch.empty((b["m"], b["cout"]), device="cuda")
    best = float("inf")
    for _ in range(5):
        t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        t0.record()
        st = tsp.lib().tsp_c2s_part(ptr(b["x"]), b["n"], b["cin"], ptr(b["nbr"]), ptr(b["plan"]), ptr(b["mask"]),
                                    ptr(b["mstart"]), ptr(b["gidx"]), b["m"], b["cout"], ptr(b["cnbr"]), ptr(b["cplan"]),
                                    ctypes.byref(_weights(tsp, b["p"])), ptr(out), None, 2, ptr(ws), ws_bytes, 0, 1, 0, -1,
                                    ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        t1.record()
        torch.cuda.synchronize()
        assert st == 0
        best = min(best, t0.elapsed_time(t1) * 1e3)
    return best


@pytest.mark.parametrize("n,cin,cout", [(24001, 256, 128), (30001, 256, 128), (14001, 256, 128), (12001, 512, 256), (9001, 256, 384)])
@pytest.mark.parametrize("keep", list(MASKS))
def test_uneven_octants(gpu_lib, shells, n, cin, cout, keep):
    """Each octant's tiles are its own (none is empty or reads its rows from memory), a plan that does
    not pay is not run, and the block is the same bits either way. A mask that keeps the octants
    unevenly runs about as fast as with a workspace without room for the plan: within a factor of 2
    here, where tiles of parents far apart, or eight times the fullest octant's tiles, take 3 to 6."""
    import torch
    print(f"[octant plan] {keep} n={n} {cin}->{cout}", flush=True)
    b = _block(gpu_lib, shells, n, cin, cout, MASKS[keep])
    full, less = _bytes(gpu_lib, b), _without_plan(n, b["m"], cin, cout)
    ws = torch.empty(full, dtype=torch.uint8, device="cuda")
    st, got = _run(gpu_lib, b, ws, full)
    assert st == 0
    if full > less:   # (the plan's state is the first of its pieces)
        state = ws[less:less + 37 * 4].view(torch.int32).tolist()
        fits, spare, direct, total, most = state[:5]
        tiles, base, rows, count = (np.array(state[5 + 8 * k:13 + 8 * k]) for k in range(4))
        kept = (b["mask"].reshape(n, 8) != 0).sum(0).cpu().numpy()
        assert np.array_equal(count, kept) and np.array_equal(tiles, -(-kept // rows))
        assert total == tiles.sum() and most == tiles.max() and np.array_equal(base, np.cumsum(tiles) - tiles)
        assert direct == 0 and (rows <= 512).all()
        if fits:
            assert most <= -(-n // 512)
        if keep in ("one full", "half full") or (n == 14001 and keep != "rare"):   # (14 K: a round on either plan)
            assert not fits
        elif keep in ("half", "rare") and n != 14001:
            assert fits
    st, want = _run(gpu_lib, b, ws, less)
    assert st == 0 and torch.equal(got, want)
    assert _front_us(gpu_lib, b, ws, full) < 2 * _front_us(gpu_lib, b, ws, less) + 50


def _part(tsp, b, ws, ws_bytes, out, part, t0=0, nt=-1):
    import torch
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    return tsp.lib().tsp_c2s_part(ptr(b["x"]), b["n"], b["cin"], ptr(b["nbr"]), ptr(b["plan"]), ptr(b["mask"]),
                                  ptr(b["mstart"]), ptr(b["gidx"]), b["m"], b["cout"], ptr(b["cnbr"]), ptr(b["cplan"]),
                                  ctypes.byref(_weights(tsp, b["p"])), ptr(out), None, 2, ptr(ws), ws_bytes, 0, part, t0, nt,
                                  ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))


@pytest.mark.parametrize("n,cin,cout", [(24001, 256, 128), (12001, 512, 256)])
def test_parts(gpu_lib, shells, n, cin, cout):
    """The front part once, then conv2 over ranges of the child plan's tiles, and all parts at once on
    a stream of its own: the same bits, and nothing outside the range is written."""
    import torch
    print(f"[octant plan] parts n={n} {cin}->{cout}", flush=True)
    b = _block(gpu_lib, shells, n, cin, cout, [0.5] * 8, key="f16")
    full = _bytes(gpu_lib, b)
    ws = torch.empty(full, dtype=torch.uint8, device="cuda")
    st, want = _run(gpu_lib, b, ws, full)
    assert st == 0
    ws.fill_(0xA5)
    out = torch.full((b["m"], cout), float("nan"), device="cuda")
    tiles = -(-b["m"] // 512)
    assert _part(gpu_lib, b, ws, full, out, 1) == 0 and bool(out.isnan().all())
    cuts = [0, 1, tiles // 3, tiles - 1, tiles]
    for t0, t1 in zip(cuts[:-1], cuts[1:]):
        assert _part(gpu_lib, b, ws, full, out, 2, t0, t1 - t0) == 0
        torch.cuda.synchronize()
        assert int((~out[:, 0].isnan()).sum()) == min(b["m"], 512 * t1)
    assert torch.equal(out, want)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        st, got = _run(gpu_lib, b, ws, full)
    torch.cuda.current_stream().wait_stream(side)
    assert st == 0 and torch.equal(got, want)


@pytest.mark.parametrize("bad", ["weight inf", "weight nan", "row 0 nan"])
@pytest.mark.parametrize("n,cin,cout", [(24001, 256, 128), (30001, 256, 128), (12001, 512, 256)])
def test_values_not_finite(gpu_lib, shells, n, cin, cout, bad):
    """On the octant plan and on the parents' plan (whose conv is tested against the other kernels): the
    same values where they are numbers, NaN in the same places."""
    import torch
    print(f"[octant plan] {bad} n={n} {cin}->{cout}", flush=True)
    b = _block(gpu_lib, shells, n, cin, cout, [0.5] * 8)
    value = float("inf") if bad.endswith("inf") else float("nan")
    if bad.startswith("weight"):
        b["p"]["conv1.weight"][3 * cout + 7, 4, 11] = value   # (an octant's channel)
        b["p"]["conv1.packed"] = gpu_lib.conv_weight_pack(b["p"]["conv1.weight"])
    else:
        b["x"][0, 5] = value
    full, less = _bytes(gpu_lib, b), _without_plan(n, b["m"], cin, cout)
    assert less < full
    ws = torch.empty(full, dtype=torch.uint8, device="cuda")
    (st, got), (st2, want) = _run(gpu_lib, b, ws, full), _run(gpu_lib, b, ws, less)
    assert st == 0 and st2 == 0
    assert bool(want.isnan().any()) and torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got.nan_to_num(0.0), want.nan_to_num(0.0))


def test_captured(gpu_lib, shells):
    """The block in a captured graph, replayed with an even mask and with one that keeps two octants whole
    (the same number of children): each replay decides for its own mask, and matches the eager block."""
    import torch
    print("[octant plan] captured", flush=True)
    n, cin, cout = 24000, 256, 128
    even = _block(gpu_lib, shells, n, cin, cout, [0.5] * 8, counts=[n // 2] * 8)
    full_two = _block(gpu_lib, shells, n, cin, cout, [0.5] * 8, counts=[n] * 2 + [n // 3] * 6)
    assert even["m"] == full_two["m"]
    size, less = _bytes(gpu_lib, even), _without_plan(n, even["m"], cin, cout)
    ws = torch.empty(size, dtype=torch.uint8, device="cuda")
    want, took = {}, {}
    for name, b in (("even", even), ("two", full_two)):
        b["p"] = even["p"]
        st, want[name] = _run(gpu_lib, b, ws, size)
        assert st == 0
        took[name] = int(ws[less:less + 4].view(torch.int32)[0])
    assert took["even"] == 1
    live = {k: even[k].clone() for k in ("x", "nbr", "plan", "mask", "gidx", "mstart", "cnbr", "cplan")}
    b = {**even, **live}
    out = torch.empty((b["m"], cout), device="cuda")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        assert _part(gpu_lib, b, ws, size, out, 3) == 0
    for name, src in (("even", even), ("two", full_two), ("two", full_two), ("even", even)):
        for k, t in live.items():
            t.copy_(src[k])
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert int(ws[less:less + 4].view(torch.int32)[0]) == took[name]
        assert torch.equal(out, want[name])
