"""GPU parity of tsp_linear with at most 16 outputs (csrc/linear_thin.hip) against the fp64 product
of the same 16-bit values: fp32 accumulation (1e-5, as the other linears), and with 16-bit output the
f32 result rounded once. Sizes around a wave's 64 rows and a launch's whole grid, each channel step
count, and output counts the library GEMM does not take."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ci,co", [(1, 32, 1), (63, 64, 7), (64, 64, 6), (65, 128, 15), (257, 256, 3), (1000, 512, 9),
                                     (2048 * 256 + 17, 64, 7)])
@pytest.mark.parametrize("key", ["bf16", "f16"])
def test_linear_thin(gpu_lib, n, ci, co, key):
    import torch
    print(f"[linear thin] n={n} ci={ci} co={co} {key}", flush=True)
    dt = torch.bfloat16 if key == "bf16" else torch.float16
    g = torch.Generator(device="cuda")
    g.manual_seed(n + ci + co)
    x = torch.randn((n, ci), generator=g, device="cuda").to(dt)
    w = (torch.randn((co, ci), generator=g, device="cuda") / ci ** 0.5).to(dt)
    b = torch.randn(co, generator=g, device="cuda")
    prod = (x.double()[:, None, :] * w.double()[None]).sum(2) if n <= 2000 else x.double() @ w.double().t()
    out = gpu_lib.linear(x, w, b, out_dtype=torch.float32)
    ref = prod + b.double()
    assert ((out.double() - ref).abs().max() / ref.abs().max()).item() < 1e-5
    assert torch.equal(gpu_lib.linear(x, w, b), out.to(dt))
    bare = gpu_lib.linear(x, w, out_dtype=torch.float32)
    assert ((bare.double() - prod).abs().max() / prod.abs().max()).item() < 1e-5


def test_linear_thin_keeps_rows_apart(gpu_lib):
    """An Inf or a NaN in a row of x reaches that row of the output alone."""
    import torch
    x = torch.ones((130, 64), dtype=torch.float16, device="cuda")
    x[3, 5], x[129, 0] = float("inf"), float("nan")
    w = torch.ones((7, 64), dtype=torch.float16, device="cuda")
    out = gpu_lib.linear(x, w, out_dtype=torch.float32).cpu().numpy()
    assert np.isinf(out[3]).all() and np.isnan(out[129]).all()
    keep = np.delete(np.arange(130), [3, 129])
    assert (out[keep] == 64).all()
