"""GPU parity: the linear for more rows than a verify block (both of its forms) against the fp64 oracle.

bf16 outputs: one rounding (2^-9 of the value) of an fp32 sum; 4e-3 of the largest output covers it.  fp32 outputs:
fp32 sums of K products (24 + q) x, at most K 2^-24 of sum |24 + q| |x| |s|, observed 3e-7 of the norm; bound 2e-6.
"""
import numpy as np
import pytest
import torch

from oracle import w4

pytestmark = pytest.mark.gpu


def _case(pkg, m, n, k, group, scale_dtype, seed):
    gen = torch.Generator().manual_seed(seed)
    x = torch.randn((m, k), generator=gen).to(torch.bfloat16)
    return x, pkg.synthetic.int4_weight(gen, (n, k), group, scale_dtype)


@pytest.mark.parametrize("m,n,k,group,scale_dtype,layout", [
    (33, 32, 512, 128, torch.bfloat16, "portable"),      # one part of half its columns, a k-block a wave
    (1, 96, 1536, 128, torch.float32, "portable"),       # a K the small kernels do not take; three k-blocks a wave
    (65, 160, 2560, 256, torch.bfloat16, "portable"),    # a row past two parts, five k-blocks a wave
    (64, 512, 2048, 128, torch.float32, "tiled"),
    (333, 96, 4096, 256, torch.float32, "portable"),
    (70, 20768, 2048, 128, torch.bfloat16, "tiled"),     # 164 tiles: six rows in the second, 32 columns in the last
    (10300, 288, 512, 256, torch.float32, "portable"),   # tiles of one fragment and a half, same group twice
    (640, 4352, 1536, 128, torch.float32, "portable"),   # whole tiles, an even count of k-blocks
])
def test_linear_matches_oracle(pkg, device, m, n, k, group, scale_dtype, layout):
    print(f"linear m={m} n={n} k={k} g={group} {scale_dtype} {layout}", flush=True)
    x, weight = _case(pkg, m, n, k, group, scale_dtype, seed=m + n)
    weight.scales[3] = 0            # a row of zero scales
    weight.scales[5, 0] = 0         # a zero first group, a zero last group
    weight.scales[6, -1] = 0
    w = weight.to(device)
    if layout == "tiled":
        w = w.tiled()
    rows = torch.cat((torch.arange(min(m, 40)), torch.arange(max(0, m - 40), m))).unique()
    golden = w4.qlinear(x[rows], weight.packed.numpy(), weight.scales, group)
    for dtype, bound in ((torch.bfloat16, 4e-3), (torch.float32, 2e-6)):
        y = pkg.ops.qlinear(x.to(device), w, out_dtype=dtype)
        assert torch.equal(y, pkg.ops.qlinear(x.to(device), w, out_dtype=dtype))
        got = y.cpu()[rows].double().numpy()
        assert np.isfinite(got).all() and tuple(y.shape) == (m, n)
        error = np.linalg.norm(got - golden) / np.linalg.norm(golden)
        assert error <= bound, (dtype, error)
        assert (got[:, 3] == 0).all()


@pytest.mark.parametrize("m,n", [(70, 64), (70, 20768)])
def test_linear_keeps_a_bad_row_to_itself(pkg, device, m, n):
    """An infinity or a NaN in a row of x reaches no other row."""
    x, weight = _case(pkg, m, n, 512, 128, torch.bfloat16, seed=9)
    w = weight.to(device)
    y = pkg.ops.qlinear(x.to(device), w)
    bad = x.clone()
    bad[7, 100] = float("inf")
    bad[69, 5] = float("nan")
    z = pkg.ops.qlinear(bad.to(device), w)
    keep = torch.tensor([i for i in range(m) if i not in (7, 69)], device=device)
    assert torch.equal(y[keep], z[keep])
    assert not torch.isfinite(z[7]).any() and torch.isnan(z[69]).all()


@pytest.mark.parametrize("m,n,k", [(70, 64, 2048), (70, 20768, 1024), (640, 4352, 1536)])
@pytest.mark.parametrize("group,scale_dtype", [(128, torch.bfloat16), (256, torch.float32)])
def test_linear_scales_of_any_magnitude(pkg, device, m, n, k, group, scale_dtype):
    """Group scales far from the usual: each column to its own norm (2e-6: module docstring), zeros exactly, an infinite
    or NaN scale in its own column only.  Both forms take every one."""
    print(f"linear scales m={m} n={n} k={k} g={group} {scale_dtype}", flush=True)
    x, weight = _case(pkg, m, n, k, group, scale_dtype, seed=m)
    s = weight.scales
    groups = s.shape[1]
    for col, value in ((1, 1e-22), (2, 1e-25), (3, 0.0), (4, 1e-33), (5, 1e12), (6, 1e30), (7, -1e-22), (8, -0.01)):
        s[col] = value
    s[9, ::2], s[10, 1::2] = 1e-25, 1e-25            # small beside usual ones
    s[11, ::2], s[12, 1::2] = 0.0, 0.0
    s[13, 0], s[14, -1] = 1e25, 1e25                 # a large group first, or last
    s[15, groups // 2], s[16, groups // 2] = 1e25, 1e-25
    s[17] = torch.logspace(-20, 20, groups).to(scale_dtype)
    s[18] = torch.logspace(20, -20, groups).to(scale_dtype)
    s[20, 1], s[21, 0] = float("inf"), float("nan")
    s[n - 1] = 1e-22
    rows = torch.cat((torch.arange(36), torch.arange(m - 36, m))).unique()
    for layout in ("portable", "tiled"):
        if layout == "tiled" and (group != 128 or k not in (1024, 2048)):
            continue
        w = weight.to(device)
        y = pkg.ops.qlinear(x.to(device), w if layout == "portable" else w.tiled(), out_dtype=torch.float32)
        got = y.cpu()[rows].double().numpy()
        golden = w4.qlinear(x[rows], weight.packed.numpy(), torch.where(s.isfinite(), s, 0), group)
        finite = [c for c in range(n) if c not in (20, 21)]
        norm = np.linalg.norm(golden[:, finite], axis=0)
        error = np.linalg.norm(got[:, finite] - golden[:, finite], axis=0)
        worst = np.argmax(error - 2e-6 * norm)
        assert (error <= 2e-6 * norm).all(), (layout, finite[worst], error[worst], norm[worst])
        assert (got[:, 3] == 0).all() and not np.isfinite(got[:, 20]).any() and np.isnan(got[:, 21]).all()
