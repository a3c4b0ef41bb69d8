"""Differentiable FP32 SGM on the GPU against the FP64 CPU reference
(oracle/dsgm_oracle.cpp, itself pinned by finite differences in
tests/test_dsgm_oracle.py).  Tolerances: disparity and S within 1e-5
relative, gradients within 1e-4 relative (norm-wise and element-wise against
the largest entry)."""
import numpy as np
import pytest
import torch

import oracle
from fasterstereocuda_amd.diff_sgm import census_cost_volume, diff_sgm

pytestmark = pytest.mark.gpu

T = 0.1


def _inputs(B, H, W, D, seed):
    rng = np.random.default_rng(seed)
    cost = rng.random((B, H, W, D)).astype(np.float32)
    p1 = rng.uniform(0.05, 0.2, (B, H, W)).astype(np.float32)
    p2 = rng.uniform(0.5, 2.0, (B, H, W)).astype(np.float32)
    gt = rng.uniform(0, D - 1, (B, H, W)).astype(np.float32)
    return cost, p1, p2, gt


def _rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


# even and odd widths and heights, lines of fewer steps than the load
# pipeline's depth (rows of 1, 2 and 3 pixels), and D = 64, 128, 256
@pytest.mark.parametrize("B,H,W,D", [(2, 33, 40, 64), (1, 32, 97, 128), (1, 20, 64, 256),
                                     (2, 45, 70, 128), (1, 7, 1, 64), (2, 5, 2, 64),
                                     (1, 9, 3, 128)])
def test_forward_backward_match_fp64(cuda, B, H, W, D):
    print(f"[dsgm] B{B} H{H} W{W} D{D}", flush=True)
    cost, p1, p2, gt = _inputs(B, H, W, D, seed=H + W + D)
    tc = torch.from_numpy(cost).to(cuda).requires_grad_(True)
    t1 = torch.from_numpy(p1).to(cuda).requires_grad_(True)
    t2 = torch.from_numpy(p2).to(cuda).requires_grad_(True)
    tg = torch.from_numpy(gt).to(cuda)
    disp = diff_sgm(tc, t1, t2, T)
    loss = (disp - tg).abs().mean(dim=(1, 2)).sum()     # per-image mean L1
    loss.backward()
    for b in range(B):
        S, d_ref, l_ref = oracle.dsgm_forward(cost[b], p1[b], p2[b], gt[b], T)
        gC, g1, g2, _ = oracle.dsgm_backward(cost[b], p1[b], p2[b], gt[b], T)
        d = disp[b].detach().cpu().numpy()
        assert np.abs(d - d_ref).max() <= 1e-5 * max(1.0, np.abs(d_ref).max()), "disparity"
        for name, got, ref in (("dC", tc.grad[b], gC), ("dP1", t1.grad[b], g1), ("dP2", t2.grad[b], g2)):
            g = got.cpu().numpy().astype(np.float64)
            assert _rel(g, ref) <= 1e-4, f"{name} rel err {_rel(g, ref):.2e}"
            assert np.abs(g - ref).max() <= 1e-4 * np.abs(ref).max(), f"{name} max err"


# both directions of a row pair at once: widths 4 .. 9 around the load ring and
# the middle pixel (odd widths), one row, an odd last row
@pytest.mark.parametrize("B,H,W,D", [(1, 1, 1, 64), (1, 1, 4, 128), (2, 2, 5, 64), (1, 3, 6, 256), (1, 5, 7, 128),
                                     (1, 2, 8, 64), (3, 3, 9, 128), (1, 6, 16, 256), (1, 4, 17, 64)])
def test_row_pairs_match_fp64(cuda, B, H, W, D):
    test_forward_backward_match_fp64(cuda, B, H, W, D)


# many images of few rows, which take the form that walks bands of four rows
# for two directions together: last bands of 1 to 4 rows, a single band (no
# state handed between bands), lines shorter than the skew of a band's rows
@pytest.mark.parametrize("B,H,W,D", [(141, 13, 70, 128), (188, 10, 33, 64), (560, 3, 9, 64),
                                     (140, 16, 1, 128), (280, 7, 2, 64), (187, 12, 130, 128),
                                     (98, 13, 20, 256)]
                         # too many waves for one launch of all directions, too few
                         # bands for the above: one pass per direction and set
                         + [(12, 97, 71, 64), (12, 83, 90, 128), (200, 7, 5, 64),
                            (180, 5, 9, 128), (90, 3, 7, 256), (240, 1, 8, 64), (120, 17, 1, 128)])
def test_many_images_match_fp64(cuda, B, H, W, D):
    print(f"[dsgm] B{B} H{H} W{W} D{D}", flush=True)
    cost, p1, p2, gt = _inputs(B, H, W, D, seed=B + H + W + D)
    tc = torch.from_numpy(cost).to(cuda).requires_grad_(True)
    t1 = torch.from_numpy(p1).to(cuda).requires_grad_(True)
    t2 = torch.from_numpy(p2).to(cuda).requires_grad_(True)
    disp = diff_sgm(tc, t1, t2, T)
    (disp - torch.from_numpy(gt).to(cuda)).abs().mean(dim=(1, 2)).sum().backward()
    for b in (0, 1, B // 2, B - 1):
        _, d_ref, _ = oracle.dsgm_forward(cost[b], p1[b], p2[b], gt[b], T)
        gC, g1, g2, _ = oracle.dsgm_backward(cost[b], p1[b], p2[b], gt[b], T)
        d = disp[b].detach().cpu().numpy()
        assert np.abs(d - d_ref).max() <= 1e-5 * max(1.0, np.abs(d_ref).max()), "disparity"
        for name, got, ref in (("dC", tc.grad[b], gC), ("dP1", t1.grad[b], g1), ("dP2", t2.grad[b], g2)):
            g = got.cpu().numpy().astype(np.float64)
            assert _rel(g, ref) <= 1e-4, f"{name} rel err {_rel(g, ref):.2e}"
            assert np.abs(g - ref).max() <= 1e-4 * np.abs(ref).max(), f"{name} max err"


# the bands' form where it is taken: narrow images (last bands of 1 to 4 rows),
# and wide ones from the number of cells on that it needs
@pytest.mark.parametrize("B,H,W,D", [(41, 41, 16, 64), (41, 42, 5, 64), (41, 43, 2, 64), (45, 40, 1, 64),
                                     (36, 41, 1, 128), (36, 42, 13, 128), (36, 44, 3, 128), (36, 43, 4, 256),
                                     (36, 41, 9, 256), (130, 13, 112, 128), (98, 14, 70, 256), (90, 18, 271, 64)])
def test_bands_match_fp64(cuda, B, H, W, D):
    test_many_images_match_fp64(cuda, B, H, W, D)


# Rows whose pairs pass 2^32 bytes: the separate passes' 64-bit offsets.  A stretch
# of columns is cut off by penalties P2 < 0 on both sides of its ends: the last term
# then wins everywhere, L = C + P2, and nothing is handed across.  So the stretch
# equals its own columns alone, up to a constant in S at its ends (and the penalty
# gradients there).  Costs and penalties are multiples of 1/64, so L and S are exact
# and the disparities equal; a gradient is a sum of the same four terms in another
# order, within 4 roundings of terms not much above the largest.
def test_very_long_rows(cuda):
    H, W, D, n = 2, 3000001, 256, 64
    print(f"[dsgm long rows] {W}x{H} D{D}", flush=True)
    g = torch.Generator(device=cuda).manual_seed(5)

    def ints(lo, hi, *shape):
        return torch.randint(lo, hi, shape, dtype=torch.uint8, device=cuda, generator=g).to(torch.float32).div_(64)

    cost = ints(0, 64, 1, H, W, D).requires_grad_(True)
    p1, p2, gd = ints(4, 16, 1, H, W), ints(32, 128, 1, H, W), ints(0, 64, 1, H, W) - 0.5
    starts = [0, W // 4, W // 2, W - n - 1234567 // 2, W - n]
    for a in starts:
        for x in (a - 1, a, a + n - 1, a + n):
            if 0 <= x < W:
                p2[:, :, x] = -1 / 64
    p1.requires_grad_(True)
    p2.requires_grad_(True)
    disp = diff_sgm(cost, p1, p2, T)
    disp.backward(gd)
    for a in starts:
        cut = slice(a, a + n)
        args = [x.detach()[:, :, cut].contiguous().requires_grad_(True) for x in (cost, p1, p2)]
        part = diff_sgm(*args, T)
        part.backward(gd[:, :, cut].contiguous())
        np.testing.assert_array_equal(disp.detach()[:, :, cut].cpu().numpy(), part.detach().cpu().numpy(),
                                      err_msg=f"disparity from column {a}")
        for name, x, y in zip(("dC", "dP1", "dP2"), (cost, p1, p2), args):
            got, ref = x.grad[:, :, cut].cpu().numpy(), y.grad.cpu().numpy()
            if name != "dC":
                got, ref = got[:, :, 1:-1], ref[:, :, 1:-1]
            assert np.abs(ref).max() > 0 and np.abs(got - ref).max() <= 1e-5 * np.abs(ref).max(), f"{name} from {a}"


def test_deterministic_and_repeatable(cuda):
    cost, p1, p2, gt = _inputs(2, 40, 50, 64, seed=1)
    outs = []
    for _ in range(2):
        tc = torch.from_numpy(cost).to(cuda).requires_grad_(True)
        t1 = torch.from_numpy(p1).to(cuda).requires_grad_(True)
        t2 = torch.from_numpy(p2).to(cuda).requires_grad_(True)
        disp = diff_sgm(tc, t1, t2, T)
        (disp - torch.from_numpy(gt).to(cuda)).abs().mean().backward()
        outs.append([x.detach().cpu().numpy() for x in (disp, tc.grad, t1.grad, t2.grad)])
    for a, b in zip(*outs):
        np.testing.assert_array_equal(a.view(np.uint32), b.view(np.uint32))


def test_census_cost_volume(cuda):
    rng = np.random.default_rng(0)
    left = rng.integers(0, 256, (2, 30, 80), dtype=np.uint8)
    right = rng.integers(0, 256, (2, 30, 80), dtype=np.uint8)
    c = census_cost_volume(torch.from_numpy(left).to(cuda), torch.from_numpy(right).to(cuda), 64)
    for b in range(2):
        cl = oracle.census(left[b], 1, False)
        cr = oracle.census(right[b], 1, True)
        ref = oracle.cost(cl, cr, 0, 64, True, 1).astype(np.float32) / np.float32(63.0)
        np.testing.assert_array_equal(c[b].cpu().numpy(), ref)


def test_bad_shapes_raise(cuda):
    x = torch.zeros((1, 4, 4, 96), device=cuda)
    p = torch.zeros((1, 4, 4), device=cuda)
    with pytest.raises(ValueError):
        diff_sgm(x, p, p)
