"""The fused Q/K/V convolution kernels on the GPU against the CPU oracle.

Bars: FP32 inputs <= 1e-5 relative L2 against the FP32 oracle; BF16 inputs
<= 2e-2 against the FP32 oracle on the same BF16-rounded inputs.  Outputs
q, k, v and gradients dx, dw.  Includes the reference's screen geometry
(8 rows x 4,096 tokens, 8 heads of 128, conv_size 4) at full size.
"""

from __future__ import annotations

import pytest
import torch

from conftest import rel_l2
from oracle import qkv_conv_oracle as co

pytestmark = pytest.mark.gpu

FP32_TOL = 1e-5
BF16_TOL = 2e-2
EPS = 1e-6


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("needs a HIP device")
    from delta_feedback_experiment_amd import _lib

    _lib.lib()
    return torch.device("cuda:0")


def make(B, T, H, d, W, dtype, w_dtype=torch.float32, seed=0):
    gen = torch.Generator().manual_seed(seed)
    x = torch.randn(B, T, 3 * H * d, generator=gen).to(dtype)
    w = (0.5 * torch.randn(3 * H * d, W, generator=gen)).to(w_dtype)
    do = [torch.randn(B, T, H * d, generator=gen).to(dtype) for _ in range(3)]
    return x, w, do


def run_case(dev, B, T, H, d, W, dtype, w_dtype=torch.float32, seed=0):
    from delta_feedback_experiment_amd import pkda_qkv_conv

    x, w, do = make(B, T, H, d, W, dtype, w_dtype, seed)
    P = H * d
    xl = x.float().requires_grad_()
    wl = w.float().requires_grad_()
    ref = co.qkv_conv_reference(xl, wl, d, 2 * P, EPS, out_dtype=torch.float32)
    gref = torch.autograd.grad(ref, (xl, wl), [t.float() for t in do])
    xd, wd = x.to(dev).requires_grad_(), w.to(dev).requires_grad_()
    out = pkda_qkv_conv(xd, wd, d, 2 * P, EPS)
    got = torch.autograd.grad(out, (xd, wd), [t.to(dev) for t in do])
    torch.cuda.synchronize()
    errs = {n: rel_l2(a.float(), b) for n, a, b in zip(("q", "k", "v"), out, ref)}
    errs["dx"] = rel_l2(got[0].float(), gref[0])
    errs["dw"] = rel_l2(got[1].float(), gref[1])
    assert out[0].dtype == dtype and got[0].dtype == dtype and got[1].dtype == w_dtype
    return errs


@pytest.mark.parametrize("W", [1, 2, 3, 4])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_conv_matches_oracle(dev, W, d, dtype):
    print(f"[gpu] qkv conv W={W} d={d} {dtype}", flush=True)
    errs = run_case(dev, 2, 100, 3, d, W, dtype, seed=W + d)  # 100 = one full tile + a partial one
    print("  " + " ".join(f"{n}={e:.2e}" for n, e in errs.items()), flush=True)
    tol = FP32_TOL if dtype == torch.float32 else BF16_TOL
    assert all(e < tol for e in errs.values()), errs


@pytest.mark.parametrize("T", [1, 2, 3, 64, 65])
def test_conv_short_and_boundary_lengths(dev, T):
    print(f"[gpu] qkv conv T={T}", flush=True)
    errs = run_case(dev, 3, T, 2, 32, 4, torch.float32, seed=T)
    assert all(e < FP32_TOL for e in errs.values()), errs


def test_conv_bf16_weights(dev):
    print("[gpu] qkv conv bf16 weights", flush=True)
    errs = run_case(dev, 2, 70, 2, 64, 4, torch.bfloat16, w_dtype=torch.bfloat16, seed=9)
    assert all(e < BF16_TOL for e in errs.values()), errs


def test_conv_backward_is_deterministic(dev):
    from delta_feedback_experiment_amd.conv import pkda_qkv_conv_backward

    x, w, do = make(4, 300, 4, 64, 4, torch.bfloat16, seed=11)
    args = [t.to(dev) for t in (x, w, *do)]
    a = pkda_qkv_conv_backward(*args, 64, 2 * 256, EPS)
    b = pkda_qkv_conv_backward(*args, 64, 2 * 256, EPS)
    torch.cuda.synchronize()
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


def test_conv_screen_geometry_full_size(dev):
    """8 rows x 4,096 tokens, 8 heads of 128 (projection width 1,024), 4 taps."""
    print("[gpu] qkv conv screen geometry B8 T4096 P1024", flush=True)
    errs = run_case(dev, 8, 4096, 8, 128, 4, torch.bfloat16, seed=21)
    print("  " + " ".join(f"{n}={e:.2e}" for n, e in errs.items()), flush=True)
    assert all(e < BF16_TOL for e in errs.values()), errs


@pytest.mark.parametrize("B,T,H,d,W", [
    (1, 1, 1, 32, 1),     # 96 columns of one partial
    (37, 2, 1, 32, 3),    # 288 columns, 37 partials: more than a workgroup has slots, fewer than classes
    (3, 65, 6, 128, 1),   # 2,304 columns, 6 partials
    (300, 1, 8, 128, 4),  # 12,288 columns, 300 partials
])
def test_conv_weight_gradient_sums(dev, B, T, H, d, W):
    """dw's partials over every width of the column sums, fewer and more of
    them than a column has classes; FP32, so the FP32 bar holds the sums."""
    print(f"[gpu] qkv conv dw sums B={B} T={T} H={H} d={d} W={W}", flush=True)
    errs = run_case(dev, B, T, H, d, W, torch.float32, seed=B + W)
    assert all(e < FP32_TOL for e in errs.values()), errs


@pytest.mark.parametrize("B,T,H,d", [
    (22, 1001, 8, 128),  # tiles of 32 and 64 tokens, a last tile of 9 and 41
    (11, 1003, 8, 128),  # 32 and 32
    (6, 998, 8, 128),    # 16 and 16: groups of four and a pair
    (3, 33, 2, 64),      # 8 and 16: a last tile of one token
])
def test_conv_tiles_match_oracle(dev, B, T, H, d):
    """Every tile length the sizes choose, forward and backward, with a last
    tile and a last group that are not whole; FP32 at the FP32 bar (the dw
    sums of both sides are FP32 over B T tokens)."""
    from delta_feedback_experiment_amd import pkda_qkv_conv

    print(f"[gpu] qkv conv tiles B={B} T={T} H={H} d={d}", flush=True)
    x, w, do = (t.to(dev) if torch.is_tensor(t) else [g.to(dev) for g in t]
                for t in make(B, T, H, d, 4, torch.float32, seed=T))
    leaves = [x.requires_grad_(), w.requires_grad_()]
    ref = co.qkv_conv_reference(*leaves, d, 2 * H * d, EPS)
    out = pkda_qkv_conv(*leaves, d, 2 * H * d, EPS)
    grads = zip(torch.autograd.grad(out, leaves, do), torch.autograd.grad(ref, leaves, do))
    for name, (a, b) in zip(("q", "k", "v", "dx", "dw"), list(zip(out, ref)) + list(grads)):
        assert rel_l2(a, b) < FP32_TOL, name


def test_conv_keeps_infinities_and_nan(dev):
    """The sigmoid's reciprocal keeps a division's results at the ends: silu
    of a large negative input is zero, of infinities and NaN what torch's
    a / (1 + e^-a) gives."""
    from delta_feedback_experiment_amd import pkda_norm_gate, pkda_qkv_conv

    print("[gpu] sigmoid ends", flush=True)
    vals = torch.tensor([0.0, -80.0, -88.9, -200.0, 200.0, 3e38, -3e38, float("inf"), float("-inf"), float("nan")],
                        device=dev)
    x = torch.zeros(1, 1, 3 * 32, device=dev)
    x[0, 0, 64:64 + len(vals)] = vals  # the V slab: no norm
    v = pkda_qkv_conv(x, torch.ones(96, 1, device=dev), 32, 64, EPS)[2][0, 0, :len(vals)]
    torch.testing.assert_close(v, vals / (1 + torch.exp(-vals)), rtol=1e-5, atol=1e-30, equal_nan=True)
    gate = torch.zeros(1, 64, device=dev)
    gate[0, :len(vals)] = vals
    y = pkda_norm_gate(torch.ones(1, 64, device=dev), gate, torch.ones(64, device=dev), 0.0)[0]
    torch.testing.assert_close(y, torch.sigmoid(gate), rtol=1e-5, atol=1e-30, equal_nan=True)


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("B,T", [(2500, 1), (64, 39)])
def test_conv_norm_sum_order(dev, d, B, T):
    """The L2 norm's sum of squares: chains of eight channels (the second
    square rounded by itself, the others fused onto it in turn) that add in
    pairs, whatever number of channels a lane holds; the token kernel's too.
    From the same channels without the norm, and a correctly rounded inverse
    root, Q and K follow bit for bit in the rows where the hardware's root is
    the correctly rounded one: 89 % of them, as against 77 to 81 % with a sum
    of chains of four, which is an ulp off in many rows.  (The fused sums are
    taken in FP64, whose own rounding moves an FP32 result with a chance of
    2^-29.)"""
    from delta_feedback_experiment_amd import pkda_qkv_conv, pkda_qkv_conv_cached_

    print(f"[gpu] qkv conv norm sum order d={d} B={B} T={T}", flush=True)
    H = 3
    x, w, _ = make(B, T, H, d, 4, torch.float32, seed=d)
    x, w = x.to(dev), w.to(dev)
    plain = pkda_qkv_conv(x, w, d, 0, EPS)
    got = pkda_qkv_conv(x, w, d, 2 * H * d, EPS)
    for y, n in list(zip(plain, got))[:2]:
        y, n = y.reshape(B, T, H, d), n.reshape(B, T, H, d)
        c = y.reshape(B, T, H, d // 8, 8)
        ss = c[..., 1] * c[..., 1]
        for j in (0, 2, 3, 4, 5, 6, 7):
            ss = (c[..., j].double().square() + ss.double()).float()
        while ss.shape[-1] > 1:
            ss = ss[..., 0::2] + ss[..., 1::2]
        r = (ss + EPS).double().rsqrt().float()
        assert (n == y * r).all(-1).float().mean() > 0.85
    if T == 1:
        pool = torch.zeros(B, 3, 3 * H * d, device=dev)
        cached = pkda_qkv_conv_cached_(x, w, d, 2 * H * d, EPS, pool, continue_state=True)
        for a, b in zip(cached, got):
            assert torch.equal(a, b)
