"""The FP32 networks on the MI355X: the exact split-fp16 conv / dense mode, fp32 GroupNorm,
LayerNorm and attention, and whole FP32 networks against the reference's recorded FP32
Torch-CPU outputs.

Per-op bound, the reference's own for its exact mode (tests/test_native_kernels.py:37-39,
232-236): |err| <= (8 * 2^-23 + 4 * 2^-22) * sum|terms| + 2^-23 * |expected| against
float64 (twice the magnitude where taps are summed before the split: the upsample conv,
test_native_kernels.py:271-290). Whole networks: the reference's FP32 fixture bound,
atol 2e-6 and rtol 2e-5 (tests/test_equivalence.py:62-73), against ``unet_mask`` (LMNet's
FP32 UNet with cross attention) and ``vq_float32`` (the FP32 decoder, quantized and not).
"""

from __future__ import annotations

import ctypes
import json

import numpy as np
import pytest
import torch

from oracle import attention as oatt
from oracle import conv as ocv
from oracle import fixture_weights as ofw
from oracle import norm as onm
from tests.conftest import ACCUMULATION_EPS, load_fixture

pytestmark = pytest.mark.gpu

SPLIT_ERROR = 4 * 2.0 ** -22   # tests/test_native_kernels.py:39


def fp32_case(shape, out_c, seed, k=3):
    """tests/test_native_kernels.py:238-252: channel scales over several decades put many
    lo parts near fp16's subnormal range, which the 2^11 scaling must survive."""
    rng = np.random.default_rng(seed)
    scales = np.exp(rng.normal(size=(1, shape[1], 1, 1, 1)) * 2)
    x = (rng.normal(size=shape) * scales).astype(np.float32).astype(np.float64)
    w = (rng.normal(size=(out_c, shape[1], k, k, k)) * (k ** 3 * shape[1]) ** -0.5).astype(np.float32).astype(np.float64)
    b = (rng.normal(size=(out_c,)) * 0.1).astype(np.float32).astype(np.float64)
    return x, w, b


def dev32(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).to(dev)


def ndhwc(a):
    return np.ascontiguousarray(a.transpose(0, 2, 3, 4, 1))


def host(t):
    return t.double().cpu().numpy()


def assert_near_fp32(actual, expected, magnitude, extra=0.0):
    """``extra``: a relative error of the operands beyond their split (per unit magnitude)."""
    bound = (ACCUMULATION_EPS + SPLIT_ERROR + extra) * magnitude + 2.0 ** -23 * np.abs(expected)
    err = np.abs(actual - expected)
    assert np.all(err <= bound), f"max excess {np.max(err - bound):.3e} (max err {err.max():.3e})"


@pytest.mark.parametrize(("shape", "out_c", "stride"), [
    ((1, 4, 5, 7, 9), 16, 1),     # padded input channels
    ((1, 16, 6, 5, 4), 1, 1),     # a single output channel
    ((2, 24, 7, 6, 9), 40, 2),    # stride 2, padded output channels
    ((1, 64, 4, 6, 5), 128, 1),
    ((1, 32, 16, 20, 20), 64, 1),  # streamed kernel products (2C = 64, 2O = 128)
])
def test_fp32_exact_conv_matches_float64(pkg, dev, shape, out_c, stride) -> None:
    """tests/test_native_kernels.py:255-276."""
    x, w, b = fp32_case(shape, out_c, sum(shape))
    y = pkg.ops.nax_conv3d(dev32(ndhwc(x), dev), pkg.ops.pack_weight(dev32(w, dev)), dev32(b, dev), stride=stride)
    torch.cuda.synchronize()
    assert y.dtype == torch.float32
    expected = ocv.conv3d(x, w, b, stride=stride)
    mag = ocv.conv3d_magnitude(x, w, b, stride=stride)
    assert_near_fp32(host(y).transpose(0, 4, 1, 2, 3), expected, mag)


def test_fp32_exact_conv_upsamples_with_bias_and_residual(pkg, dev) -> None:
    """tests/test_native_kernels.py:279-306: the conv of a nearest 2x upsampling with a
    per-batch bias and a residual, against float64 at twice the magnitude bound."""
    x, w, _ = fp32_case((2, 32, 3, 5, 4), 16, 23)
    rng = np.random.default_rng(23)
    bias = rng.normal(size=(2, 16)).astype(np.float32).astype(np.float64)
    res = rng.normal(size=(2, 16, 6, 10, 8)).astype(np.float32).astype(np.float64)
    y = pkg.ops.nax_conv3d(dev32(ndhwc(x), dev), pkg.ops.pack_upsample_weight(dev32(w, dev)), dev32(bias, dev),
                           upsample=True, residual=dev32(ndhwc(res), dev))
    torch.cuda.synchronize()
    up = ocv.upsample_nearest2(x)
    expected = ocv.conv3d(up, w) + bias[:, :, None, None, None] + res
    mag = ocv.conv3d_magnitude(up, w) + np.abs(bias)[:, :, None, None, None] + np.abs(res)
    assert_near_fp32(host(y).transpose(0, 4, 1, 2, 3), expected, 2 * mag)


def test_fp32_fused_prologue_shift_scale_and_concat(pkg, dev) -> None:
    """concat([x, skip]) through the fp32 GroupNorm affine + SiLU prologue, per-batch bias
    plus fp32 shift, output scale and residual."""
    x, w, _ = fp32_case((2, 48, 5, 6, 7), 32, 31)
    rng = np.random.default_rng(31)
    gamma, beta = rng.normal(size=48), rng.normal(size=48) * 0.3
    aff = onm.group_norm_affine(x, gamma, beta, groups=16, eps=1e-5).astype(np.float32).astype(np.float64)
    bias = rng.normal(size=(2, 32)).astype(np.float32).astype(np.float64)
    shift = rng.normal(size=(2, 32)).astype(np.float32).astype(np.float64)
    res = rng.normal(size=(2, 32, 5, 6, 7)).astype(np.float32).astype(np.float64)
    xd = ndhwc(x)
    y = pkg.ops.nax_conv3d(dev32(xd[..., :16], dev), pkg.ops.pack_weight(dev32(w, dev)), dev32(bias, dev),
                           x1=dev32(xd[..., 16:], dev), affine=dev32(aff, dev), silu=True, shift=dev32(shift, dev),
                           residual=dev32(ndhwc(res), dev), output_scale=0.5)
    torch.cuda.synchronize()
    prep = onm.silu(onm.apply_affine(x, aff))
    expected = ocv.conv3d(prep, w, bias + shift) * 0.5 + res
    mag = ocv.conv3d_magnitude(prep, w, bias + shift) * 0.5 + np.abs(res)
    # the prepared input is an fp32 value on the device (affine, SiLU) before its split:
    # a few more fp32 ulps per operand
    assert_near_fp32(host(y).transpose(0, 4, 1, 2, 3), expected, mag, extra=4 * 2.0 ** -23)


@pytest.mark.parametrize(("shape", "out_c"), [
    ((1, 64, 19, 32, 38), 64),    # LMNet's full-resolution grid: 128-voxel bricks, two k-groups
    ((1, 40, 16, 24, 32), 72),    # the same tiling with a partial chunk and partial row block
    ((2, 136, 3, 5, 6), 40),      # a small grid: 32-voxel bricks, four k-groups, 3 chunks
])
def test_fp32_exact_conv_tilings_with_group_norm_prologue(pkg, dev, shape, out_c) -> None:
    """The one-pass exact conv's tilings (chosen by grid size) through the fp32 GroupNorm
    affine + SiLU prologue and a residual, against float64 at the exact-mode bound."""
    x, w, b = fp32_case(shape, out_c, sum(shape) + out_c)
    rng = np.random.default_rng(out_c)
    c = shape[1]
    aff = np.stack([rng.normal(size=(shape[0], c)), rng.normal(size=(shape[0], c)) * 0.3], -1)
    aff = aff.astype(np.float32).astype(np.float64)
    res = rng.normal(size=(shape[0], out_c) + shape[2:]).astype(np.float32).astype(np.float64)
    y = pkg.ops.nax_conv3d(dev32(ndhwc(x), dev), pkg.ops.pack_weight(dev32(w, dev)), dev32(b, dev),
                           affine=dev32(aff, dev), silu=True, residual=dev32(ndhwc(res), dev))
    torch.cuda.synchronize()
    prep = onm.silu(onm.apply_affine(x, aff))
    expected = ocv.conv3d(prep, w, b) + res
    mag = ocv.conv3d_magnitude(prep, w, b) + np.abs(res)
    assert_near_fp32(host(y).transpose(0, 4, 1, 2, 3), expected, mag, extra=4 * 2.0 ** -23)


@pytest.mark.parametrize(("shape", "c0", "out_c", "up", "act"), [
    ((1, 16, 17, 33, 65), 16, 16, False, None),    # 16 rows, one chunk; partial bricks on every axis
    ((2, 16, 9, 23, 41), 16, 3, False, "silu"),    # a partial output quad
    ((1, 48, 13, 19, 61), 16, 16, False, None),    # concat: three chunks from two inputs
    ((1, 36, 13, 19, 61), 32, 32, False, "gelu"),  # a chunk of four channels
    ((1, 8, 16, 17, 57), 8, 32, False, None),      # half a chunk, 32 rows
    ((1, 20, 5, 9, 17), 20, 32, True, None),       # the upsampled grid
    ((1, 64, 16, 16, 36), 32, 96, False, None),    # three row blocks
    ((1, 96, 17, 18, 33), 48, 16, False, None),    # six chunks, 125 bricks
    ((1, 96, 16, 15, 33), 96, 32, False, None),    # 80 bricks: the 64-row tile's four k-groups
    ((1, 160, 16, 16, 60), 160, 32, False, "silu"),  # 128 bricks: the 64-row tile's two
])
def test_fp32_narrow_output_conv(pkg, dev, shape, c0, out_c, up, act) -> None:
    """The 16- and 32-row tiles, and the 64-row ones where they are faster, at the exact-mode bound,
    through the GroupNorm affine + SiLU prologue and the whole epilogue."""
    x, w, _ = fp32_case(shape, out_c, sum(shape) + out_c)
    rng = np.random.default_rng(out_c + c0)
    n, c = shape[:2]
    aff = np.stack([rng.normal(size=(n, c)), rng.normal(size=(n, c)) * 0.3], -1).astype(np.float32).astype(np.float64)
    grid = tuple(2 * v for v in shape[2:]) if up else shape[2:]
    bias, shift = (rng.normal(size=(n, out_c)).astype(np.float32).astype(np.float64) for _ in range(2))
    res = rng.normal(size=(n, out_c) + grid).astype(np.float32).astype(np.float64)
    xd = ndhwc(x)
    pack = pkg.ops.pack_upsample_weight if up else pkg.ops.pack_weight
    y = pkg.ops.nax_conv3d(dev32(xd[..., :c0], dev), pack(dev32(w, dev)), dev32(bias, dev), upsample=up,
                           x1=dev32(xd[..., c0:], dev) if c0 < c else None, affine=dev32(aff, dev), silu=True,
                           shift=dev32(shift, dev), residual=dev32(ndhwc(res), dev), output_scale=0.5, act=act)
    torch.cuda.synchronize()
    prep = onm.silu(onm.apply_affine(x, aff))
    prep = ocv.upsample_nearest2(prep) if up else prep
    expected = ocv.conv3d(prep, w, bias + shift) * 0.5 + res
    mag = ocv.conv3d_magnitude(prep, w, bias + shift) * 0.5 + np.abs(res)
    if act:   # both have slopes below 1.13; their fp32 evaluation adds a few ulps
        expected = onm.gelu(expected) if act == "gelu" else onm.silu(expected)
        mag = 1.13 * mag + 4 * np.abs(expected)
    assert_near_fp32(host(y).transpose(0, 4, 1, 2, 3), expected, mag, extra=4 * 2.0 ** -23)


def test_fp32_silu_of_extreme_values(pkg, dev) -> None:
    """silu(v) through the prologue of a 1x1x1 identity conv: from where exp(-v) underflows to
    where it overflows, as v / (1 + exp(-v)) gives it (large negative v: 0), within 4 ulps."""
    v = np.array([0.0, 1e-30, -1e-30, 0.5, -0.5, 17.25, -17.25, 87.0, -87.0, 89.5, -89.5, -104.0, 300.0, -300.0, 6e4,
                  -6e4], np.float32)
    x = torch.from_numpy(np.tile(v, (1, 1, 1, 4, 1))).to(dev)
    y = pkg.ops.nax_conv3d(x, pkg.ops.pack_weight(torch.eye(16, device=dev)), silu=True)
    with np.errstate(over="ignore"):
        want = v.astype(np.float64) / (1 + np.exp(-v.astype(np.float64)))
    # the split keeps 22 bits and is absolute below 2^-24 (fp16's subnormal step over 2^11)
    np.testing.assert_allclose(host(y)[0, 0, 0, 0], want, rtol=4 * 2.0 ** -22, atol=2.0 ** -35)


def test_fp32_silu_over_its_range(pkg, dev) -> None:
    """silu as the epilogue of a 1x1x1 identity conv, whose sums are the inputs themselves (at most 22
    significant bits), within 3 ulps (exp2 and the quotient one each, the exponent's rest a half) down to
    where 1 + exp(-v) overflows, and within the least normal value's 2^5 beyond; -inf gives NaN."""
    rng = np.random.default_rng(4)
    v = np.concatenate([np.linspace(-88.7, 88, 60000), np.linspace(-88.72, -87, 4000), rng.normal(size=4000) * 8,
                        -np.exp2(rng.uniform(-60, 6, 2000)), np.exp2(rng.uniform(-60, 15, 2000)),
                        [0.0, -88.72, -88.0, -87.4, -89.0, -104.0, -300.0, 6e4]])
    v = v[:len(v) // 32 * 32].astype(np.float32)
    v = (v.view(np.uint32) & ~np.uint32(3)).view(np.float32)   # 22 bits
    x = torch.from_numpy(v.reshape(1, 1, 1, -1, 32)).to(dev)
    y = pkg.ops.nax_conv3d(x, pkg.ops.pack_weight(torch.eye(32, device=dev)), act="silu")
    sums = host(pkg.ops.nax_conv3d(x, pkg.ops.pack_weight(torch.eye(32, device=dev)))).ravel()
    want = sums / (1 + np.exp(-sums))
    got = host(y).ravel()
    far = sums < -88.72
    np.testing.assert_allclose(got[~far], want[~far], rtol=3 * 2.0 ** -23, atol=0)
    np.testing.assert_allclose(got[far], want[far], rtol=0, atol=2.0 ** -121)


@pytest.mark.parametrize("k", [1, 3])
def test_fp32_unaligned_concat_with_batched_affine(pkg, dev, k) -> None:
    """Channel counts that are not multiples of 4 (element-wise input reads), two batch items
    with their own GroupNorm affine and bias through the pointwise (flattened) and 3x3x3
    tilings, a y slice of a wider tensor."""
    rng = np.random.default_rng(40 + k)
    x, w, _ = fp32_case((2, 19, 3, 9, 11), 37, 40 + k, k=k)
    aff = np.stack([rng.normal(size=(2, 19)), rng.normal(size=(2, 19)) * 0.3], -1).astype(np.float32)
    bias = rng.normal(size=(2, 37)).astype(np.float32).astype(np.float64)
    xd = ndhwc(x)
    out = torch.zeros((2, 3, 9, 11, 40), dtype=torch.float32, device=dev)
    pkg.ops.nax_conv3d(dev32(xd[..., :6], dev), pkg.ops.pack_weight(dev32(w, dev)), dev32(bias, dev),
                       x1=dev32(xd[..., 6:], dev), affine=dev32(aff, dev), silu=True, out=out[..., 1:38])
    torch.cuda.synchronize()
    prep = onm.silu(onm.apply_affine(x, aff.astype(np.float64)))
    expected = ocv.conv3d(prep, w, bias)
    mag = ocv.conv3d_magnitude(prep, w, bias)
    got = host(out)
    assert np.all(got[..., 0] == 0) and np.all(got[..., 38:] == 0)
    assert_near_fp32(got[..., 1:38].transpose(0, 4, 1, 2, 3), expected, mag, extra=4 * 2.0 ** -23)


@pytest.mark.parametrize("act", [None, "gelu", "silu"])
def test_fp32_dense(pkg, dev, act) -> None:
    """Dense layers in the exact mode, with the fp32 GELU / SiLU epilogue."""
    rng = np.random.default_rng(3)
    x = rng.normal(size=(1, 200, 96)).astype(np.float32).astype(np.float64)
    w = (rng.normal(size=(160, 96)) / np.sqrt(96)).astype(np.float32).astype(np.float64)
    b = (rng.normal(size=160) * 0.1).astype(np.float32).astype(np.float64)
    y = pkg.ops.dense(dev32(x, dev), pkg.ops.pack_weight(dev32(w, dev)), dev32(b, dev), act=act)
    torch.cuda.synchronize()
    pre = x @ w.T + b
    mag = np.abs(x) @ np.abs(w).T + np.abs(b)
    got = host(y)
    if act is None:
        assert_near_fp32(got, pre, mag)
    else:
        f = onm.gelu if act == "gelu" else onm.silu
        # the activation's slope is below 1.13; its fp32 evaluation adds a few ulps
        np.testing.assert_allclose(got, f(pre), rtol=4 * 2.0 ** -23, atol=1.13 * ((ACCUMULATION_EPS + SPLIT_ERROR) * mag.max() + 2.0 ** -22))


def test_fp32_group_norm_and_layer_norm(pkg, dev) -> None:
    rng = np.random.default_rng(4)
    x = (rng.normal(size=(2, 48, 5, 6, 7)) * 3 + 1).astype(np.float32).astype(np.float64)
    gamma, beta = rng.normal(size=48).astype(np.float32), rng.normal(size=48).astype(np.float32)
    xd = ndhwc(x)
    aff = host(pkg.ops.group_norm_affine(dev32(xd[..., :32], dev), dev32(gamma, dev), dev32(beta, dev), groups=16,
                                         eps=1e-5, x1=dev32(xd[..., 32:], dev)))
    want = onm.group_norm_affine(x, gamma.astype(np.float64), beta.astype(np.float64), groups=16, eps=1e-5)
    np.testing.assert_allclose(aff, want, rtol=1e-5, atol=1e-6)
    t = rng.normal(size=(300, 96)).astype(np.float32).astype(np.float64) * 2
    g, bb = rng.normal(size=96).astype(np.float32), rng.normal(size=96).astype(np.float32)
    got = host(pkg.ops.layer_norm(dev32(t, dev), dev32(g, dev), dev32(bb, dev), 1e-5))
    np.testing.assert_allclose(got, onm.layer_norm(t, g.astype(np.float64), bb.astype(np.float64), 1e-5),
                               rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize(("shape", "c1", "groups", "mean"), [
    ((1, 8, 16, 32, 1), 0, 1, 0.0),      # the smallest group of the two-launch form, unaligned rows
    ((1, 4, 9, 15, 32), 0, 32, 0.0),     # just below it
    ((2, 17, 19, 23, 48), 16, 16, 50.0), # 12 threads per voxel (four idle), a group across both inputs
    ((1, 16, 17, 19, 1024), 0, 32, 0.0), # one voxel slot per workgroup
    ((1, 11, 13, 40, 6), 3, 3, -3.0),    # unaligned concat: one channel per thread
    ((3, 21, 22, 23, 16), 0, 16, 1e3),   # one channel per group, mean >> deviation
])
def test_fp32_group_norm_of_large_tensors(pkg, dev, shape, c1, groups, mean) -> None:
    """Bound: the offset beta - scale * mean carries scale * mean's rounding, so the absolute
    part grows with |mean| / deviation (2^-20 of it: the mean's and the scale's few ulps)."""
    rng = np.random.default_rng(6)
    x = (rng.normal(size=shape) * 2 + mean).astype(np.float32)
    c = shape[-1]
    gamma, beta = rng.normal(size=c).astype(np.float32), rng.normal(size=c).astype(np.float32)
    x0, x1 = dev32(x[..., :c - c1], dev), dev32(x[..., c - c1:], dev) if c1 else None
    aff = host(pkg.ops.group_norm_affine(x0, dev32(gamma, dev), dev32(beta, dev), groups=groups, eps=1e-5, x1=x1))
    want = onm.group_norm_affine(x.astype(np.float64).transpose(0, 4, 1, 2, 3), gamma.astype(np.float64),
                                 beta.astype(np.float64), groups=groups, eps=1e-5)
    np.testing.assert_allclose(aff, want, rtol=2e-6, atol=2e-6 + 2.0 ** -20 * abs(mean))


@pytest.mark.parametrize(("shape", "c1"), [((1, 8, 16, 33, 16), 0), ((2, 17, 19, 23, 48), 16), ((1, 4, 9, 13, 6), 0),
                                           ((1, 11, 13, 40, 6), 3)])
@pytest.mark.parametrize("mean", [1e20, -3e37, 1e38])
def test_fp32_group_norm_of_huge_values(pkg, dev, shape, c1, mean) -> None:
    """Values whose squares overflow, with deviations whose squares do not: statistics as small
    tensors' (one launch) have them, finite and within 2^-20 of the values. (Scale: 1 / deviation.)"""
    rng = np.random.default_rng(8)
    dev_ = 1e16
    x = (mean + rng.normal(size=shape) * dev_).astype(np.float32)
    c, groups = shape[-1], 2
    x0, x1 = dev32(x[..., :c - c1], dev), dev32(x[..., c - c1:], dev) if c1 else None
    gamma = dev32(np.full(c, 1e-3), dev)
    aff = host(pkg.ops.group_norm_affine(x0, gamma, dev32(np.zeros(c), dev), groups=groups, eps=1e-5, x1=x1))
    g64 = x.astype(np.float64).reshape(shape[0], -1, groups, c // groups)
    std, mu = (np.repeat(f(g64, axis=(1, 3)), c // groups, axis=1) for f in (np.std, np.mean))
    if dev_ > 2 ** -20 * abs(mean):   # the deviations are more than the values' rounding
        np.testing.assert_allclose(aff[..., 0], 1e-3 / std, rtol=1e-4)
    np.testing.assert_allclose(-aff[..., 1] / aff[..., 0], mu, rtol=2.0 ** -20)


@pytest.mark.parametrize("batch", [2, 5])
def test_fp32_group_norm_of_an_item_does_not_depend_on_its_batch(pkg, dev, batch) -> None:
    """Each item's statistics in the two-launch form: the bits of that item alone."""
    rng = np.random.default_rng(batch)
    x = dev32(rng.normal(size=(batch, 64, 66, 67, 16)), dev)
    gamma, beta = (dev32(rng.normal(size=16), dev) for _ in range(2))
    aff = pkg.ops.group_norm_affine(x, gamma, beta, groups=8, eps=1e-5)
    for b in range(batch):
        assert torch.equal(aff[b:b + 1], pkg.ops.group_norm_affine(x[b:b + 1], gamma, beta, groups=8, eps=1e-5))


@pytest.mark.parametrize(("lq", "lk", "d"), [(64, 3, 16), (300, 300, 32), (129, 77, 64), (8, 8, 16)])
def test_fp32_attention_matches_float64(pkg, dev, lq, lk, d) -> None:
    rng = np.random.default_rng(lq + lk + d)
    q, k, v = (rng.normal(size=(2, 3, n, d)).astype(np.float32).astype(np.float64) for n in (lq, lk, lk))
    o = pkg.ops.attention(dev32(q, dev), dev32(k, dev), dev32(v, dev), d ** -0.5)
    torch.cuda.synchronize()
    assert o.dtype == torch.float32
    np.testing.assert_allclose(host(o), oatt.attention(q, k, v, d ** -0.5), rtol=2e-5, atol=2e-6)


@pytest.mark.parametrize(("batch", "length", "keys", "heads"), [(1, 96, 64, 2), (2, 32, 160, 1), (1, 1056, 96, 2)])
def test_fp32_attention_reference_cases(pkg, dev, batch, length, keys, heads) -> None:
    """The reference's FP32 flash-attention cases (tests/test_native_kernels.py:395-458:
    32-wide heads, q and k scaled by 2 for peaked rows that move the running maximum) at
    its FP32 bound, atol 2e-5 -- here on the split-fp16 MFMA kernel."""
    rng = np.random.default_rng(length + keys)
    q, k, v = ((rng.normal(size=(batch, heads, n, 32)) * sc).astype(np.float32).astype(np.float64)
               for n, sc in ((length, 2.0), (keys, 2.0), (keys, 1.0)))
    o = pkg.ops.attention(dev32(q, dev), dev32(k, dev), dev32(v, dev), 32 ** -0.5)
    torch.cuda.synchronize()
    got = host(o)
    assert np.all(np.isfinite(got))
    np.testing.assert_allclose(got, oatt.attention(q, k, v, 32 ** -0.5), rtol=0, atol=2e-5)


def test_fp32_attention_lmnet_length(pkg, dev) -> None:
    """LMNet's 23,104-token FP32 self-attention (two 32-wide heads; mlx_model.py:74-76,
    _attention.py:27-28) on the split-fp16 MFMA kernel, every 97th query row against float64
    at the reference's FP32 bound (atol 2e-5)."""
    n, heads = 23104, 2
    rng = np.random.default_rng(23104)
    q, k, v = ((rng.normal(size=(1, heads, n, 32)) * sc).astype(np.float32) for sc in (2.0, 2.0, 1.0))
    print(f"fp32 attention {n} tokens x {heads} heads", flush=True)
    o = pkg.ops.attention(dev32(q, dev), dev32(k, dev), dev32(v, dev), 32 ** -0.5)
    torch.cuda.synchronize()
    rows = np.arange(0, n, 97)
    got = host(o)[:, :, rows]
    want = oatt.attention(q[:, :, rows].astype(np.float64), k.astype(np.float64), v.astype(np.float64), 32 ** -0.5)
    np.testing.assert_allclose(got, want, rtol=0, atol=2e-5)


@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize(("batch", "heads", "lq", "lk"), [
    (1, 1, 1, 609),       # one query, a last block of one key, as many key ranges as it takes
    (2, 2, 129, 640),     # a query tile of one row, whole key blocks
    (1, 3, 128, 1311),    # ranges of unequal length
    (1, 1, 40000, 615),   # enough query tiles for one range: no merge
])
def test_fp32_attention_key_ranges(pkg, dev, d, batch, heads, lq, lk) -> None:
    """The three-launch form (at least 20 key blocks) on head-interleaved views of one fused
    projection, with scores that rise along the keys (the exponent base moves in every range)
    and one query whose scores lie 80 below the others', against float64; also without the
    workspace (the one-launch kernel), through the C ABI."""
    rng = np.random.default_rng(lq + lk + d)
    f = heads * d
    q = rng.normal(size=(batch, lq, f)).astype(np.float32)
    kv = rng.normal(size=(batch, lk, 2 * f)).astype(np.float32)
    kv[..., :f] *= np.linspace(0.2, 4, lk, dtype=np.float32)[None, :, None]
    q[:, 0] *= 8
    qd, kvd = dev32(q, dev), dev32(kv, dev)
    o = pkg.ops.flash_attention(qd, kvd[..., :f], kvd[..., f:], heads=heads, scale=d ** -0.5)
    o2 = torch.empty_like(o)
    a = pkg.ops._attn_args(qd.unflatten(2, (heads, d)), kvd[..., :f].unflatten(2, (heads, d)),
                           kvd[..., f:].unflatten(2, (heads, d)), o2.unflatten(2, (heads, d)), d ** -0.5, None)
    assert a.workspace_bytes > 0
    a.workspace, a.workspace_bytes = None, 0
    assert pkg._lib.lib.ldx_attention(ctypes.byref(a), torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    rows = np.unique(np.concatenate([[0], rng.integers(0, lq, 64), [lq - 1]]))
    split = lambda t: t.astype(np.float64).reshape(batch, -1, heads, d).transpose(0, 2, 1, 3)  # noqa: E731
    want = oatt.attention(split(q[:, rows]), split(kv[..., :f]), split(kv[..., f:]), d ** -0.5)
    for got in (o, o2):
        np.testing.assert_allclose(split(host(got[:, rows])), want, rtol=0, atol=2e-5)


@pytest.mark.parametrize("d", [32, 64])
def test_fp32_attention_of_many_small_probabilities(pkg, dev, d) -> None:
    """Every 64th key's score is 11 to 18 (log2 units) above those of the others, which are equal and
    alone have values: the output is the sum of their small probabilities, in which equal rounding
    errors add. Bound: a probability keeps 2^-22 of itself (hi / lo), the rounding of its exponent
    (2^-23 of 18) and exp2 2^-20.4, the sums of 47 blocks 2^-19 in the worst order: 4e-6 of the value."""
    lk, lq = 1504, 256
    gaps = np.linspace(11, 18, lq)
    q = np.zeros((1, lq, d), np.float32)
    q[..., 0] = gaps / 1.44269504088896341
    k, v = np.zeros((1, lk, d), np.float32), np.ones((1, lk, d), np.float32)
    k[0, 5::64, 0], v[0, 5::64] = 1, 0
    high = len(range(5, lk, 64))
    got = host(pkg.ops.flash_attention(dev32(q, dev), dev32(k, dev), dev32(v, dev), heads=1, scale=1.0))
    p = np.exp2(-q[0, :, 0].astype(np.float64) * np.log2(np.e))
    want = ((lk - high) * p / (high + (lk - high) * p))[None, :, None]
    np.testing.assert_allclose(got, np.broadcast_to(want, got.shape), rtol=4e-6, atol=0)


@pytest.mark.parametrize("d", [32, 64])
def test_fp32_attention_split_kernel_agrees_with_the_valu_kernel(pkg, dev, monkeypatch, d) -> None:
    """The split-fp16 MFMA kernel and the FP32 VALU flash kernel (LDX_ATTN_F32=valu) on the
    same ragged inputs: both within FP32 error of each other."""
    rng = np.random.default_rng(d)
    q, k, v = (rng.normal(size=(2, 3, n, d)).astype(np.float32) for n in (257, 333, 333))
    args = [dev32(t, dev) for t in (q, k, v)]
    mfma = host(pkg.ops.attention(*args, d ** -0.5))
    monkeypatch.setenv("LDX_ATTN_F32", "valu")
    valu = host(pkg.ops.attention(*args, d ** -0.5))
    torch.cuda.synchronize()
    np.testing.assert_allclose(mfma, valu, rtol=2e-5, atol=2e-6)


def test_fp32_unet_matches_recorded_torch(pkg, dev) -> None:
    """LMNet's FP32 network (the ``unet_mask`` recording: cross attention to a context, 16-wide
    heads) at the reference's FP32 bound, atol 2e-6, rtol 2e-5."""
    z = load_fixture("unet_mask")
    assert z["dtype"].item() == "float32"
    c = json.loads(z["config"].item())
    cfg = pkg.unet.UnetConfig(c["model_channels"], c["num_res_blocks"], tuple(c["attention_resolutions"]),
                              tuple(c["channel_mult"]), c["num_head_channels"], c["skip_context"])
    w = ofw.unet_fixture_weights(int(z["weight_seed"]), skip_context=cfg.skip_context)
    net = pkg.unet.LdmUnet(w, cfg, dtype=torch.float32)
    out = net(dev32(z["x"], dev), torch.from_numpy(z["timesteps"]).to(dev), dev32(z["context"], dev))
    torch.cuda.synchronize()
    got, rec = host(out), z["output"].astype(np.float64)
    print(f"unet_mask fp32: max abs {np.abs(got - rec).max():.3e}")
    np.testing.assert_allclose(got, rec, atol=2e-6, rtol=2e-5)


def test_fp32_vq_decoder_matches_recorded_torch(pkg, dev) -> None:
    """The FP32 VQ decoder: decode(z) (fp32 quantization, then the decoder) and the
    unquantized decode against the ``vq_float32`` recording at atol 2e-6, rtol 2e-5."""
    z = load_fixture("vq_float32")
    dec = pkg.vq.VqDecoder(ofw.vq_fixture_weights(int(z["weight_seed"])), dtype=torch.float32)
    zt = dev32(z["z"], dev)
    for key, quantize in (("decoded_unquantized", False), ("decoded", True)):
        got = host(dec(zt, quantize=quantize))
        rec = z[key].astype(np.float64)
        print(f"vq fp32 {key}: max abs {np.abs(got - rec).max():.3e}")
        np.testing.assert_allclose(got, rec, atol=2e-6, rtol=2e-5)
