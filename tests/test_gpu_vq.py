"""The nearest-codebook search on the MI355X (ldx_vq_nearest4, ldx_vq_squared_norms4) against
the oracle, bit for bit: indices, norms and straight-through values are integer or
exactly-rounded results, so nothing but equality is accepted. Cases restate the reference's
own tests (tests/test_vq_optimized.py:27-94): strided batches of a 2,048-entry codebook,
first-index ties at midpoints and duplicate entries, NaN distances from fp16 norm overflow,
and a one-entry codebook; plus a config-sized search (51,200 latent vectors x 8,192 codes)
checked on sampled rows."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import vq as ovq

pytestmark = pytest.mark.gpu

DTYPES = {"float16": (torch.float16, np.float16), "float32": (torch.float32, np.float32)}


def _bits(a: np.ndarray) -> np.ndarray:
    return a.view(np.uint16 if a.dtype == np.float16 else np.uint32)


def _search(pkg, dev, flat: np.ndarray, codebook: np.ndarray, tt):
    z = torch.from_numpy(flat).to(dev).to(tt).contiguous()
    cb = torch.from_numpy(codebook).to(dev).to(tt).contiguous()
    norms = pkg.ops.squared_norms4(cb)
    q = torch.empty_like(z)
    idx = pkg.ops.nearest_codebook4(z, cb, norms, quantized=q)
    torch.cuda.synchronize()
    return idx.cpu().numpy(), q.cpu().numpy(), norms.cpu().numpy()


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize(("positions", "entries"), [(1, 2048), (2, 33), (3, 1), (31, 2), (32, 32), (33, 31)])
def test_nearest_codebook_first_index_at_ties(pkg, dev, dtype, positions, entries) -> None:
    """Duplicate entries, midpoints between neighbours and the entries themselves (and a
    zero vector) as latents: the indices, norms and straight-through values equal the
    oracle's bit for bit (tests/test_vq_optimized.py:54-94)."""
    tt, nt = DTYPES[dtype]
    rng = np.random.default_rng(317)
    cb = rng.normal(size=(entries, 4)).astype(np.float32)
    if entries > 3:
        cb[-1] = cb[0]
        cb[3] = -cb[2]
    pts = np.concatenate([(cb[:-1] + cb[1:]) / 2, cb, np.zeros((1, 4))]).astype(np.float32)
    pts = np.tile(pts, (positions // len(pts) + 1, 1))[:positions]
    cbt, ptt = cb.astype(nt), pts.astype(nt)
    idx, q, norms = _search(pkg, dev, ptt, cbt, tt)
    want_idx, want_q = ovq.quantize4(ptt, cbt, nt)
    np.testing.assert_array_equal(_bits(norms), _bits(ovq.squared_norms4(cbt, nt)))
    np.testing.assert_array_equal(idx, want_idx)
    np.testing.assert_array_equal(_bits(q), _bits(want_q))
    # fp16 squared norms overflow on finite values: NaN distances keep first-index priority
    special = np.array([[np.nan, 0, 0, 0], [300, 1, -2, 3]], np.float32).astype(nt)
    idx, _, _ = _search(pkg, dev, special, cbt, tt)
    np.testing.assert_array_equal(idx, ovq.nearest_codebook4(special, cbt, nt))


@pytest.mark.parametrize("dtype", list(DTYPES))
def test_quantize_strided_batches(pkg, dev, dtype) -> None:
    """A strided (2, 4, 9, 8, 7) latent against 2,048 codes through VqDecoder.quantize: the
    straight-through values equal the oracle's bit for bit (tests/test_vq_optimized.py:27-51)."""
    tt, nt = DTYPES[dtype]
    rng = np.random.default_rng(2701)
    cb = rng.normal(size=(2048, 4)).astype(np.float32).astype(nt)
    z = rng.normal(size=(2, 4, 9, 8, 14)).astype(np.float32).astype(nt)[..., ::2]
    zt = torch.from_numpy(np.ascontiguousarray(z)).to(dev).permute(0, 2, 3, 4, 1)   # NDHWC view, strided
    dec = pkg.vq.VqDecoder({"quantize.embedding.weight": cb})
    got = dec.quantize(zt, tt)
    torch.cuda.synchronize()
    flat = z.transpose(0, 2, 3, 4, 1).reshape(-1, 4)
    _, want = ovq.quantize4(flat, cb, nt)
    np.testing.assert_array_equal(_bits(got.cpu().numpy().reshape(-1, 4)), _bits(want))


def test_replacing_the_codebook_replaces_its_norms(pkg, dev) -> None:
    """A decoder whose codebook is replaced selects from the new codebook
    (tests/test_vq_optimized.py:97-113)."""
    dec = pkg.vq.VqDecoder({"quantize.embedding.weight": np.array([[0, 0, 0, 0], [2, 0, 0, 0]], np.float32)})
    z = torch.tensor([[[[[1.75, 0, 0, 0]]]]], dtype=torch.float32, device=dev)
    first = dec.quantize(z, torch.float32)
    dec.set_codebook(np.array([[1, 0, 0, 0], [20, 0, 0, 0]], np.float32))
    second = dec.quantize(z, torch.float32)
    torch.cuda.synchronize()
    assert first.reshape(4).tolist() == [2, 0, 0, 0]
    assert second.reshape(4).tolist() == [1, 0, 0, 0]


@pytest.mark.parametrize("dtype", list(DTYPES))
def test_config_sized_search_on_sampled_rows(pkg, dev, dtype) -> None:
    """51,200 latent vectors (a 32 x 40 x 40 latent) against 8,192 codes, four code chunks
    through LDS: 1,024 sampled rows (first and last included) equal the oracle."""
    tt, nt = DTYPES[dtype]
    rng = np.random.default_rng(99)
    cb = rng.normal(size=(8192, 4)).astype(nt)
    flat = rng.normal(size=(51200, 4)).astype(nt)
    idx, q, _ = _search(pkg, dev, flat, cb, tt)
    rows = np.unique(np.concatenate([[0, 51199], rng.integers(0, 51200, 1022)]))
    want_idx, want_q = ovq.quantize4(flat[rows], cb, nt)
    np.testing.assert_array_equal(idx[rows], want_idx)
    np.testing.assert_array_equal(_bits(q[rows]), _bits(want_q))


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize(("positions", "entries"), [(81920, 64), (82001, 2049), (81919, 4130), (97, 6143), (33, 65),
                                                    (24576, 64), (24577, 2049), (24576, 4130)])
def test_search_edges_of_chunks_and_schedules(pkg, dev, dtype, positions, entries) -> None:
    """Both schedules around their boundaries (fp16: whole scans from 81,920 positions; FP32: bounds
    above 24,576) and code counts around the 64-code chunks and 2,048-code stages; duplicates
    across chunks, values near zero and large, an all-zero and a non-finite latent: sampled rows
    and the last ones equal the oracle."""
    tt, nt = DTYPES[dtype]
    rng = np.random.default_rng(positions + entries)
    cb = (rng.normal(size=(entries, 4)) * np.exp2(rng.integers(-12, 5, (entries, 1)))).astype(nt)
    cb[-1] = cb[entries // 2] = cb[1]
    flat = (rng.normal(size=(positions, 4)) * np.exp2(rng.integers(-12, 5, (positions, 1)))).astype(nt)
    flat[-1], flat[-2], flat[-3], flat[-4] = cb[1], 0, cb[-2], np.inf
    idx, q, _ = _search(pkg, dev, flat, cb, tt)
    rows = np.unique(np.concatenate([[0], positions - 1 - np.arange(32), rng.integers(0, positions, 512)]))
    with np.errstate(invalid="ignore", over="ignore"):
        want_idx, want_q = ovq.quantize4(flat[rows], cb, nt)
    np.testing.assert_array_equal(idx[rows], want_idx)
    np.testing.assert_array_equal(_bits(q[rows][:-4]), _bits(want_q[:-4]))


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize(("positions", "entries"), [(1, 1), (300, 2), (257, 63), (257, 64), (24577, 128), (24577, 129),
                                                    (32768, 256), (32769, 256), (32769, 250), (81920, 249),
                                                    (32769, 257)])
def test_search_of_few_codes(pkg, dev, dtype, positions, entries) -> None:
    """Codebooks on both sides of the scan's boundaries, with duplicates, a non-finite code in every
    third case, zeros and infinite latents: sampled rows and the last ones equal the oracle."""
    tt, nt = DTYPES[dtype]
    rng = np.random.default_rng(positions + entries)
    cb, flat = rng.normal(size=(entries, 4)).astype(nt), rng.normal(size=(positions, 4)).astype(nt)
    cb[-1] = cb[entries // 2]
    if entries > 2 and (positions + entries) % 3 == 0:
        cb[entries - 2, 1] = np.inf
    if positions > 4:
        flat[-1], flat[-2], flat[-3, 0], flat[-4, 1] = cb[0], 0, np.inf, np.nan
    idx, q, _ = _search(pkg, dev, flat, cb, tt)
    rows = np.unique(np.concatenate([[0], np.maximum(positions - 1 - np.arange(300), 0), rng.integers(0, positions, 512)]))
    with np.errstate(invalid="ignore", over="ignore"):
        want_idx, want_q = ovq.quantize4(flat[rows], cb, nt)
    np.testing.assert_array_equal(idx[rows], want_idx)
    ok = ~np.isnan(want_q)
    np.testing.assert_array_equal(np.isnan(q[rows]), ~ok)
    np.testing.assert_array_equal(_bits(q[rows])[ok], _bits(want_q)[ok])


@pytest.mark.parametrize(("positions", "entries"), [(40, 8192), (82000, 8192), (82000, 200)])
def test_half_dots_are_rounded_to_fp32_first(pkg, dev, positions, entries) -> None:
    """fp16 latents whose chosen code depends on the dot's rounding to fp32 before fp16 (one fused
    rounding gives another index): every schedule takes the oracle's."""
    rng = np.random.default_rng(417792)
    cb, flat = (rng.normal(size=(n, 4)).astype(np.float32).astype(np.float16) for n in (8192, 409600))
    flat = np.resize(flat[[15652, 277019, 392416]], (positions, 4))
    if entries < 8192:
        cb = np.concatenate([cb[[7303, 7232, 2805, 3631, 6794, 5333]], cb[:entries - 6]])
    idx, _, _ = _search(pkg, dev, flat, cb, torch.float16)
    want, _ = ovq.quantize4(flat[:3], cb, np.float16)
    if entries == 8192:
        np.testing.assert_array_equal(want, [7232, 3631, 5333])
    np.testing.assert_array_equal(idx, np.resize(want, positions))


def test_search_rejects_bad_arguments(pkg, dev) -> None:
    """Shape and dtype errors raise before anything is launched."""
    z = torch.zeros((3, 4), dtype=torch.float16, device=dev)
    cb = torch.zeros((5, 4), dtype=torch.float32, device=dev)
    with pytest.raises(ValueError):
        pkg.ops.nearest_codebook4(z, cb, torch.zeros(5, dtype=torch.float32, device=dev))
    with pytest.raises(ValueError):
        pkg.ops.nearest_codebook4(torch.zeros((3, 3), dtype=torch.float16, device=dev), cb.half(),
                                  torch.zeros(5, dtype=torch.float16, device=dev))
    with pytest.raises(ValueError):
        pkg.ops.squared_norms4(torch.zeros((0, 4), dtype=torch.float16, device=dev))


@pytest.mark.parametrize(("kind", "positions", "entries"), [
    ("normal", 24576, 1025), ("normal", 24577, 1024), ("normal", 24833, 1), ("normal", 25000, 65),
    ("crowded", 24600, 4133),      # many codes within the bounds' error of the least
    ("repeated", 24600, 1500),     # every code eight times: the exact search of whole workgroups
    ("lattice", 30001, 700),       # exact ties at midpoints
    ("tiny", 24700, 2047), ("large", 24700, 2047),   # large: beyond the powers of two that scale
    ("mixed", 24700, 3000), ("nan code", 24700, 300), ("infinite code", 24700, 300), ("zero codes", 24700, 129),
])
def test_search_from_bounds(pkg, dev, kind, positions, entries) -> None:
    """FP32 above 24,576 positions, which searches only the chunks that fp16 bounds leave: every
    index (of sampled rows, and of rows with NaN, infinite, zero and huge components) equals the
    oracle's, for data on which the bounds decide little or nothing."""
    rng = np.random.default_rng(positions + entries)
    cb, flat = rng.normal(size=(entries, 4)), rng.normal(size=(positions, 4))
    if kind == "crowded":
        cb[entries // 3:] = rng.uniform(-1, 1, (entries - entries // 3, 4)) / entries
    elif kind == "repeated":
        cb = cb[rng.integers(0, entries // 8, entries)]
    elif kind == "lattice":
        cb, flat = rng.integers(-2, 3, cb.shape) * 1.0, rng.integers(-3, 4, flat.shape) / 2
    elif kind == "tiny":
        cb, flat = cb * 3e-3, flat * 1e-4
    elif kind == "large":
        cb, flat = cb * 1e7, flat * 1e7
    elif kind == "mixed":
        cb = cb * np.exp2(rng.integers(-12, 3, (entries, 1)))
        flat = flat * np.exp2(rng.integers(-30, 30, (positions, 1)))
    elif kind == "zero codes":
        cb = cb * 0
    cb, flat = cb.astype(np.float32), flat.astype(np.float32)
    if kind.endswith("code"):
        cb[entries // 3, 1] = np.nan if kind == "nan code" else np.inf
    flat[3], flat[5, 2], flat[7, 1], flat[9] = 0, np.nan, -np.inf, 1e15
    idx, _, _ = _search(pkg, dev, flat, cb, torch.float32)
    rows = np.unique(np.concatenate([np.arange(16), positions - 1 - np.arange(16), rng.integers(0, positions, 400)]))
    with np.errstate(invalid="ignore", over="ignore"):
        want, _ = ovq.quantize4(flat[rows], cb, np.float32)
    np.testing.assert_array_equal(idx[rows], want)


@pytest.mark.parametrize("kind", ["doubled dot overflows", "around overflow", "subnormal", "around underflow"])
@pytest.mark.parametrize("positions", [70, 24700])
def test_search_beyond_the_normal_range(pkg, dev, kind, positions) -> None:
    """FP32 distances that overflow or are subnormal, below 24,577 positions and above: a dot whose
    double overflows beside an infinite sum of norms is a NaN, which wins. Every row equals the
    oracle's."""
    rng = np.random.default_rng(positions)
    cb, flat = rng.normal(size=(130, 4)), rng.normal(size=(positions, 4))
    if kind == "doubled dot overflows":
        cb, flat = cb * 0, flat * 1e19
        cb[100] = 1.2e19, 1.2e19, 0, 0
        cb[77] = 1.1e19, 0, 0, 0
        flat[:2] = [1e19, 1e19, 0, 0], [1.6e19, 0, 0, 0]
    else:
        lo, hi = {"around overflow": (55, 66), "subnormal": (-76, -70), "around underflow": (-68, -55)}[kind]
        cb, flat = (v * np.exp2(rng.integers(lo, hi, (len(v), 1))) for v in (cb, flat))
    cb, flat = cb.astype(np.float32), flat.astype(np.float32)
    idx, _, _ = _search(pkg, dev, flat, cb, torch.float32)
    with np.errstate(invalid="ignore", over="ignore"):
        want, _ = ovq.quantize4(flat, cb, np.float32)
    if kind == "doubled dot overflows":
        assert want[0] == 100 and want[1] == 77
    np.testing.assert_array_equal(idx, want)


@pytest.mark.parametrize("positions", [3000, 24700])
@pytest.mark.parametrize("scale", [2.0 ** -20, 1.0, 1e5])
def test_search_of_near_ties_between_chunks(pkg, dev, positions, scale) -> None:
    """Pairs of codes in different 64-code chunks (every fourth pair with a third) at the same distance
    to the latents but for a few ulps of the distance, at norms 200 times that distance, where
    the bounds are widest beside it: every row equals the oracle's."""
    rng = np.random.default_rng(positions)
    cb = rng.normal(size=(192, 4))
    cb *= 60 / np.linalg.norm(cb, axis=1, keepdims=True)
    unit = lambda v: v / np.linalg.norm(v, axis=-1, keepdims=True)  # noqa: E731
    n = 24
    centre, u = 8 * unit(rng.normal(size=(n, 4))), unit(rng.normal(size=(n, 4)))
    v = rng.normal(size=(n, 4))
    v = unit(v - (v * u).sum(1, keepdims=True) * u)
    cb[:n], cb[128:128 + n] = centre + 0.5 * u, centre - 0.5 * u
    cb[64:64 + n:4] = (centre + 0.5 * v)[::4]
    i = rng.integers(0, n, positions)
    w = rng.normal(size=(positions, 4))
    for axis in (u[i], v[i] - (v[i] * u[i]).sum(1, keepdims=True) * u[i]):   # w orthogonal to u and v
        w -= (w * axis).sum(1, keepdims=True) * axis
    ulp = 2.0 ** -17   # of the norms' sum, 128, in FP32
    flat = centre[i] + 0.2 * unit(w) + u[i] * rng.integers(-4, 5, (positions, 1)) * ulp / 2
    cb, flat = (cb * scale).astype(np.float32), (flat * scale).astype(np.float32)
    idx, _, _ = _search(pkg, dev, flat, cb, torch.float32)
    d = ovq.distances4(flat, cb, np.float32)
    two = np.sort(d, axis=1)[:, :2].astype(np.float64)
    assert np.median(two[:, 1] - two[:, 0]) <= 4 * ulp * scale ** 2
    np.testing.assert_array_equal(idx, np.argmin(d, axis=1))
