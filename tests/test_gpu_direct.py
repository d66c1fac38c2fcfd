"""Direct all-pairs kernels through the C ABI (nbh_fcompute_direct).

FP64: bit-exact with the oracle `simple` restatement for any n (tails,
work-group sizes).  FP32 tiles: relative force error against the FP64 oracle
within the stated bound.
"""
import ctypes as C

import numpy as np
import pytest

import oracle_lib
from hip_capi import Ctx
from nbody_amd import native, nbody_data

pytestmark = pytest.mark.gpu

NBH_FP64, NBH_FP32, NBH_FP32_CORR, NBH_FP64_BLOCK = 0, 1, 2, 3

# Bounds on the relative error |a32 - a64| / |a64| of the FP32-tile kernel.
# Sources enter as FP32 offsets from the work-group's first target and the
# interaction uses v_rsq_f32, so the absolute error is a few FP32 ulps of the
# largest pair terms.  RMS and p99 over bodies stay under 1e-5; the maximum is
# set by the few bodies whose net acceleration nearly cancels (|a| far below
# its pair terms), where the same absolute error is a larger fraction.
FP32_MAX_REL = 1e-3
FP32_P99_REL = 1e-5
FP32_RMS_REL = 1e-5


@pytest.fixture(scope="module")
def ctx():
    c = Ctx(0)
    yield c
    c.close()


def _state(kind: str, n: int, seed: int):
    d = nbody_data()
    d.set_quiet(True)
    d.generate(kind, n, seed)
    return oracle_lib.state_from_data(d)


def _run(ctx, y, m, prec, bs=0):
    n = len(m)
    dy, dm, df = ctx.put(y), ctx.put(m), ctx.alloc(6 * n)
    native.check(ctx.lib.nbh_fcompute_direct(ctx.h, dy.ptr, dm.ptr, df.ptr, n, prec, bs), "fcompute")
    return df.read()


# (up to 4096 bodies on 256 CUs the work-group size is checked and chooses nothing)
@pytest.mark.parametrize("n,bs", [(1, 0), (7, 64), (100, 128), (1000, 256), (1024, 64), (1500, 1024)])
def test_fp64_bit_exact(ctx, n, bs):
    y, m = _state("ball", n, 11 + n)
    f = _run(ctx, y, m, NBH_FP64, bs)
    f0 = oracle_lib.fcompute_simple(y, m)
    assert np.array_equal(f, f0)


def _edge_state(n):
    """A ball in which some tiles hold operands outside the bare sequences' range."""
    y, m = _state("ball", n, 5 + n)
    if n > 70:
        m[n // 3] = 1e-70
        y[n - 2] = 2e6
        y[[0, n, 2 * n]] = y[[n // 2, n + n // 2, 2 * n + n // 2]]      # a coincident pair
    return y, m


# edges of the FP64 direct sums: 16 targets and 64 sources (terms through LDS, up to
# one work-group per CU: 4096 bodies on 256 CUs), 32 targets and 32 sources (turns)
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 63, 64, 65, 127, 129, 4095, 4096, 4097, 4128, 4161, 6001])
@pytest.mark.parametrize("law", [NBH_FP64, NBH_FP64_BLOCK])
def test_fp64_bit_exact_at_tile_edges(ctx, n, law):
    y, m = _edge_state(n)
    f = _run(ctx, y, m, law)
    f0 = oracle_lib.fcompute_simple(y, m, threads=0) if law == NBH_FP64 else oracle_lib.fcompute_block(y, m)
    assert np.array_equal(f, f0)


@pytest.mark.parametrize("n", [114687, 114689, 131071, 131073, 172032, 229375, 229376, 262143, 262144])
def test_fp64_large_matches_sampled_targets(ctx, n):
    """On both sides of the switches between turns and a target per work-item (7/8 of two,
    three and four waves per SIMD, and above, on 256 CUs) against the per-target sums of
    nbh_direct_sample, which keeps the same order."""
    y, m = _state("plummer", n, 9)
    idx = np.unique(np.concatenate([np.arange(0, n, 4099), [n - 2, n - 1]])).astype(np.uint32)
    dy, dm, df, di, da = ctx.put(y), ctx.put(m), ctx.alloc(6 * n), ctx.put_raw(idx), ctx.alloc(3 * len(idx))
    native.check(ctx.lib.nbh_fcompute_direct(ctx.h, dy.ptr, dm.ptr, df.ptr, n, NBH_FP64, 0), "fcompute")
    native.check(ctx.lib.nbh_direct_sample(ctx.h, dy.ptr, dm.ptr, n, di.ptr, len(idx), da.ptr), "direct_sample")
    f = df.read()
    assert np.array_equal(f[3 * n:].reshape(3, n)[:, idx].T, da.read().reshape(-1, 3))
    assert np.array_equal(f[:3 * n], y[3 * n:])


def _odd_roots(c, bits):
    """The odd M with M^2 = c (mod 2^bits), c = 1 (mod 8)."""
    m = 1
    for k in range(4, bits + 1):            # M^2 = c (mod 2^(k - 1)) -> (mod 2^k)
        if (m * m - c) % (1 << k):
            m += 1 << (k - 2)
    half = 1 << (bits - 1)
    return {r % (1 << bits) for r in (m, -m, m + half, half - m)}


def _hard_operands(count):
    """(r^2, -a) whose root and whose quotient a / (r^2 sqrt(r^2)) lie next to the middle
    of two doubles: r^2 = (M^2 - c) / 2^s with M odd of 54 bits, and a = (Q B - r) / 2^54
    with Q odd of 54 bits and B the denominator's significand, small odd c and r.  The
    root's last step multiplies by 1 / (2 sqrt(x)) (1 + d), |d| <= 1.5 (2^-24.18)^2 =
    2^-47.8 from v_rsq_f64's error, so a root M - c / (2 M) is sure to round right where
    |c| / 2^54 > |d|: |c| > 75."""
    rng = np.random.default_rng(1)
    r2 = []
    for k in [k for k in range(-1000, 1000) if abs(8 * k + 1) > 75]:
        for s in (54, 55):
            for m in _odd_roots(8 * k + 1, s):
                t = m * m - (8 * k + 1) >> s
                if m >> 53 == 1 and t >> 52 == 1:
                    # t 2^s has the root M: an even power of two leaves it as hard
                    r2.append(np.ldexp(float(t), s % 2 - 52 + 2 * int(rng.integers(-10, 20))))
    r2 = np.array(r2[:count // 2])
    r2 = np.concatenate([r2, 10.0 ** rng.uniform(-7, 12, count - len(r2))])
    a = np.empty(count)
    for i, b in enumerate(r2 * np.sqrt(r2)):
        b = int(np.ldexp(np.frexp(b)[0], 53))
        while b % 2 == 0:
            b >>= 1
        inv = pow(b, -1, 1 << 54)
        for r in range(1, 100, 2):
            q = (r if i % 2 else -r) * inv % (1 << 54)
            if q >> 53 == 1:
                break
        a[i] = np.ldexp(float(q * b - (r if i % 2 else -r) >> 54), -52)
    return r2, a


# terms through LDS, in turns and a target per work-item
@pytest.mark.parametrize("n", [4001, 20011, 1 << 18])
def test_fp64_quotients_next_to_midpoints(ctx, n):
    """The bare root and quotient round as IEEE's where that is hardest.  Body 0 is so
    heavy that every other body's sum is the one term it receives from it."""
    r2, a = (v[np.arange(n - 1) % len(v)] for v in _hard_operands(min(n - 1, 20010)))
    # RN(dx^2) + RN(dy^2) = r^2: dx from below, dy^2 the few ulps that are missing
    dx = np.sqrt(r2) * (1 - 2.0 ** -51)
    dy = np.sqrt(r2 - dx * dx)
    keep = dx * dx + dy * dy == r2
    assert keep.mean() > 0.99
    heavy = 2.0 ** 190
    y = np.zeros((6, n))
    y[0, 1:], y[1, 1:] = dx, dy
    m = np.concatenate([[heavy], a * 2.0 ** -150])
    f = _run(ctx, y.reshape(-1), m, NBH_FP64)[3 * n:].reshape(3, n)[:, 1:]
    coeff = (-m[1:] * heavy) / (r2 * np.sqrt(r2))
    for got, d in ((f[0], dx), (f[1], dy)):
        assert np.array_equal(got[keep], ((d * coeff) / m[1:])[keep])


def _sampled_sums(y, m, idx, law):
    """Accelerations of bodies idx, terms added in index order (cumsum adds in order)."""
    n = len(m)
    pos = y[:3 * n].reshape(3, n)
    out = np.empty((3, len(idx)))
    for k, i in enumerate(idx):
        d = pos[:, i, None] - pos
        r2 = np.maximum(d[0] * d[0] + d[1] * d[1] + d[2] * d[2], 1e-8)
        if law == NBH_FP64:
            c = (-1.0 * m[i] * m) / (r2 * np.sqrt(r2))
            c[i] = 0.0                                     # the self pair is left out: its term is a zero
            out[:, k] = [np.cumsum(np.concatenate([[0.0], d[a] * c]))[-1] / m[i] for a in range(3)]
        else:
            c = m / (np.sqrt(r2) * r2)
            out[:, k] = [np.cumsum(np.concatenate([[0.0], -(d[a] * c)]))[-1] for a in range(3)]
    return out


# a target per work-item: two waves on every SIMD of 256 CUs nearly full (work-groups of
# 64, 128, 256: 118011 bodies), and more than four (every work-group size: above 2^18)
@pytest.mark.parametrize("n,bs", [(118011, 0), (118011, 64), (118011, 128), (131072, 256), (262144 + 77, 512),
                                  (262144 + 77, 1024), (262144 + 1, 64), (262144 + 3, 192)])
@pytest.mark.parametrize("law", [NBH_FP64, NBH_FP64_BLOCK])
def test_fp64_target_per_lane_bit_exact(ctx, n, bs, law):
    """Ragged last work-groups and tiles of every size, both laws, and bodies and tiles
    with operands out of the bare sequences' range."""
    y, m = _edge_state(n)
    m[n // 5] = 1e70
    idx = np.array([0, 1, 63, 64, n // 3, n // 2, n // 5, n // 5 + 1, n - 3, n - 2, n - 1, 255, 256, 1023, 1024, 77777])
    f = _run(ctx, y, m, law, bs)
    assert np.array_equal(f[:3 * n], y[3 * n:])
    assert np.array_equal(f[3 * n:].reshape(3, n)[:, idx], _sampled_sums(y, m, idx, law))


def test_fp64_clamp_and_coincident(ctx):
    """Pairs closer than 1e-4 use r^2 = 1e-8; coincident bodies contribute 0."""
    pos = np.array([[0, 0, 0], [1e-5, 0, 0], [1e-5, 0, 0], [1, 2, 3]], dtype=np.float64)
    m = np.array([1.0, 2.0, 3.0, 4.0])
    y = np.concatenate([pos[:, 0], pos[:, 1], pos[:, 2], np.zeros(12)])
    f = _run(ctx, y, m, NBH_FP64)
    assert np.array_equal(f, oracle_lib.fcompute_simple(y, m))
    # body 0 sees bodies 1, 2 at distance 1e-5 through the clamp: a = m dx / 1e-12
    ax_near = (2.0 + 3.0) * 1e-5 / (1e-8 * np.sqrt(1e-8))
    assert abs(f[3 * 4 + 0] - ax_near) / ax_near < 1e-3


def test_fp64_rejects_bad_args(ctx):
    lib = ctx.lib
    d = ctx.alloc(6)
    assert lib.nbh_fcompute_direct(ctx.h, None, d.ptr, d.ptr, 1, NBH_FP64, 0) == 1
    assert lib.nbh_fcompute_direct(ctx.h, d.ptr, d.ptr, d.ptr, 1, NBH_FP64, 0) == 1   # y == f
    e = ctx.alloc(6)
    assert lib.nbh_fcompute_direct(ctx.h, d.ptr, d.ptr, e.ptr, 1, NBH_FP64, 100) == 1  # bad block size
    assert lib.nbh_fcompute_direct(ctx.h, d.ptr, d.ptr, e.ptr, 1, 7, 0) == 1          # bad precision


def _rel_err(f, f0, n):
    a = f[3 * n:].reshape(3, n)
    a0 = f0[3 * n:].reshape(3, n)
    rel = np.linalg.norm(a - a0, axis=0) / np.linalg.norm(a0, axis=0)
    return rel


@pytest.mark.parametrize("kind,n", [("plummer", 4096), ("ball", 3000), ("plummer", 20000), ("cube", 8192)])
def test_fp32_accuracy(ctx, kind, n):
    y, m = _state(kind, n, 5)
    f = _run(ctx, y, m, NBH_FP32)
    f0 = oracle_lib.fcompute_simple(y, m, threads=0)
    assert np.array_equal(f[:3 * n], y[3 * n:])          # velocity copy is exact
    _check_rel(_rel_err(f, f0, n))


def _check_rel(rel):
    rms = float(np.sqrt(np.mean(rel ** 2)))
    p99 = float(np.percentile(rel, 99))
    assert rel.max() < FP32_MAX_REL, f"max rel {rel.max():.3e}"
    assert p99 < FP32_P99_REL, f"p99 rel {p99:.3e}"
    assert rms < FP32_RMS_REL, f"rms rel {rms:.3e}"


# blocks of 256, 512, 1024 and 2048 bodies (1, 2, 4, 8 per lane), odd and even
# numbers of blocks, last blocks of one body, one 64-body row and one missing body
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 255, 256, 257, 511, 513, 769, 1025, 4095, 4097, 24575, 24576, 24577,
                               49151, 49153, 163839, 163841])
def test_fp32_block_edges(ctx, n):
    """Every pair once: a block pair left out or met twice shows as an error of at
    least a few bodies in n, far above FP32 rounding."""
    y, m = _state("ball", n, 3 + n)
    m = m * np.random.default_rng(n).uniform(0.5, 1.5, n)
    f = _run(ctx, y, m, NBH_FP32)
    f64 = _run(ctx, y, m, NBH_FP64)
    assert np.array_equal(f[:3 * n], y[3 * n:])
    if n > 1:
        _check_rel(_rel_err(f, f64, n))
    assert np.array_equal(f, _run(ctx, y, m, NBH_FP32))      # the same bits again
    fc = _run(ctx, y, m, NBH_FP32_CORR)
    if n > 1:
        e, ec = _rel_err(f, f64, n), _rel_err(fc, f64, n)
        assert ec.mean() <= 1.5 * e.mean()
        if n > 64:                 # beyond the window of 32 on either side
            assert np.sqrt(np.mean(ec ** 2)) < np.sqrt(np.mean(e ** 2)) and ec.max() <= e.max()


@pytest.mark.parametrize("scale", [1e-3, 1e9])
def test_fp32_far_apart_and_clamped(ctx, scale):
    """Distances whose cube leaves FP32 (1e9) and distances around the clamp (1e-3)."""
    n = 3000
    y, m = _state("ball", n, 8)
    y[:3 * n] *= scale
    f = _run(ctx, y, m, NBH_FP32)
    f64 = _run(ctx, y, m, NBH_FP64)
    rel = np.linalg.norm((f - f64)[3 * n:].reshape(3, n), axis=0)
    rel /= np.sqrt(np.mean(np.sum(f64[3 * n:].reshape(3, n) ** 2, axis=0)))
    assert np.sqrt(np.mean(rel ** 2)) < FP32_RMS_REL and rel.max() < FP32_MAX_REL


# sizes with blocks of 256, 512, 1024 and 2048 bodies
@pytest.mark.parametrize("n,halo,clump", [(8192, 10.0, 1e-3), (40000, 100.0, 1e-2), (100000, 10.0, 1e-3),
                                          (200000, 100.0, 1e-2)])
@pytest.mark.parametrize("prec", [NBH_FP32, NBH_FP32_CORR])
def test_fp32_clump_in_a_wide_state(ctx, n, halo, clump, prec):
    """Half the bodies in a clump 10^4 times smaller than the ball around it.  Offsets
    taken close to the clump leave its pairs a few FP32 roundings (8 x 2^-24 bounds
    those of offsets, r^2, rsq, products and sums in the median); offsets taken in the ball
    round at 10^4 x 2^-24 = 6e-4 of the clump's size, and the median of the clump's bodies
    is then 4e-6 to 2e-4.  The few bodies that share their 1024 with the ball keep such
    errors, whichever origin the others have: one in a hundred may, no bound on the
    maximum."""
    rng = np.random.default_rng(n)

    def ball(k, r):
        u = rng.standard_normal((3, k))
        return u * (r * rng.random(k) ** (1 / 3) / np.linalg.norm(u, axis=0))

    k = n // 2
    pos = np.concatenate([ball(n - k, halo), ball(k, clump) + 1.0], axis=1)
    order = rng.permutation(n)
    y = np.concatenate([pos[:, order].reshape(-1), np.zeros(3 * n)])
    m = rng.uniform(0.5, 1.5, n) / n
    rel = _rel_err(_run(ctx, y, m, prec), _run(ctx, y, m, NBH_FP64), n)
    inside = rel[order >= n - k]
    print(f"\n[fp32] n={n} clump median {np.median(inside):.2e} p99 {np.percentile(inside, 99):.2e}, "
          f"ball median {np.median(rel[order < n - k]):.2e}")
    assert np.median(inside) < 8 * 2.0 ** -24
    assert np.percentile(inside, 99) < halo / clump * 2.0 ** -24
    assert np.median(rel[order < n - k]) < 8 * 2.0 ** -24


def test_fp32_matches_fp64_kernel_large(ctx):
    """At 2^17 bodies (no CPU reference needed) the FP32 tiles agree with the
    FP64 kernel, which is bit-exact with the oracle at every smaller size."""
    n = 1 << 17
    y, m = _state("plummer", n, 3)
    f32 = _run(ctx, y, m, NBH_FP32)
    f64 = _run(ctx, y, m, NBH_FP64)
    _check_rel(_rel_err(f32, f64, n))
    # momentum balance of the FP64 kernel: sum m a ~ 0 relative to sum m |a|
    a = f64[3 * n:].reshape(3, n)
    assert np.linalg.norm((a * m).sum(axis=1)) / np.sum(m * np.linalg.norm(a, axis=0)) < 1e-12


def test_fp32_corr_close_pair_far_from_origin(ctx):
    """A close pair 10 units from the tiles' origin: the FP32 rounding of the
    offsets (about 7e-7 here) is a 1e-3 error on their 1e-3 separation, which the
    FP64 correction pass removes; the other bodies keep FP32 accuracy or better."""
    rng = np.random.default_rng(3)
    n = 64
    pos = rng.normal(size=(n, 3)) * 0.3
    pos[-2] = [10.0, 0.0, 0.0]
    pos[-1] = [10.00123456789, 0.000333333, -0.000271828]   # no multiple of the float spacing
    m = rng.uniform(0.5, 1.5, n) / n
    y = np.concatenate([pos[:, 0], pos[:, 1], pos[:, 2], rng.normal(size=3 * n)])
    f0 = oracle_lib.fcompute_simple(y, m)
    e32 = _rel_err(_run(ctx, y, m, NBH_FP32), f0, n)
    fc = _run(ctx, y, m, NBH_FP32_CORR)
    assert np.array_equal(fc[:3 * n], y[3 * n:])
    ec = _rel_err(fc, f0, n)
    print(f"\n[fp32 correction] close pair rel err: FP32 {e32[-2:].max():.2e}, corrected {ec[-2:].max():.2e}; "
          f"others max {e32[:-2].max():.2e} -> {ec[:-2].max():.2e}")
    assert e32[-2:].min() > 1e-5                  # the FP32 tiles do lose the pair
    assert ec[-2:].max() < 1e-7
    assert ec.max() < 1e-6


# blocks of 256, 512, 1024 and 2048 bodies
@pytest.mark.parametrize("n,kb", [(1024, 256), (24576, 512), (49152, 1024), (163840, 2048)])
def test_fp32_corr_takes_out_the_tiles_own_terms(ctx, n, kb):
    """All bodies but two without mass, so that each of the two receives one term: the
    correction pass must find the tiles' FP32 term to the last bit, for neighbours in one
    block and in two, and leave the FP64 term (a few roundings of 2^-53; an FP32 term that
    differs in its last bit leaves 3e-8)."""
    rng = np.random.default_rng(n)
    # order along the curve: x, as y and z stay in the first of 1024 cells (the last body
    # alone sets the box)
    x = (np.arange(n) + 0.6 * rng.random(n)) / n
    pos = np.stack([x, 9e-4 * rng.random(n), 9e-4 * rng.random(n)])
    pos[:, -1] = 1.0
    y = np.concatenate([pos.reshape(-1), np.zeros(3 * n)])
    for a, b in [(kb - 1, kb), (2 * kb - 3, 2 * kb + 5), (3 * kb - 1, 3 * kb + 1), (kb + 7, kb + 9), (kb + 63, kb + 64)]:
        m = np.zeros(n)
        m[[a, b]] = rng.uniform(0.5, 1.5, 2)
        f = _run(ctx, y, m, NBH_FP32_CORR)[3 * n:].reshape(3, n)
        d = pos[:, b] - pos[:, a]
        w = d / max(d @ d, 1e-8) ** 1.5
        for got, want in ((f[:, a], m[b] * w), (f[:, b], -m[a] * w)):
            assert np.linalg.norm(got - want) < 1e-14 * np.linalg.norm(want), (a, b)


# blocks of 512, 256, 1024 and 2048 bodies
@pytest.mark.parametrize("kind,n", [("plummer", 32768), ("cube", 16384), ("cube", 65537), ("plummer", 200003)])
def test_fp32_corr_accuracy(ctx, kind, n):
    """With the correction pass the force error against the FP64 kernel drops
    below that of the FP32 tiles alone (largest and RMS relative error)."""
    y, m = _state(kind, n, 7)
    f64 = _run(ctx, y, m, NBH_FP64)
    e32 = _rel_err(_run(ctx, y, m, NBH_FP32), f64, n)
    ec = _rel_err(_run(ctx, y, m, NBH_FP32_CORR), f64, n)
    r32, rc = float(np.sqrt(np.mean(e32 ** 2))), float(np.sqrt(np.mean(ec ** 2)))
    print(f"\n[fp32 correction] {kind} n={n}: rms {r32:.2e} -> {rc:.2e}, max {e32.max():.2e} -> {ec.max():.2e}")
    _check_rel(ec)
    assert rc < r32 and ec.max() < e32.max()
