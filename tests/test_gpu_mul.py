"""GPU: batched products (schoolbook kernels and the two-prime binary64 NTT)
bit-exact against GMP's mpn_mul through the oracle.

Shapes: the schoolbook size classes, every NTT plan class (one tile; column +
row; two columns + row), the 1024-limb boundary of the reference
(batch_arith_test.cu:99-103), random shapes with random strides in the style
of batch_mul_ntt_test.cu:531-556, and broadcast operands."""
import ctypes
import time

import numpy as np
import pytest

import gpupi_amd as g
import oracle_ffi as of
from helpers import DEFAULT_NTT_MIN_LIMBS, rand_rows, to_int

pytestmark = pytest.mark.gpu
PAD = 0xDEADBEEF


def oracle_mul(A, B, sa=None, sb=None):
    n = A.shape[0]
    hc = of.HostArray.empty(n, A.shape[1] + B.shape[1])
    assert of.lib().o_mul(of.HostArray(A, sa).oarray(), of.HostArray(B, sb).oarray(), hc.oarray()) == 0
    return hc.rows()


def device_mul(ctx, A, B, sa=None, sb=None, sc_extra=1, b_broadcast=False):
    n = A.shape[0]
    lc = A.shape[1] + B.shape[1]
    ba, Aa = g.upload_rows(A, sa)
    bb, Ba = g.upload_rows(B if not b_broadcast else B[:1], sb)
    if b_broadcast:
        Ba = Ba.view(batch_size=n, stride=0)
    sc = lc + sc_extra
    bc, Ca = g.upload_rows(np.full((n, sc), PAD, dtype=np.uint32), sc)
    Ca.length = lc
    g.check(ctx.mul(Aa, Ba, Ca), "mul")
    g.synchronize()
    full = bc.download(np.uint32, count=n * sc).reshape(n, sc)
    assert np.all(full[:, lc:] == PAD), "write past the product"
    return full[:, :lc]


SCHOOLBOOK = [(1000, 1, 1), (777, 3, 3), (500, 4, 6), (300, 16, 9), (64, 100, 16), (40, 17, 17),
              (33, 64, 64), (9, 200, 150), (5, 512, 512), (3, 1000, 24), (2, 5000, 3000), (2, 8192, 8192)]
NTT = [(1, 8, 8), (100, 9, 7), (64, 32, 32), (17, 100, 100), (9, 513, 512), (5, 1024, 1024), (3, 2048, 2047),
       (2, 2049, 2047), (4, 3000, 1000), (3, 4097, 4095), (2, 10000, 9000), (2, 65536, 65536),
       (1, 300000, 200000), (1, 1048576, 1048576), (3, 2097152, 1), (1, 2097153, 2097152)]


@pytest.mark.parametrize("n,la,lb", SCHOOLBOOK, ids=[f"N{n}_{a}x{b}" for n, a, b in SCHOOLBOOK])
def test_schoolbook(ctx, n, la, lb):
    g.check(ctx.set_ntt_threshold(1 << 30))
    try:
        rng = np.random.default_rng(100)
        for mode in ("random", "ones"):
            A = rand_rows(rng, n, la, mode)
            B = rand_rows(rng, n, lb, mode)
            assert np.array_equal(device_mul(ctx, A, B, la + 3, lb + 1), oracle_mul(A, B, la + 3, lb + 1))
    finally:
        g.check(ctx.set_ntt_threshold(384))


@pytest.mark.parametrize("n,la,lb", NTT, ids=[f"N{n}_{a}x{b}" for n, a, b in NTT])
def test_ntt(ctx, n, la, lb):
    g.check(ctx.set_ntt_threshold(2))
    try:
        rng = np.random.default_rng(1234)
        for mode in ("random", "ones"):
            A = rand_rows(rng, n, la, mode)
            B = rand_rows(rng, n, lb, mode)
            assert np.array_equal(device_mul(ctx, A, B), oracle_mul(A, B)), mode
    finally:
        g.check(ctx.set_ntt_threshold(384))


SQUARES = [(5, 900, None), (3, 20000, None), (2, 20000, 20003), (1, 3000000, None), (4, 3000, 0)]


@pytest.mark.parametrize("n,la,stride", SQUARES, ids=[f"N{n}_{a}_s{s}" for n, a, s in SQUARES])
def test_ntt_square(ctx, n, la, stride):
    # A * A through one operand (the library transforms it once): one tile,
    # two and three levels, rows at a stride, and one row at stride 0
    g.check(ctx.set_ntt_threshold(2))
    try:
        rng = np.random.default_rng(la + n)
        for mode in ("random", "ones"):
            A = rand_rows(rng, 1 if stride == 0 else n, la, mode)
            buf, Aa = g.upload_rows(A, None if stride in (None, 0) else stride)
            if stride == 0:
                Aa = Aa.view(batch_size=n, stride=0)
                A = np.repeat(A, n, axis=0)
            lc = 2 * la
            bc, Ca = g.upload_rows(np.full((n, lc + 1), PAD, dtype=np.uint32), lc + 1)
            Ca.length = lc
            g.check(ctx.mul(Aa, Aa, Ca), "mul")
            g.synchronize()
            full = bc.download(np.uint32, count=n * (lc + 1)).reshape(n, lc + 1)
            assert np.all(full[:, lc:] == PAD), "write past the product"
            assert np.array_equal(full[:, :lc], oracle_mul(A, A)), mode
    finally:
        g.check(ctx.set_ntt_threshold(384))


ALIGNED = [(4, 3000, 2900), (3, 40000, 30000), (2, 300000, 200000), (1, 1 << 20, 1 << 20)]


@pytest.mark.parametrize("n,la,lb", ALIGNED, ids=[f"N{n}_{a}x{b}" for n, a, b in ALIGNED])
def test_ntt_aligned_rows(ctx, n, la, lb):
    # output rows 16-byte aligned (stride a multiple of 4 limbs): the final
    # carry pass runs four limbs per lane; all-ones operands make carry
    # chains cross its 1024-limb chunks
    g.check(ctx.set_ntt_threshold(2))
    try:
        rng = np.random.default_rng(la)
        for mode in ("random", "ones", "top"):
            A = rand_rows(rng, n, la, mode)
            B = rand_rows(rng, n, lb, mode)
            extra = (-(la + lb)) % 4 + 4
            assert np.array_equal(device_mul(ctx, A, B, sc_extra=extra), oracle_mul(A, B)), mode
    finally:
        g.check(ctx.set_ntt_threshold(384))


def test_boundary_shapes(ctx):
    # batch_arith_test.cu:99-103: 512+512 (naive there), 513+512, 2200+2200
    rng = np.random.default_rng(7)
    for la, lb in [(512, 512), (513, 512), (2200, 2200)]:
        A = rand_rows(rng, 6, la)
        B = rand_rows(rng, 6, lb)
        assert np.array_equal(device_mul(ctx, A, B), oracle_mul(A, B))


def test_random_shapes_and_strides(ctx):
    # batch_mul_ntt_test.cu:531-556 style: log-uniform lengths, random split, strides L+1..8
    rng = np.random.default_rng(100)
    for _ in range(24):
        total = int(2 ** rng.uniform(1, 15))
        la = max(1, int(rng.integers(1, total + 1)))
        lb = max(1, total - la) if total > la else 1
        n = max(1, int(50000 // (la + lb)))
        n = min(n, 200)
        sa = la + int(rng.integers(0, 8))
        sb = lb + int(rng.integers(0, 8))
        A = rand_rows(rng, n, la)
        B = rand_rows(rng, n, lb)
        assert np.array_equal(device_mul(ctx, A, B, sa, sb, sc_extra=int(rng.integers(1, 5))),
                              oracle_mul(A, B, sa, sb)), (n, la, lb)


def test_broadcast_operand(ctx):
    # convert_decimal multiplies every row by one power (stride 0); above
    # one tile the power's last level is transformed once for every row
    rng = np.random.default_rng(3)
    for n, la, lb, mode in [(33, 10, 7, "random"), (33, 300, 300, "random"), (33, 1500, 2500, "random"),
                            (33, 9000, 7000, "random"), (5, 70000, 60000, "ones"), (3, 600000, 400000, "random")]:
        A = rand_rows(rng, n, la, mode)
        B = np.repeat(rand_rows(rng, 1, lb, mode), n, axis=0)
        assert np.array_equal(device_mul(ctx, A, B, b_broadcast=True), oracle_mul(A, B)), (n, la, lb)


def every_size_case(k):
    # La + Lb in (2^(k-1), 2^k]: transform size 2^k, unequal operands
    total = (1 << k) - (k % 3)
    la = total // 2 + k
    return max(1, min(64, (1 << 22) >> k)), la, total - la


EVERY_K = list(range(4, 25))
SLOW_K = [25, 26, 27]


@pytest.mark.parametrize("k", EVERY_K + [pytest.param(k, marks=pytest.mark.slow) for k in SLOW_K],
                         ids=[f"K2^{k}" for k in EVERY_K + SLOW_K])
def test_ntt_every_transform_size(ctx, k):
    # one case per transform size: every in-tile DFT size and level split
    g.check(ctx.set_ntt_threshold(2))
    try:
        n, la, lb = every_size_case(k)
        rng = np.random.default_rng(k)
        A = rand_rows(rng, n, la)
        B = rand_rows(rng, n, lb)
        assert np.array_equal(device_mul(ctx, A, B), oracle_mul(A, B)), (n, la, lb)
    finally:
        g.check(ctx.set_ntt_threshold(384))


def device_mul_shared(ctx, A1, A2, B, b_rows=None, b_broadcast=False):
    # C1 = A1 B, C2 = A2 B through one batch_mp_mul_shared call; B has
    # b_rows >= max(rows) rows, or one row at stride 0
    n1, n2 = A1.shape[0], A2.shape[0]
    lb = B.shape[1]
    b1, A1a = g.upload_rows(A1, A1.shape[1] + 2)
    b2, A2a = g.upload_rows(A2, A2.shape[1] + 1)
    bb, Ba = g.upload_rows(B[:1] if b_broadcast else B, lb + 3)
    if b_broadcast:
        Ba = Ba.view(batch_size=max(n1, n2), stride=0)
    outs = []
    arrs = []
    for n, la in ((n1, A1.shape[1]), (n2, A2.shape[1])):
        lc = la + lb
        bc, Ca = g.upload_rows(np.full((n, lc + 1), PAD, dtype=np.uint32), lc + 1)
        Ca.length = lc
        outs.append((bc, n, lc))
        arrs.append(Ca)
    g.check(ctx.mul_shared(A1a, A2a, Ba, arrs[0], arrs[1]), "mul_shared")
    g.synchronize()
    res = []
    for bc, n, lc in outs:
        full = bc.download(np.uint32, count=n * (lc + 1)).reshape(n, lc + 1)
        assert np.all(full[:, lc:] == PAD), "write past the product"
        res.append(full[:, :lc])
    return res


SHARED = [  # (N1, L1, N2, L2, rows of B, L_b)
    (7, 3000, 8, 4000, 8, 2500),          # two levels, one transform size, N1 < N2
    (3, 300000, 3, 290000, 4, 240000),    # two levels, one row of B unused
    (2, 2500000, 3, 2200000, 3, 2000000),  # three levels
    (1, 40000, 2, 30000, 2, 20000),
    (2, 100000, 3, 90000, 3, 80000),      # K = 2^18: last level 2^10
    (2, 200000, 2, 180000, 2, 150000),    # K = 2^19: last level 2^11
    (1, 10000000, 1, 9000000, 1, 8000000),  # K = 2^25: three levels, last 2^11
    (5, 100, 5, 90, 5, 80),               # schoolbook: two plain products
    (4, 1000, 4, 5000, 4, 700),           # different transform sizes: two plain products
    (6, 600, 6, 700, 6, 900),             # one tile each: two plain products
]


@pytest.mark.parametrize("n1,l1,n2,l2,nb,lb", SHARED, ids=[f"{a}x{b}_{c}x{d}_B{e}x{f}" for a, b, c, d, e, f in SHARED])
def test_mul_shared(ctx, n1, l1, n2, l2, nb, lb):
    rng = np.random.default_rng(n1 * 31 + l1)
    A1 = rand_rows(rng, n1, l1)
    A2 = rand_rows(rng, n2, l2)
    B = rand_rows(rng, nb, lb)
    C1, C2 = device_mul_shared(ctx, A1, A2, B)
    assert np.array_equal(C1, oracle_mul(A1, B[:n1]))
    assert np.array_equal(C2, oracle_mul(A2, B[:n2]))


def test_mul_shared_broadcast_and_tree_shape(ctx):
    rng = np.random.default_rng(77)
    # B one row at stride 0
    A1 = rand_rows(rng, 5, 9000)
    A2 = rand_rows(rng, 4, 7000)
    B = rand_rows(rng, 1, 6000)
    C1, C2 = device_mul_shared(ctx, A1, A2, B, b_broadcast=True)
    assert np.array_equal(C1, oracle_mul(A1, np.repeat(B, 5, axis=0)))
    assert np.array_equal(C2, oracle_mul(A2, np.repeat(B, 4, axis=0)))
    # carry chains: all-ones operands
    A1 = rand_rows(rng, 2, 50000, "ones")
    A2 = rand_rows(rng, 3, 60000, "ones")
    B = rand_rows(rng, 3, 40000, "ones")
    C1, C2 = device_mul_shared(ctx, A1, A2, B)
    assert np.array_equal(C1, oracle_mul(A1, B[:2]))
    assert np.array_equal(C2, oracle_mul(A2, B))


def test_shared_and_broadcast_across_chunks(ctx):
    # more rows than one launch chunk holds (rows * K > 2^28): the shared
    # operand's transform per chunk, and a broadcast operand transformed once
    # in the first chunk and reused by the next
    rng = np.random.default_rng(11)
    n, la, lb = 4100, 40000, 25000  # K = 2^16: 4096 rows per chunk
    A1 = rand_rows(rng, n, la)
    A2 = rand_rows(rng, n - 3, la - 7000)
    B = rand_rows(rng, n, lb)
    C1, C2 = device_mul_shared(ctx, A1, A2, B)
    assert np.array_equal(C1, oracle_mul(A1, B))
    assert np.array_equal(C2, oracle_mul(A2, B[:n - 3]))
    Bb = rand_rows(rng, 1, lb)
    C1, C2 = device_mul_shared(ctx, A1, A2, Bb, b_broadcast=True)
    assert np.array_equal(C1, oracle_mul(A1, np.repeat(Bb, n, axis=0)))
    assert np.array_equal(C2, oracle_mul(A2, np.repeat(Bb, n - 3, axis=0)))


def test_mul_shared_rejects_bad_shapes(ctx):
    rng = np.random.default_rng(3)
    A = rand_rows(rng, 4, 5000)
    B = rand_rows(rng, 2, 5000)  # fewer rows than the products
    ba, Aa = g.upload_rows(A)
    bb, Ba = g.upload_rows(B)
    bc1, C1 = g.upload_rows(np.zeros((4, 10000), dtype=np.uint32))
    bc2, C2 = g.upload_rows(np.zeros((4, 10000), dtype=np.uint32))
    assert ctx.mul_shared(Aa, Aa, Ba, C1, C2) != 0
    assert ctx.mul_shared(Aa, Aa, Aa, C1, C1) != 0  # outputs alias each other


def valid_splits(k):
    # every column split the kernels cover: (m0, m1) with m1 = 0 for two levels
    out = []
    for m0 in range(5, 10):
        for m1 in ([0] if k <= 21 else range(5, 10)):
            rest = k - m0 - m1
            if 6 <= rest <= 12:
                out.append((m0, m1))
    return out


SPLIT_K = [13, 16, 18, 20, 22, 23, 24]


@pytest.mark.parametrize("k", SPLIT_K, ids=[f"K2^{k}" for k in SPLIT_K])
def test_ntt_every_split(ctx, k):
    # the same product under every level split: bit-identical to the
    # built-in plan's product and to GMP
    g.check(ctx.set_ntt_threshold(2))
    default = g.ntt_get_split(k)
    try:
        n, la, lb = every_size_case(k)
        n = min(n, 4)
        rng = np.random.default_rng(100 + k)
        A = rand_rows(rng, n, la)
        B = rand_rows(rng, n, lb)
        want = oracle_mul(A, B)
        splits = valid_splits(k)
        assert len(splits) >= 2
        for m0, m1 in splits:
            g.ntt_set_split(k, m0, m1)
            levels = g.ntt_get_split(k)
            assert levels[0] == m0 and sum(levels) == k and (m1 == 0 or levels[1] == m1)
            assert np.array_equal(device_mul(ctx, A, B), want), (m0, m1)
    finally:
        g.ntt_set_split(k, 0)
        g.check(ctx.set_ntt_threshold(384))
    assert g.ntt_get_split(k) == default


SPLIT = [  # one row with L + 2 S <= K: the longer operand runs as two pieces at K / 2
    (3000000, 500000, "random"),    # K = 2^22
    (500000, 3000000, "random"),    # the longer operand second
    (2200000, 900000, "ones"),      # carries through the seam
    (6000000, 1000001, "top"),      # K = 2^23
]
SPLIT_MANY = [  # one row with S far shorter than L: many pieces at a small transform
    (4194309, 3000, "random"),      # K = 2^23, pieces of 2^16 - 2^17 points
    (3000, 4194309, "ones"),        # the longer operand second, carries through every seam
    (1500000, 40000, "top"),        # K = 2^21
    (1048600, 200000, "random"),    # K = 2^21, a few pieces
    (2500001, 70001, "sparse"),
]


@pytest.mark.parametrize("la,lb,mode", SPLIT, ids=[f"{a}x{b}_{m}" for a, b, m in SPLIT])
def test_unbalanced_product_splits_and_stays_exact(ctx, la, lb, mode):
    rng = np.random.default_rng(la ^ lb)
    A = rand_rows(rng, 1, la, mode)
    B = rand_rows(rng, 1, lb, mode)
    want = oracle_mul(A, B)
    g.kernel_stats_reset(True)
    try:
        got = device_mul(ctx, A, B, sa=la + 3, sb=lb + 1)
        sizes = {name.split("@2^")[1] for name, *_ in g.kernel_stats(by_size=True)}
    finally:
        g.kernel_stats_reset(False)
    k = (la + lb - 1).bit_length()
    assert str(k - 1) in sizes and str(k) not in sizes, sizes
    assert np.array_equal(got, want)
    # the plain form keeps the reference's one product at K points
    with g.Context() as plain:
        plain.set_form(g.FORM_PLAIN)
        assert np.array_equal(device_mul(plain, A, B), want)


@pytest.mark.parametrize("la,lb,mode", SPLIT_MANY, ids=[f"{a}x{b}_{m}" for a, b, m in SPLIT_MANY])
def test_very_unbalanced_product_runs_in_pieces_and_stays_exact(ctx, la, lb, mode):
    rng = np.random.default_rng(la + 7 * lb)
    A = rand_rows(rng, 1, la, mode)
    B = rand_rows(rng, 1, lb, mode)
    want = oracle_mul(A, B)
    g.kernel_stats_reset(True)
    try:
        got = device_mul(ctx, A, B, sa=la + 1, sb=lb + 2)
        sizes = {int(name.split("@2^")[1]) for name, *_ in g.kernel_stats(by_size=True)}
    finally:
        g.kernel_stats_reset(False)
    k = (la + lb - 1).bit_length()
    assert sizes and max(sizes) <= k - 2, sizes
    assert np.array_equal(got, want)
    # the same pairs through the ragged call (pieces too) and mixed with a
    # pair that stays whole
    C = rand_rows(rng, 1, 5000)
    D = rand_rows(rng, 1, 4000)
    bufs = [g.DeviceBuffer.from_array(x[0]) for x in (A, B, C, D)]
    outs = [g.DeviceBuffer.from_array(np.full(n + 1, PAD, dtype=np.uint32)) for n in (la + lb, 9000)]
    g.check(ctx.mul_ragged([(bufs[0].ptr, bufs[1].ptr, outs[0].ptr, la, lb),
                            (bufs[2].ptr, bufs[3].ptr, outs[1].ptr, 5000, 4000)]), "mul_ragged")
    g.synchronize()
    o0, o1 = outs[0].download(np.uint32), outs[1].download(np.uint32)
    assert o0[-1] == PAD and o1[-1] == PAD
    assert np.array_equal(o0[:-1], want[0])
    assert np.array_equal(o1[:-1], oracle_mul(C, D)[0])


LAUNCH_K = [10, 16, 20, 23, 24]


@pytest.mark.parametrize("k", LAUNCH_K, ids=[f"K2^{k}" for k in LAUNCH_K])
def test_ntt_every_launch_shape(ctx, k):
    # every tile-pairing mask (each column level kind paired or not) and
    # XCD chunks from the plain order to 256 tiles: bit-identical to GMP;
    # K = 2^23 and 2^24 have 2^7- and 2^8-point second levels, so every kind
    # meets both block shapes
    g.check(ctx.set_ntt_threshold(2))
    builtin = g.ntt_get_launch()
    try:
        n, la, lb = every_size_case(k)
        n = min(n, 4)
        rng = np.random.default_rng(300 + k)
        A = rand_rows(rng, n, la)
        B = rand_rows(rng, n, lb)
        want = oracle_mul(A, B)
        for mask in range(16):
            for chunk in ((0, 3, 5, 8) if mask in (0, 15) else (5,)):
                g.ntt_set_launch(mask, chunk)
                assert g.ntt_get_launch() == (mask, chunk)
                assert np.array_equal(device_mul(ctx, A, B), want), (mask, chunk)
    finally:
        g.ntt_set_launch(*builtin)
        g.check(ctx.set_ntt_threshold(384))
    assert g.ntt_get_launch() == builtin


def test_shared_products_every_launch_shape(ctx):
    # the paired last level (two products sharing B) under the extreme shapes
    rng = np.random.default_rng(77)
    A1, A2 = rand_rows(rng, 3, 70000), rand_rows(rng, 2, 65000)
    B = rand_rows(rng, 3, 60000)
    want1, want2 = oracle_mul(A1, B[:3]), oracle_mul(A2, B[:2])
    builtin = g.ntt_get_launch()
    try:
        for mask, chunk in ((0, 0), (15, 8), (5, 5), (10, 2)):
            g.ntt_set_launch(mask, chunk)
            c1, c2 = device_mul_shared(ctx, A1, A2, B)
            assert np.array_equal(c1, want1) and np.array_equal(c2, want2), (mask, chunk)
    finally:
        g.ntt_set_launch(*builtin)


def test_launch_shape_rejects_bad_values():
    builtin = g.ntt_get_launch()
    for mask, chunk in ((16, 5), (5, 9), (5, -1)):
        with pytest.raises(ValueError):
            g.ntt_set_launch(mask, chunk)
    assert g.ntt_get_launch() == builtin


@pytest.mark.slow
def test_ntt_three_level(ctx):
    # K = 2^23 and 2^25: two column levels + the contiguous level
    g.check(ctx.set_ntt_threshold(2))
    try:
        rng = np.random.default_rng(5)
        for la, lb in [(1 << 22, (1 << 22) - 5), (1 << 24, 1 << 24)]:
            A = rand_rows(rng, 1, la)
            B = rand_rows(rng, 1, lb)
            assert np.array_equal(device_mul(ctx, A, B), oracle_mul(A, B))
    finally:
        g.check(ctx.set_ntt_threshold(384))


def ragged_case(ctx, lengths, seed, mode="random"):
    """Upload pairs (rand_rows mode), run one ragged call, return (device C rows, host A, B)."""
    rng = np.random.default_rng(seed)
    bufs, items, As, Bs, Cs = [], [], [], [], []
    for la, lb in lengths:
        A = rand_rows(rng, 1, la, mode) if la else np.zeros((1, 0), np.uint32)
        B = rand_rows(rng, 1, lb, mode) if lb else np.zeros((1, 0), np.uint32)
        ba = g.DeviceBuffer.from_array(A.reshape(-1)) if la else None
        bb = g.DeviceBuffer.from_array(B.reshape(-1)) if lb else None
        bc = g.DeviceBuffer.from_array(np.full(la + lb + 1, PAD, dtype=np.uint32))
        bufs += [ba, bb, bc]
        items.append((ba.ptr if ba else None, bb.ptr if bb else None, bc.ptr, la, lb))
        As.append(A)
        Bs.append(B)
        Cs.append(bc)
    err = ctx.mul_ragged(items)
    g.synchronize()
    out = [c.download(np.uint32, count=la + lb + 1) for c, (la, lb) in zip(Cs, lengths)]
    return err, out, As, Bs, bufs


def test_ragged_products(ctx):
    # one call with schoolbook, one-tile, column+row and three-level sizes,
    # zero-length operands and repeated transform sizes
    lengths = [(0, 0), (5, 0), (0, 7), (1, 1), (3, 17), (100, 90), (1000, 900), (2048, 2048), (2049, 1),
               (3000, 3000), (5000, 1200), (4095, 1), (65536, 30000), (40000, 50000), (1 << 20, 1 << 20),
               (2097153, 5), (12, 70000), (700, 700), (1000, 900)]
    err, out, As, Bs, _ = ragged_case(ctx, lengths, 21)
    assert err == 0
    for (la, lb), C, A, B in zip(lengths, out, As, Bs):
        assert C[-1] == PAD, (la, lb)
        if la and lb:
            assert np.array_equal(C[:-1], oracle_mul(A, B)[0]), (la, lb)
        else:
            assert not np.any(C[:-1]), (la, lb)


def test_ragged_pieces_and_shared_operands(ctx):
    # one ragged call where rows share B operands: items naming one buffer
    # (whole products of one transform size, a prefix of it, the buffer on
    # the A side) and split products (two pieces, many pieces, the longer
    # operand on either side, two products with one shorter operand, all-ones
    # carries through every seam); every C ends at its length
    rng = np.random.default_rng(41)
    ops = {
        "b": rand_rows(rng, 1, 30000)[0], "a1": rand_rows(rng, 1, 40000)[0], "a2": rand_rows(rng, 1, 50000)[0],
        "a3": rand_rows(rng, 1, 35000)[0], "s": rand_rows(rng, 1, 3000)[0], "l1": rand_rows(rng, 1, 4194309)[0],
        "l2": rand_rows(rng, 1, 1500000)[0], "t1": rand_rows(rng, 1, 3000000)[0],
        "t2": rand_rows(rng, 1, 500000)[0], "o1": rand_rows(rng, 1, 2500001, "ones")[0],
        "o2": rand_rows(rng, 1, 70001, "ones")[0],
    }
    bufs = {k: g.DeviceBuffer.from_array(v) for k, v in ops.items()}
    # (A, B, A length, B length): lengths up to the buffer's
    pairs = [("a1", "b", 40000, 30000), ("a2", "b", 50000, 30000), ("a3", "b", 35000, 30000),
             ("a1", "b", 40000, 20000), ("b", "a3", 30000, 35000), ("l1", "s", 4194309, 3000),
             ("s", "l2", 3000, 1500000), ("t1", "t2", 3000000, 500000), ("t2", "t1", 500000, 3000000),
             ("o1", "o2", 2500001, 70001), ("a2", "b", 50000, 30000)]
    outs, items = [], []
    for a, b, la, lb in pairs:
        c = g.DeviceBuffer.from_array(np.full(la + lb + 1, PAD, dtype=np.uint32))
        outs.append(c)
        items.append((bufs[a].ptr, bufs[b].ptr, c.ptr, la, lb))
    g.kernel_stats_reset(True)
    try:
        g.check(ctx.mul_ragged(items), "mul_ragged")
        g.synchronize()
        sizes = {int(name.split("@2^")[1]) for name, *_ in g.kernel_stats(by_size=True)}
    finally:
        g.kernel_stats_reset(False)
    assert max(sizes) <= 21, sizes  # every long product ran in pieces
    for (a, b, la, lb), c in zip(pairs, outs):
        got = c.download(np.uint32, count=la + lb + 1)
        assert got[-1] == PAD, (a, b, la, lb)
        want = oracle_mul(ops[a][:la].reshape(1, -1), ops[b][:lb].reshape(1, -1))[0]
        assert np.array_equal(got[:-1], want), (a, b, la, lb)


def test_ragged_one_tile_products_of_all_ones(ctx):
    # the largest coefficients a one-tile product meets (2^11 products of
    # two all-ones limbs: above 2^74), through the per-item operand path
    lengths = [(2048, 2048), (2047, 2049), (1024, 1000), (300, 200), (2000, 96), (129, 127)]
    err, out, As, Bs, _ = ragged_case(ctx, lengths, 9, "ones")
    assert err == 0
    for (la, lb), C, A, B in zip(lengths, out, As, Bs):
        assert C[-1] == PAD, (la, lb)
        assert np.array_equal(C[:-1], oracle_mul(A, B)[0]), (la, lb)


@pytest.mark.parametrize("k", [4, 5, 6, 7, 8, 9, 10, 11, 12])
def test_one_tile_products_of_all_ones_every_size(ctx, k):
    # the one-tile kernel at every transform size 2^4..2^12 (with the
    # crossover lowered, so that the small sizes reach it) on all-ones
    # operands, whose coefficients are the largest a product of that size
    # meets; uniform and ragged calls
    g.check(ctx.set_ntt_threshold(2))
    try:
        K = 1 << k
        lengths = [(K // 2, K // 2), (K - 1, 1), (K // 2 + 1, K // 2 - 1), (3 * K // 8, 3 * K // 8 + 1)]
        err, out, As, Bs, _ = ragged_case(ctx, lengths, 9, "ones")
        assert err == 0
        for (la, lb), C, A, B in zip(lengths, out, As, Bs):
            assert C[-1] == PAD, (la, lb)
            assert np.array_equal(C[:-1], oracle_mul(A, B)[0]), (la, lb)
        A = np.full((5, K // 2), 0xFFFFFFFF, dtype=np.uint32)
        assert np.array_equal(device_mul(ctx, A, A.copy()), oracle_mul(A, A))
    finally:
        g.check(ctx.set_ntt_threshold(384))


def test_ragged_matches_uniform_call(ctx):
    # the same pairs through batch_mp_mul one by one
    lengths = [(3000, 2000), (777, 4000), (20000, 1), (9000, 9000)]
    err, out, As, Bs, _ = ragged_case(ctx, lengths, 5)
    assert err == 0
    for (la, lb), C, A, B in zip(lengths, out, As, Bs):
        assert np.array_equal(C[:-1], device_mul(ctx, A, B)[0])


def test_ragged_rejects_aliasing(ctx):
    buf = g.DeviceBuffer.from_array(np.ones(64, dtype=np.uint32))
    assert ctx.mul_ragged([(buf.ptr, buf.ptr + 64, buf.ptr, 8, 8)]) != 0
    assert ctx.mul_ragged([(None, buf.ptr, buf.ptr + 128, 8, 8)]) != 0


def test_tuner_times_every_launch_shape_and_restores_it(ctx):
    from gpupi_amd import tune
    ops = tune.Operands(20, seed=8)
    before = (g.ntt_get_launch(), g.group_stage_get_shape())
    res = tune.tune_launch(ctx, ops, ks=(14, 17, 20), reps=1)
    assert sorted(v for v, _ in res["pair_mask"]) == list(range(16))
    assert sorted(v for v, _ in res["xcd_chunk_log2"]) == list(range(9))
    assert sorted(v for v, _ in res["group_blocks"]) == [1, 2, 4, 8, 16]
    assert all(ms > 0 for key in ("pair_mask", "xcd_chunk_log2", "group_blocks") for _, ms in res[key])
    assert (g.ntt_get_launch(), g.group_stage_get_shape()) == before


def test_tuner_times_every_split_and_restores_the_plan(ctx):
    from gpupi_amd import tune
    ops = tune.Operands(20, seed=5)
    before = g.ntt_get_split(15)
    res = tune.tune_splits(ctx, ops, 15, reps=1)
    assert sorted(lv for lv, _ in res) == sorted((m0, 15 - m0) for m0, _ in tune.splits(15))
    assert all(ms > 0 for _, ms in res) and res[0][1] <= res[-1][1]
    assert g.ntt_get_split(15) == before
    # the tree's pattern: two products sharing an operand, every split exact
    ops = tune.Operands(20, seed=6, shared=True)
    before = g.ntt_get_split(16)
    res = tune.tune_splits(ctx, ops, 16, reps=1, shared=True)
    assert sorted(lv for lv, _ in res) == sorted((m0, 16 - m0) for m0, _ in tune.splits(16))
    assert g.ntt_get_split(16) == before


# Lengths around the matrix-core products' edges: a block of 32 digits (8
# limbs), 32 blocks (256 limbs, a tile and a step of the shorter operand), the
# one-, two- and four-group shapes, the longest total and one past it.
MFMA_SHAPES = [(17, 17), (18, 40), (63, 64), (64, 64), (120, 136), (127, 130), (128, 128), (17, 3000), (247, 249),
               (248, 248), (255, 256), (256, 257), (300, 212), (511, 513), (512, 512), (760, 776), (1016, 1016),
               (1016, 3072), (1025, 1023), (127, 3961), (1500, 1700), (2040, 2048), (2044, 2044), (2044, 2045)]


@pytest.mark.parametrize("la,lb", MFMA_SHAPES)
@pytest.mark.parametrize("n", [1, 3, 513])
def test_matrix_core_products(la, lb, n):
    """Products of 17..4088 limbs against Python integers: random limbs and
    the words at which the recoding to signed digits and the carries run
    longest (0x7f7f7f7f passes the recoding's carry on, all ones and powers of
    two pass the product's), rows apart, a broadcast operand, both operand
    orders; nothing is written past a row."""
    rng = np.random.default_rng(la * 5000 + lb + n)
    words = (0, 0x7F7F7F7F, 0x7F7F7F80, 0x80808080, 0xFFFFFFFF, 1)
    kinds = len(words) + 2

    def rows(count, length, shift):
        out = rng.integers(0, 1 << 32, size=(count, length), dtype=np.uint32)
        for i in range(count):
            k = (i + shift) % kinds
            if k < len(words):
                out[i] = words[k]
            elif k == len(words):  # long runs of both kinds
                out[i, : length // 2] = 0x7F7F7F7F
        return out

    def value(x):
        return int.from_bytes(np.ascontiguousarray(x).tobytes(), "little")

    with g.Context() as ctx:
        for shift in range(kinds) if n < kinds else (3,):
            A, B = rows(n, la, shift), rows(n, lb, 5 * shift + 1)
            bufa, va = g.upload_rows(A, la + 3, 0xDEADBEEF)
            bufb, vb = g.upload_rows(B, lb + 1, 0xDEADBEEF)
            want = [value(a) * value(b) for a, b in zip(A, B)]
            for x, y in ((va, vb), (vb, va)):
                bufc, vc = g.upload_rows(np.zeros((n, la + lb), np.uint32), la + lb + 2, 0xABCD1234)
                g.check(ctx.mul(x, y, vc))
                g.synchronize()
                full = bufc.download(np.uint32).reshape(n, la + lb + 2)
                assert [value(r[: la + lb]) for r in full] == want
                assert (full[:, la + lb:] == 0xABCD1234).all()
        # one row of A against every row of B
        bufc, vc = g.upload_rows(np.zeros((n, la + lb), np.uint32))
        g.check(ctx.mul(va.view(stride=0), vb, vc))
        g.synchronize()
        got = g.download_rows(vc, bufc)
        assert [value(r) for r in got] == [value(A[0]) * value(b) for b in B]


@pytest.mark.parametrize("k", [13, 14, 16, 18, 20, 21, 22, 23, 24])
def test_truncated_transforms(ctx, k):
    """Products whose transforms use only some of their 16 parts: totals at
    and next to every pair of parts of 2^k points, one row and several, equal
    and unequal lengths, a broadcast operand, a square and a shared pair with
    different numbers of parts, against GMP; nothing is written past a row."""
    # sizes set by hand (to the built-in ones) keep short launches on full tiles
    g.ntt_set_split(k, *(g.ntt_get_split(k)[:-1] if k < 20 else (0,)))
    try:
        truncated_products(ctx, k)
    finally:
        g.ntt_set_split(k, 0)


def truncated_products(ctx, k):
    rng = np.random.default_rng(k)
    K = 1 << k
    totals = sorted({min(max(K * t // 16 + d, K // 2 + 1), K) for t in (8, 10, 12, 14, 16) for d in (-1, 0, 1)})
    if k > 20:
        totals = totals[1::3]
    for i, total in enumerate(totals):
        la = total // 2 if i % 2 else total // 2 - total // 11
        lb = total - la
        n = 3 if k < 18 and i % 3 == 0 else 1
        A, B = rand_rows(rng, n, la, "random" if i % 4 else "ones"), rand_rows(rng, n, lb, "random" if i % 5 else "ones")
        assert np.array_equal(device_mul(ctx, A, B), oracle_mul(A, B)), (total, n)
        if n > 1:
            assert np.array_equal(device_mul(ctx, A, B, b_broadcast=True), oracle_mul(A, np.repeat(B[:1], n, axis=0)))
        if i % 3 == 1:
            buf, va = g.upload_rows(A)
            bufc, vc = g.upload_rows(np.zeros((n, 2 * la), np.uint32))
            g.check(ctx.mul(va, va, vc), "square")
            g.synchronize()
            assert np.array_equal(g.download_rows(vc, bufc), oracle_mul(A, A))
    la1, la2, lb = K // 4 + 5, K // 2 - 3, K // 4 + 77
    A1, A2, B = (rand_rows(rng, 1, n, "random") for n in (la1, la2, lb))
    (b1, v1), (b2, v2), (bb, vb) = g.upload_rows(A1), g.upload_rows(A2), g.upload_rows(B)
    c1, w1 = g.upload_rows(np.zeros((1, la1 + lb), np.uint32))
    c2, w2 = g.upload_rows(np.zeros((1, la2 + lb), np.uint32))
    g.check(ctx.mul_shared(v1, v2, vb, w1, w2), "mul_shared")
    g.synchronize()
    assert np.array_equal(g.download_rows(w1, c1), oracle_mul(A1, B))
    assert np.array_equal(g.download_rows(w2, c2), oracle_mul(A2, B))


@pytest.mark.parametrize("k", [13, 14, 15, 16, 17, 18, 19])
def test_thin_tiles(ctx, k):
    """Few products of 2^k points run on thin tiles, the same call with the
    level sizes set by hand on full ones: both give GMP's product for full and
    half-full transforms, lopsided and all-ones operands, padded rows, a
    broadcast operand on either side, squares and shared pairs, and around
    the number of rows where the thin tiles end."""
    rng = np.random.default_rng(900 + k)
    K = 1 << k
    builtin = g.ntt_get_split(k)[:-1]

    def both(run, want):
        for sizes in ((0,), builtin):
            g.ntt_set_split(k, *sizes)
            try:
                assert all(np.array_equal(x, y) for x, y in zip(run(), want)), sizes
            finally:
                g.ntt_set_split(k, 0)

    for n, la, lb, mode in ((1, K // 2, K // 2, "ones"), (1, K // 2, K // 2, "random"), (2, K - 4090, 4090, "random"),
                            (1, K // 4 + 1, K // 4, "random"), (1, K // 2 - 999, K // 4 + 3, "ones")):
        A, B = rand_rows(rng, n, la, mode), rand_rows(rng, n, lb, mode)
        want = oracle_mul(A, B)
        both(lambda: (device_mul(ctx, A, B, sa=la + 3, sb=lb + 1), device_mul(ctx, B, A, sc_extra=5)), (want, want))
        both(lambda: (device_mul(ctx, A, B, b_broadcast=True),), (oracle_mul(A, np.repeat(B[:1], n, axis=0)),))
        buf, va = g.upload_rows(A)
        if 2 * la <= K:
            bufc, vc = g.upload_rows(np.zeros((n, 2 * la), np.uint32))

            def square():
                g.check(ctx.mul(va, va, vc), "square")
                g.synchronize()
                return (g.download_rows(vc, bufc),)
            both(square, (oracle_mul(A, A),))
    la1, la2, lb = K // 4 + 5, K // 2 - 80, K // 4 + 77
    for n1, n2 in ((1, 1), (2, 1), (1, 2)):
        A1, A2, B = rand_rows(rng, n1, la1), rand_rows(rng, n2, la2), rand_rows(rng, max(n1, n2), lb)
        both(lambda: device_mul_shared(ctx, A1, A2, B), (oracle_mul(A1, B[:n1]), oracle_mul(A2, B[:n2])))
    for n in ((1 << 20 - k), (1 << 20 - k) + 1):
        A, B = rand_rows(rng, n, K // 2 - 1), rand_rows(rng, n, K // 2 - 4)
        both(lambda: (device_mul(ctx, A, B),), (oracle_mul(A, B),))


def test_truncated_transforms_in_ragged_calls(ctx):
    """Ragged rows of one transform size with different numbers of parts,
    some sharing an operand, with the pieces of unbalanced products."""
    rng = np.random.default_rng(16)
    K = 1 << 15
    lengths = [(K * t // 32 + d, K * t // 32) for t in range(9, 17) for d in (-1, 0)]
    lengths += [(K - 4000, 4000), (300, K - 301), (1 << 20, 5000), ((1 << 20) + 12345, 30000), (700000, 600000)]
    ops = [(rand_rows(rng, 1, a, "random")[0], rand_rows(rng, 1, b, "random")[0]) for a, b in lengths]
    shared = ops[3][1]
    ops += [(rand_rows(rng, 1, n, "random")[0], shared) for n in (K // 4 + 100, K // 2 - 1)]
    keep, items, outs = [], [], []
    sb = g.DeviceBuffer.from_array(shared)
    for a, b in ops:
        ba, bb = g.DeviceBuffer.from_array(a), sb if b is shared else g.DeviceBuffer.from_array(b)
        bc = g.DeviceBuffer(4 * (a.size + b.size))
        keep += [ba, bb]
        outs.append(bc)
        items.append((ba.ptr, bb.ptr, bc.ptr, a.size, b.size))
    g.check(ctx.mul_ragged(items), "mul_ragged")
    g.synchronize()
    for (a, b), bc in zip(ops, outs):
        want = oracle_mul(a.reshape(1, -1), b.reshape(1, -1))[0]
        assert np.array_equal(bc.download(np.uint32, count=want.size), want), (a.size, b.size)


@pytest.mark.parametrize("count", [3, 40, 300])
def test_ragged_small_products(ctx, count):
    """Ragged calls of products the matrix cores take (1..4088 limbs in all,
    every number of tile groups, one launch up to 256 of them and several
    above), with empty operands, tiny ones, a shared operand and products at
    the NTT's side of the limit, against Python integers."""
    rng = np.random.default_rng(count)
    lengths = [(1, 1), (0, 7), (5, 3000), (17, 17), (256, 257), (1016, 1016), (2044, 2044), (1016, 3072), (2045, 2044),
               (3900, 188), (4000, 3), (40, 4040), (1500, 1500), (700, 3300), (5000, 4000), (6000, 5)]
    while len(lengths) < count:
        lengths.append(tuple(int(2 ** u) for u in rng.uniform(0, 11, size=2)))
    lengths = lengths[:count] if count > 3 else [(300, 20), (1, 900), (4000, 88)]
    ops = []
    for i, (a, b) in enumerate(lengths):
        A, B = (rng.integers(0, 1 << 32, size=n, dtype=np.uint32) for n in (a, b))
        if i % 5 == 1:
            A[:] = 0x7F7F7F7F
        if i % 7 == 2:
            B[:] = 0xFFFFFFFF
        ops.append((A, ops[3][1] if i == 20 else B))
    keep, items, outs = [], [], []
    for A, B in ops:
        ba, bb = g.DeviceBuffer.from_array(A), g.DeviceBuffer.from_array(B)
        bc = g.DeviceBuffer.from_array(np.full(A.size + B.size + 1, PAD, dtype=np.uint32))
        keep += [ba, bb]
        outs.append(bc)
        items.append((ba.ptr, bb.ptr, bc.ptr, A.size, B.size))
    ctx.set_ntt_threshold(4089)
    try:
        g.check(ctx.mul_ragged(items), "mul_ragged")
        g.synchronize()
    finally:
        g.check(ctx.set_ntt_threshold(384))
    for (A, B), bc in zip(ops, outs):
        got = bc.download(np.uint32, count=A.size + B.size + 1)
        want = int.from_bytes(A.tobytes(), "little") * int.from_bytes(B.tobytes(), "little")
        assert int.from_bytes(got[:-1].tobytes(), "little") == want, (A.size, B.size)
        assert got[-1] == PAD, (A.size, B.size)


# p0 p1 / 2^80: the digits of 40 bits whose products' sums stay below p0 p1
P0P1 = ((1 << 49) - (1 << 30) + 1) * 0x1FFFE00000001
FORTY = P0P1 >> 80


@pytest.mark.parametrize("n,la,lb,mode", [
    (1, 4090, 7, "ones"), (1, 4096, 1, "random"), (2, 2049, 2049, "ones"), (3, 3276, 3277, "ones"),
    (1, 3277, 3277, "ones"), (1, 6553, 1, "ones"), (300, 3000, 3553, "random"), (300, 3001, 3553, "top"),
    (1, 20479, 20481, "ones"), (40, 20480, 20481, "ones"), (1, 163840, 163840, "ones"),
    # the longest operands of 40-bit digits, all of their bits set, and one limb more
    (1, FORTY * 40 // 32, FORTY * 40 // 32, "ones"), (1, FORTY * 40 // 32 + 1, FORTY * 40 // 32 + 1, "ones"),
    (1, 500000, FORTY * 40 // 32 - 1, "top"), (1, 1179647, 1179649, "ones"), (1, 1179649, 1179649, "ones"),
    (1, 4718593, 4718592, "random"),
])
def test_wide_digits(n, la, lb, mode):
    """Products with digits wider than a limb around the lengths where their
    number of bits or the transform changes, both ways round, padded rows, a
    square and a shared pair: GMP's product, and nothing past a row."""
    rng = np.random.default_rng(la * 3 + lb)
    with g.Context() as ctx:
        A, B = rand_rows(rng, n, la, mode), rand_rows(rng, n, lb, mode)
        want = oracle_mul(A, B)
        assert np.array_equal(device_mul(ctx, A, B, sa=la + 3, sb=lb + 1, sc_extra=5), want)
        assert np.array_equal(device_mul(ctx, B, A), want)
        if la < 200000:
            buf, va = g.upload_rows(A)
            bufc, vc = g.upload_rows(np.zeros((n, 2 * la), np.uint32))
            g.check(ctx.mul(va, va, vc), "square")
            g.synchronize()
            assert np.array_equal(g.download_rows(vc, bufc), oracle_mul(A, A))
            A2 = rand_rows(rng, n, max(1, la - la // 7), mode)
            got = device_mul_shared(ctx, A, A2, B)
            assert np.array_equal(got[0], want) and np.array_equal(got[1], oracle_mul(A2, B))
        # the same pairs as ragged rows
        outs, items = [], []
        bufs = [(g.DeviceBuffer.from_array(a), g.DeviceBuffer.from_array(b)) for a, b in zip(A[:5], B[:5])]
        for a, b in bufs:
            c = g.DeviceBuffer.from_array(np.full(la + lb + 1, PAD, dtype=np.uint32))
            outs.append(c)
            items.append((a.ptr, b.ptr, c.ptr, la, lb))
        g.check(ctx.mul_ragged(items), "mul_ragged")
        g.synchronize()
        for c, w in zip(outs, want):
            got = c.download(np.uint32, count=la + lb + 1)
            assert got[-1] == PAD and np.array_equal(got[:-1], w)


@pytest.mark.parametrize("seed,count,lo,hi", [(1, 12, 11.5, 17.0), (2, 5, 12.0, 19.5), (3, 40, 12.0, 14.0), (4, 9, 11.9, 20.5)])
def test_ragged_rows_of_several_sizes(ctx, seed, count, lo, hi):
    """Ragged pairs of few rows per transform size, which share launches, next
    to sizes of their own and unbalanced pairs in pieces: GMP's products."""
    rng = np.random.default_rng(seed)
    pairs, items = [], []
    for i in range(count):
        la, lb = (int(2.0 ** x) for x in rng.uniform(lo, hi, size=2))
        mode = ("random", "ones", "top")[i % 3]
        a, b = rand_rows(rng, 1, la, mode)[0], rand_rows(rng, 1, lb, mode)[0]
        bufs = (g.DeviceBuffer.from_array(a), g.DeviceBuffer.from_array(b),
                g.DeviceBuffer.from_array(np.full(la + lb + 1, PAD, dtype=np.uint32)))
        pairs.append((a, b, bufs))
        items.append((bufs[0].ptr, bufs[1].ptr, bufs[2].ptr, la, lb))
    g.check(ctx.mul_ragged(items), "mul_ragged")
    g.synchronize()
    for a, b, bufs in pairs:
        got = bufs[2].download(np.uint32, count=len(a) + len(b) + 1)
        assert got[-1] == PAD and np.array_equal(got[:-1], oracle_mul(a.reshape(1, -1), b.reshape(1, -1))[0])


@pytest.mark.parametrize("count", [2, 5, 168, 169, 400, 1200])
def test_small_ragged_calls_only_launch(count):
    """A ragged call of products below the NTT's threshold takes nothing of the
    context's workspace, and a capture of it replays on new operands (around
    the numbers of products that one launch's arguments hold, and above the
    number from which an eager call uploads a list)."""
    rng = np.random.default_rng(count)
    hip = g.hip()
    stream, graph, gexec = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    lengths = [(17, 17), (1, 4000), (2044, 2044)] + [tuple(int(2 ** u) for u in rng.uniform(0, 10.9, size=2))
                                                     for _ in range(count)]
    lengths = lengths[:count]
    at, items = [], []
    total = sum(2 * (a + b) for a, b in lengths)
    buf = g.DeviceBuffer(4 * total)
    word = 0
    for a, b in lengths:
        at.append(word)
        items.append((buf.ptr + 4 * word, buf.ptr + 4 * (word + a), buf.ptr + 4 * (word + a + b), a, b))
        word += 2 * (a + b)

    def fill():
        host = rng.integers(0, 1 << 32, size=total, dtype=np.uint32)
        g.check(hip.hipMemcpy(buf.ptr, host.ctypes.data, host.nbytes, 1), "hipMemcpy")
        return host

    def check(host):
        out = buf.download(np.uint32, count=total)
        for w, (a, b) in zip(at, lengths):
            x, y = (int.from_bytes(host[i:j].tobytes(), "little") for i, j in ((w, w + a), (w + a, w + a + b)))
            assert int.from_bytes(out[w + a + b:w + 2 * (a + b)].tobytes(), "little") == x * y, (a, b)

    with g.Context() as c:
        host = fill()
        g.check(c.mul_ragged(items), "mul_ragged")
        g.synchronize()
        check(host)
        assert c.workspace_size() == 0
        g.check(hip.hipStreamCreateWithFlags(ctypes.byref(stream), 1), "hipStreamCreateWithFlags")
        g.check(c.set_stream(stream), "set_stream")
        g.check(hip.hipStreamBeginCapture(stream, 1), "hipStreamBeginCapture")  # thread-local
        err = c.mul_ragged(items)
        g.check(hip.hipStreamEndCapture(stream, ctypes.byref(graph)), "hipStreamEndCapture")
        g.check(err, "mul_ragged under capture")
        g.check(hip.hipGraphInstantiate(ctypes.byref(gexec), graph, None, None, ctypes.c_size_t(0)), "instantiate")
        for _ in range(3):
            host = fill()
            g.check(hip.hipGraphLaunch(gexec, stream), "hipGraphLaunch")
            g.synchronize()
            check(host)
        g.check(hip.hipGraphExecDestroy(gexec), "hipGraphExecDestroy")
        g.check(hip.hipGraphDestroy(graph), "hipGraphDestroy")
        g.check(c.set_stream(None), "set_stream")
        g.check(hip.hipStreamDestroy(stream), "hipStreamDestroy")


@pytest.mark.parametrize("la,k", [(1100000, 21), (1500000, 22), (2700000, 23)])
def test_large_squares_run_whole(ctx, la, k):
    """A square takes one transform of its operand, at the size of the whole
    product, also where two different operands of its length run in pieces."""
    A = rand_rows(np.random.default_rng(la), 1, la)
    buf, va = g.upload_rows(A)
    bufc, vc = g.upload_rows(np.zeros((1, 2 * la), np.uint32))
    g.kernel_stats_reset(True)
    try:
        g.check(ctx.mul(va, va, vc), "square")
        g.synchronize()
        stats = {name: launches for name, launches, _, _ in g.kernel_stats(by_size=True)}
    finally:
        g.kernel_stats_reset(False)
    assert np.array_equal(g.download_rows(vc, bufc), oracle_mul(A, A))
    assert stats and all(name.endswith(f"@2^{k}") for name in stats), stats


def test_more_rows_than_one_launch_holds(ctx):
    """Matrix-core products of more rows than a launch's 2^32 threads cover
    (64 per row): the rows around the seam, the first and the last."""
    n, la, lb, seam = (1 << 26) + 77, 17, 18, (1 << 26) - 1
    rng = np.random.default_rng(26)
    A, B = rand_rows(rng, 1, la), rand_rows(rng, 1, lb)
    (ba, va), (bb, vb) = g.upload_rows(A), g.upload_rows(B)
    out = g.DeviceBuffer(4 * n * (la + lb))
    out.fill(0xAB)
    g.check(ctx.mul(va.view(batch_size=n, stride=0), vb.view(batch_size=n, stride=0),
                    g.BatchMPArray(out.ptr, la + lb, n, la + lb)), "mul")
    g.synchronize()
    want = oracle_mul(A, B)[0]
    for row in [0, 1, seam - 1, seam, seam + 1, n - 1] + [int(r) for r in rng.integers(0, n, size=50)]:
        assert np.array_equal(out.download(np.uint32, count=la + lb, offset_bytes=4 * row * (la + lb)), want), row


@pytest.mark.parametrize("n", [3, 16384, 20000])
@pytest.mark.parametrize("la,lb", [(127, 16), (128, 1), (129, 1), (129, 16), (380, 3), (1011, 12), (4087, 1), (4072, 16)])
def test_short_operand_against_long(n, la, lb):
    """Many and few rows of a short operand times a long one, around the
    lengths and the number of rows where the schoolbook kernels change or used
    to: GMP's products, and Python's for a row."""
    if n * (la + lb) > 1 << 25:
        n = (1 << 25) // (la + lb)
    rng = np.random.default_rng(la + lb)
    with g.Context() as c:
        A, B = rand_rows(rng, n, la, "ones"), rand_rows(rng, n, lb, "random")
        A[1::3] = rand_rows(rng, len(A[1::3]), la, "random")
        assert np.array_equal(device_mul(c, A, B, sa=la + 1, sb=lb + 2), oracle_mul(A, B))
        assert np.array_equal(device_mul(c, B, A), oracle_mul(B, A))
        assert to_int(device_mul(c, A[:1], B[:1])[0]) == to_int(A[0]) * to_int(B[0])


def test_short_operands_of_many_rows_take_the_matrix_cores():
    """Rows of a short operand against a long one take no longer in a batch of
    16384 than the same rows in calls of 8192 (a slower kernel for many rows
    took three to nineteen times as long)."""
    n, la, lb = 16384, 2000, 4
    rng = np.random.default_rng(5)
    with g.Context() as c:
        (ba, va), (bb, vb) = g.upload_rows(rand_rows(rng, n, la)), g.upload_rows(rand_rows(rng, n, lb))
        out = g.DeviceBuffer(4 * n * (la + lb))

        def parts(rows):
            for r in range(0, n, rows):
                g.check(c.mul(g.BatchMPArray(ba.ptr + 4 * r * la, la, rows, la),
                              g.BatchMPArray(bb.ptr + 4 * r * lb, lb, rows, lb),
                              g.BatchMPArray(out.ptr + 4 * r * (la + lb), la + lb, rows, la + lb)), "mul")

        def seconds(rows):
            best = 1e9
            for _ in range(5):
                g.synchronize()
                t0 = time.perf_counter()
                for _ in range(10):
                    parts(rows)
                g.synchronize()
                best = min(best, time.perf_counter() - t0)
            return best

        parts(n)
        assert seconds(n) < 2.0 * seconds(n // 2)


@pytest.mark.parametrize("n,la,lb,thin", [(1, 4096, 4095, True), (4, 100000, 90000, True), (200, 4096, 4095, False),
                                          (1, 1048576, 1000000, False)])
def test_kernel_statistics_name_the_kernels_that_ran(ctx, n, la, lb, thin):
    """Short launches' thin tiles have names of their own in the live
    statistics, one forward, row and inverse launch of each kind."""
    rng = np.random.default_rng(la)
    A, B = rand_rows(rng, n, la), rand_rows(rng, n, lb)
    g.kernel_stats_reset(True)
    try:
        assert np.array_equal(device_mul(ctx, A, B), oracle_mul(A, B))
        names = sorted(name for name, launches, *_ in g.kernel_stats() if launches == 1)
    finally:
        g.kernel_stats_reset(False)
    full = ["ntt_col_fwd_kernel<limbs>", "ntt_col_inv_limbs_kernel", "ntt_row_fused_kernel"]
    assert names == (["ntt_thin_fwd_kernel", "ntt_thin_inv_kernel", "ntt_thin_row_kernel"] if thin else full)


def digit_limbs(digits, bits):
    """The most limbs that make this many digits."""
    return digits * bits // 32


@pytest.mark.parametrize("k", [13, 14, 16, 18, 19, 20, 21, 22, 23])
def test_parts_of_truncated_transforms(ctx, k):
    """Products whose digits fill 10, 12, 14 or 16 parts of 2^k points exactly,
    one digit less and one more (and just over half of them), on full tiles of
    that size as the kernel statistics show: pairs of rows, a broadcast operand
    and a shared pair, against GMP; nothing is written past a row."""
    K, rng = 1 << k, np.random.default_rng(1000 + k)
    # digits of the shorter operand: 40 bits up to FORTY of them, else 36
    bits, short = (40, K // 8 - 3) if k <= 20 else (36, K // 6)
    totals = [K // 2 + 1] + [K * t // 16 + d for t in (10, 12, 14) for d in (-1, 0, 1)] + [K - 1, K]
    if k > 20:
        totals = totals[k % 2::2] + [K]
    # sizes set by hand (to the built-in ones) keep short launches on full tiles
    g.ntt_set_split(k, *(g.ntt_get_split(k)[:-1] if k < 20 else (0,)))
    try:
        for i, total in enumerate(totals):
            la, lb = digit_limbs(total - short, bits), digit_limbs(short, bits)
            A = rand_rows(rng, 2, la, ("random", "ones", "top")[i % 3])
            B = rand_rows(rng, 2, lb, ("ones", "random")[i % 2])
            g.kernel_stats_reset(True)
            assert np.array_equal(device_mul(ctx, A, B, sa=la + 1), oracle_mul(A, B)), total
            names = {name for name, *_ in g.kernel_stats(by_size=True)}
            g.kernel_stats_reset(False)
            assert names and all(n.endswith(f"@2^{k}") and "thin" not in n for n in names), (total, names)
            if i % 3 == 0:
                assert np.array_equal(device_mul(ctx, A, B, b_broadcast=True), oracle_mul(A, np.repeat(B[:1], 2, axis=0)))
                A2 = rand_rows(rng, 2, la - la // 9)
                got = device_mul_shared(ctx, A, A2, B)
                assert np.array_equal(got[0], oracle_mul(A, B)) and np.array_equal(got[1], oracle_mul(A2, B))
    finally:
        g.kernel_stats_reset(False)
        g.ntt_set_split(k, 0)


@pytest.mark.parametrize("k", [13, 15, 17])
def test_parts_of_ragged_rows(ctx, k):
    """One ragged launch of rows that fill different numbers of parts of 2^k
    points, each exactly, one digit less and one more, some sharing an operand."""
    K, rng = 1 << k, np.random.default_rng(2000 + k)
    short = K // 5
    shared = rand_rows(rng, 1, digit_limbs(short, 40))[0]
    sb = g.DeviceBuffer.from_array(shared)
    rows = []
    for i, total in enumerate([K // 2 + 1] * 9 + [K * t // 16 + d for t in (10, 12, 14) for d in (-1, 0, 1)] + [K]):
        a = rand_rows(rng, 1, digit_limbs(total - short, 40), ("random", "ones")[i % 2])[0]
        b = shared if i % 3 else rand_rows(rng, 1, digit_limbs(short, 40), "top")[0]
        rows.append((a, b, g.DeviceBuffer.from_array(a), sb if b is shared else g.DeviceBuffer.from_array(b),
                     g.DeviceBuffer.from_array(np.full(a.size + b.size + 1, PAD, dtype=np.uint32))))
    g.kernel_stats_reset(True)
    try:
        g.check(ctx.mul_ragged([(x.ptr, y.ptr, z.ptr, a.size, b.size) for a, b, x, y, z in rows]), "mul_ragged")
        g.synchronize()
        sizes = {name.split("@2^")[1] for name, *_ in g.kernel_stats(by_size=True)}
    finally:
        g.kernel_stats_reset(False)
    assert sizes == {str(k)}, sizes
    for a, b, _, _, z in rows:
        got = z.download(np.uint32, count=a.size + b.size + 1)
        assert got[-1] == PAD
        assert np.array_equal(got[:-1], oracle_mul(a.reshape(1, -1), b.reshape(1, -1))[0]), (a.size, b.size)


def test_every_tile_pairing_with_streamed_and_truncated_planes(ctx):
    """Two rows of 2^23 points whose planes go past the caches and fill 12 of
    16 parts: every tile pairing gives GMP's product."""
    rng = np.random.default_rng(23)
    la, lb = 3200000, 3500000
    A, B = rand_rows(rng, 2, la), rand_rows(rng, 2, lb, "ones")
    want = oracle_mul(A, B)
    (ba, va), (bb, vb) = g.upload_rows(A), g.upload_rows(B)
    bc, vc = g.upload_rows(np.zeros((2, la + lb), np.uint32))
    builtin = g.ntt_get_launch()
    try:
        for mask in range(16):
            g.ntt_set_launch(mask, builtin[1])
            bc.fill(0)
            g.kernel_stats_reset(True)
            g.check(ctx.mul(va, vb, vc), "mul")
            g.synchronize()
            sizes = {name.split("@2^")[1] for name, *_ in g.kernel_stats(by_size=True)}
            assert sizes == {"23"} and np.array_equal(g.download_rows(vc, bc), want), mask
    finally:
        g.kernel_stats_reset(False)
        g.ntt_set_launch(*builtin)


@pytest.mark.parametrize("leave", [384, 2, None])
def test_every_test_starts_at_the_shipped_crossover(ctx, leave):
    """The shared context sends the products to the NTT that a fresh one does,
    whatever the test before left behind: 4089 limbs in all and not 4088."""
    def ntt_kernels(c, total):
        A, B = (rand_rows(np.random.default_rng(total), 1, n) for n in (total // 2, total - total // 2))
        g.kernel_stats_reset(True)
        try:
            assert np.array_equal(device_mul(c, A, B), oracle_mul(A, B))
            return [name for name, *_ in g.kernel_stats()]
        finally:
            g.kernel_stats_reset(False)

    with g.Context() as fresh:
        for total in (500, DEFAULT_NTT_MIN_LIMBS - 1, DEFAULT_NTT_MIN_LIMBS, 5000):
            want = ntt_kernels(fresh, total)
            assert bool(want) == (total >= DEFAULT_NTT_MIN_LIMBS)
            assert ntt_kernels(ctx, total) == want, total
    if leave is not None:
        g.check(ctx.set_ntt_threshold(leave), "set_ntt_threshold")
