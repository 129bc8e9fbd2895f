"""scan! parity on the GPU: the HIP kernels (through the C ABI) against the
pinned CPU oracle. Integer scans are bit-exact; float max/min are exact (they
select an input); float + is checked against a Float64 host accumulation
with the tolerance stated per test."""
import zlib

import numpy as np
import pytest
import torch

from helpers import NP, assert_close, assert_mixed, dec, pow2_factors, product_rtol, q8_sequence

pytestmark = pytest.mark.gpu

EDGE = list(range(1, 11))
TILE_EDGES = [63, 64, 65, 255, 256, 257, 1023, 1024, 1025, 2047, 2048, 2049, 4095, 4096, 4097, 8191, 8192,
              8193, 16383, 16384, 16385, 32767, 32768, 32769, 131071, 131072, 131073, 65536 * 4 + 3]
SIZES = EDGE + TILE_EDGES + [100_003, 1_000_000]


def gen(rng, dt, n):
    if dt == np.int32:
        return rng.integers(1, 11, n).astype(np.int32)          # rand(1:10), reference scan_test.jl:51
    if dt == np.int64:
        return rng.integers(-4, 5, n).astype(np.int64)
    if dt == np.uint8:
        return rng.integers(0, 256, n).astype(np.uint8)
    return rng.random(n).astype(dt)


def run(kf, dev, x, op, f="identity", exclusive=False):
    fn = {"identity": kf.identity, "abs2": kf.abs2}[f]
    t = torch.from_numpy(x).to(dev)
    y = kf.scan(fn, op, t, exclusive=exclusive)
    torch.cuda.synchronize()
    return y.cpu().numpy()


@pytest.mark.parametrize("dt", [np.int32, np.int64, np.uint8])
@pytest.mark.parametrize("op", ["+", "max", "min"])
@pytest.mark.parametrize("exclusive", [False, True])
def test_int_scan_exact(kf, oracle, dev, dt, op, exclusive):
    rng = np.random.default_rng(zlib.crc32(f"{dt.__name__}{op}{exclusive}".encode()))
    for n in SIZES:
        x = gen(rng, dt, n)
        got = run(kf, dev, x, op, exclusive=exclusive)
        ref = oracle.scan(x, op, exclusive=exclusive)
        assert np.array_equal(got, ref), f"{dt.__name__} {op} excl={exclusive} n={n}: first diff at " \
            f"{np.nonzero(got != ref)[0][:1]}"


@pytest.mark.parametrize("dt", [np.int32, np.uint8])
def test_abs2_map_exact(kf, oracle, dev, dt):
    rng = np.random.default_rng(7)
    for n in (1, 5, 4097, 100_003):
        x = gen(rng, dt, n)
        for exclusive in (False, True):
            assert np.array_equal(run(kf, dev, x, "+", "abs2", exclusive), oracle.scan(x, "+", "abs2", exclusive))


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("op", ["max", "min"])
def test_float_minmax_exact(kf, oracle, dev, dt, op):
    rng = np.random.default_rng(11)
    for n in EDGE + [4097, 100_003]:
        x = (rng.random(n) - 0.5).astype(dt)
        for exclusive in (False, True):
            got = run(kf, dev, x, op, exclusive=exclusive)
            assert np.array_equal(got.astype(np.float64), oracle.scan(x, op, exclusive=exclusive))


def test_float_max_signed_zero_and_nan(kf, oracle, dev):
    x = np.array([0.0, -0.0, 1.0, np.nan, 2.0] * 1000, np.float32)
    for op in ("max", "min"):
        got = run(kf, dev, x, op)
        ref = oracle.scan(x, op)
        assert np.array_equal(np.isnan(got), np.isnan(ref))
        m = ~np.isnan(ref)
        assert np.array_equal(got[m], ref[m]) and np.array_equal(np.signbit(got[m]), np.signbit(ref[m]))


@pytest.mark.parametrize("dt,rtol", [(np.float32, 1e-5), (np.float64, 1e-12)])
def test_float_add_scan(kf, oracle, dev, dt, rtol):
    # U[0,1) inputs: every prefix is positive, so a relative tolerance applies
    rng = np.random.default_rng(13)
    for n in SIZES:
        x = rng.random(n).astype(dt)
        for exclusive in (False, True):
            got = run(kf, dev, x, "+", exclusive=exclusive)
            ref = oracle.scan(x, "+", exclusive=exclusive)
            assert_close(got, ref, rtol, atol=1e-30, what=f"{dt.__name__} + n={n} excl={exclusive}")
            if exclusive:
                assert got[0] == 0 and not np.signbit(got[0])


@pytest.mark.parametrize("dt", [np.int32, np.int64, np.uint8])
@pytest.mark.parametrize("exclusive", [False, True])
def test_int_product_scan_exact(kf, oracle, dev, dt, exclusive):
    # Julia `*` wraps on integers; odd factors never reach 0 modulo 2^bits,
    # so every prefix stays informative across all tile sizes
    rng = np.random.default_rng(zlib.crc32(f"mul{dt.__name__}{exclusive}".encode()))
    for n in SIZES:
        x = 2 * rng.integers(-3, 3, n) + 1
        x = (x % 256).astype(dt) if dt == np.uint8 else x.astype(dt)
        got = run(kf, dev, x, "*", exclusive=exclusive)
        ref = oracle.scan(x, "*", exclusive=exclusive)
        assert np.array_equal(got, ref), f"{dt.__name__} * excl={exclusive} n={n}: first diff at " \
            f"{np.nonzero(got != ref)[0][:1]}"


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_float_product_scan(kf, oracle, dev, dt):
    # exact: +-2 / +-1/2 factors (every prefix is a power of two), bit for bit;
    # rounded: factors in [0.999, 1.001] within the forward error bound
    # gamma_{i-1} of a product of i factors, whatever the association order
    rng = np.random.default_rng(19)
    for n in SIZES:
        x = pow2_factors(rng, n, dt)
        for exclusive in (False, True):
            got = run(kf, dev, x, "*", exclusive=exclusive)
            ref = oracle.scan(x, "*", exclusive=exclusive)
            assert np.array_equal(got.astype(np.float64), ref), f"{dt.__name__} * n={n} excl={exclusive}"
            if exclusive:
                assert got[0] == 1
        x = rng.uniform(0.999, 1.001, n).astype(dt)
        got = run(kf, dev, x, "*")
        assert_close(got, oracle.scan(x, "*"), product_rtol(dt, n), what=f"{dt.__name__} * n={n}")


def test_product_scan_reference_cases(kf, oracle, dev):
    # reference test/tests/scan/scan_test.jl:1-19: scan!(*, dst, src) on
    # Float32 U[0,1) at n = 10^7 and scan!(identity, *, dst, src) on Float64
    # at n = 1005, both against accumulate(*); the Float32 products underflow
    # within ~100 elements, hence the mixed criterion
    import operator
    rng = np.random.default_rng(20)
    x = rng.random(10**7).astype(np.float32)
    t = torch.from_numpy(x).to(dev)
    d = torch.zeros_like(t)
    kf.scan_(operator.mul, d, t)
    assert_mixed(d.cpu().numpy(), oracle.scan(x, "*"), 1e-5, what="scan!(*) Float32 10^7")
    y = rng.random(1005)
    t = torch.from_numpy(y).to(dev)
    d = torch.zeros_like(t)
    kf.scan_(kf.identity, operator.mul, d, t)
    assert_mixed(d.cpu().numpy(), oracle.scan(y, "*"), 1e-12, what="scan!(identity, *) Float64 1005")


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_quaternion_scan_q8_exact(kf, oracle, dev, dt):
    # random elements of the quaternion group {+-1, +-i, +-j, +-k}: every
    # product is exact and i j = -j i, so any reordered, dropped or repeated
    # factor shows bit for bit, at every tile shape
    import operator
    rng = np.random.default_rng(41)
    for n in SIZES:
        q = q8_sequence(rng, n, dt)
        t = torch.from_numpy(q).to(dev)
        for exclusive in (False, True):
            got = kf.scan(operator.mul, t, exclusive=exclusive).cpu().numpy()
            ref = oracle.scan(q, "*", exclusive=exclusive)
            assert np.array_equal(got.astype(np.float64), ref), f"{dt.__name__} n={n} excl={exclusive}: " \
                f"first diff at {np.nonzero((got != ref).any(1))[0][:1]}"
    # a strided view (every 3rd quaternion) takes the strided kernel, smallest tile
    q = q8_sequence(rng, 3 * 5001, dt)
    t = torch.from_numpy(q).to(dev)[::3]
    assert np.array_equal(kf.scan("*", t).cpu().numpy().astype(np.float64), oracle.scan(q[::3], "*"))


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_quaternion_scan_every_compiled_shape(kf, oracle, dev, dt):
    # the quaternion tiles (lane l holding units l*V .. l*V + V-1 of its
    # wave's chunk) at every compiled shape, around one tile and over more
    # tiles than the GPU holds at once; exact on the group {+-1, +-i, +-j, +-k}
    import operator
    probe = torch.from_numpy(q8_sequence(np.random.default_rng(0), 1, dt)).to(dev)
    shapes = sorted({kf.scan_shape(probe, "*", Nitem=v, workgroup=1024) for v in (1, 2, 4)})
    assert shapes == ([(1024, 1), (1024, 2), (1024, 4)] if dt == np.float32 else [(1024, 1), (1024, 2)])
    # and the wide shape large arrays take by default
    wide = (768, 8) if dt == np.float32 else (1024, 8)
    assert kf.scan_shape(probe, "*", Nitem=wide[1], workgroup=wide[0]) == wide
    if wide not in shapes:
        shapes.append(wide)
    rng = np.random.default_rng(47)
    for threads, items in shapes:
        tile = threads * items
        for n in (tile - 1, tile + 1, 2 * tile, 3 * tile + 5, 700 * tile + 7):
            q = q8_sequence(rng, n, dt)
            t = torch.from_numpy(q).to(dev)
            for exclusive in (False, True):
                got = kf.scan(operator.mul, t, exclusive=exclusive, Nitem=items, workgroup=threads).cpu().numpy()
                assert np.array_equal(got.astype(np.float64), oracle.scan(q, "*", exclusive=exclusive)), \
                    (threads, items, n, exclusive)


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_quaternion_scan_source_off_the_16_byte_grid(kf, oracle, dev, dt):
    # full tiles load their source striped and transpose it through LDS; a
    # source one component (4 or 8 bytes) off the 16-byte grid, with an
    # aligned destination, takes that path with unaligned 16-byte loads.
    # Exact on the group {+-1, +-i, +-j, +-k}; sizes over several wide tiles.
    import operator
    rng = np.random.default_rng(53)
    for n in (3 * 6144 + 5, 1_500_001):
        q = q8_sequence(rng, n, dt)
        flat = torch.zeros(4 * n + 4, dtype=torch.float32 if dt == np.float32 else torch.float64, device=dev)
        flat[1:1 + 4 * n] = torch.from_numpy(q.reshape(-1)).to(dev)
        src = flat[1:1 + 4 * n].view(n, 4)
        assert src.data_ptr() % 16 != 0
        for exclusive in (False, True):
            got = kf.scan(operator.mul, src, exclusive=exclusive).cpu().numpy()
            ref = oracle.scan(q, "*", exclusive=exclusive)
            assert np.array_equal(got.astype(np.float64), ref), (dt.__name__, n, exclusive)


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_quaternion_scan_destination_off_the_16_byte_grid(kf, oracle, dev, dt):
    # the tiles place 16-byte vectors on dst's grid: a destination one
    # component off it shifts every tile's virtual range (the first tile
    # partial), with the source aligned or off the grid by the same amount.
    # Exact on the group {+-1, +-i, +-j, +-k}; over several wide tiles
    # (8192-unit QuaternionF64 tiles, 6144-unit QuaternionF32 tiles).
    import operator
    tdt = torch.float32 if dt == np.float32 else torch.float64
    rng = np.random.default_rng(71)
    for n in (3 * 8192 + 7, 1_200_003):
        q = q8_sequence(rng, n, dt)
        for src_off in (0, 1):
            flat_s = torch.zeros(4 * n + 4, dtype=tdt, device=dev)
            flat_s[src_off:src_off + 4 * n] = torch.from_numpy(q.reshape(-1)).to(dev)
            src = flat_s[src_off:src_off + 4 * n].view(n, 4)
            flat_d = torch.zeros(4 * n + 4, dtype=tdt, device=dev)
            dst = flat_d[1:1 + 4 * n].view(n, 4)
            assert dst.data_ptr() % 16 != 0
            for exclusive in (False, True):
                kf.scan_(operator.mul, dst, src, exclusive=exclusive)
                ref = oracle.scan(q, "*", exclusive=exclusive)
                assert np.array_equal(dst.cpu().numpy().astype(np.float64), ref), (dt.__name__, n, src_off, exclusive)
                assert flat_d[0].item() == 0 and flat_d[-3:].abs().sum().item() == 0  # nothing stored outside


@pytest.mark.parametrize("dt,n", [(np.float64, 10**6), (np.float32, 10**4)])
def test_quaternion_scan_reference_case(kf, oracle, dev, dt, n):
    # reference test/tests/scan/scan_test.jl:22-33: scan!(identity, *, dst,
    # src) over 10^6 unit QuaternionF64 (normalised randn) against
    # accumulate(*). Bound: one Hamilton product of quaternions of norm ~1
    # adds at most gamma_4 * 2 <= 8u (normwise) and products by the identity
    # are exact, so output i (a product of i factors in some association) is
    # within 10 i u of the exact product.
    import operator
    rng = np.random.default_rng(43)
    x = rng.standard_normal((n, 4))
    q = (x / np.linalg.norm(x, axis=1, keepdims=True)).astype(dt)
    t = torch.from_numpy(q).to(dev)
    d = torch.zeros_like(t)
    kf.scan_(kf.identity, operator.mul, d, t)
    err = np.linalg.norm(d.cpu().numpy().astype(np.float64) - oracle.scan(q, "*"), axis=1)
    u = 2.0 ** -53 if dt == np.float64 else 2.0 ** -24
    bound = 10 * u * np.arange(1, n + 1)
    bad = np.nonzero(err > bound)[0]
    assert bad.size == 0, f"{bad.size} outside the bound; first at {bad[0]}: {err[bad[0]]} > {bound[bad[0]]}"


def test_golden_vectors(kf, dev, golden):
    for c in golden["scan"]:
        dt = NP[c["dtype"]]
        x = dec(c["x"], dt)
        for mode in ("inclusive", "exclusive"):
            got = run(kf, dev, x, c["op"], exclusive=mode == "exclusive")
            exp = dec(c[mode], np.float64 if dt == np.float64 else dt)
            if dt == np.float64 and c["op"] == "+":
                assert_close(got, exp, 1e-12, 1e-300, what=f"golden {c['op']} n={c['n']}")
            elif dt == np.float64:
                nan = np.isnan(exp)
                assert np.array_equal(np.isnan(got), nan)
                assert np.array_equal(got[~nan], exp[~nan])
            else:
                assert np.array_equal(got, exp), (c["dtype"], c["op"], c["n"], mode)


def test_affine_golden(kf, dev, golden):
    for c in golden["affine"]:
        ab = np.stack([dec(c["a"], np.float32), dec(c["b"], np.float32)], axis=1)
        for mode in ("inclusive", "exclusive"):
            got = kf.scan(kf.affine, torch.from_numpy(ab).to(dev), exclusive=mode == "exclusive").cpu().numpy()
            assert_mixed(got, np.array(c[mode]), 1e-5, what=f"affine golden n={c['n']} {mode}")


@pytest.mark.parametrize("n", EDGE + [2047, 2048, 2049, 100_003, 1 << 20])
def test_affine_scan(kf, oracle, dev, n):
    # BASELINE config 4 distribution: a ~ U[0.9, 1), b ~ N(0, 1); tolerance
    # |gpu - ref| <= 1e-5 * max(|ref|, 1) against the Float64 recurrence.
    rng = np.random.default_rng(n)
    ab = np.stack([rng.uniform(0.9, 1.0, n), rng.standard_normal(n)], 1).astype(np.float32)
    for exclusive in (False, True):
        got = kf.scan(kf.affine, torch.from_numpy(ab).to(dev), exclusive=exclusive).cpu().numpy()
        assert_mixed(got, oracle.scan(ab, "affine", exclusive=exclusive), 1e-5, what=f"affine n={n} excl={exclusive}")


@pytest.mark.parametrize("n", [(17 << 20) // 8 - 1, (17 << 20) // 8, 10**7 + 3])
def test_affine_scan_wide_tiles(kf, oracle, dev, n):
    # the affine pairs (8 bytes) switch from 1024 x 8-vector tiles to
    # 768 x 8-vector tiles at 17 MiB; 10^7 pairs give more tiles than the GPU
    # holds at once, so the windowed lookback runs as well
    rng = np.random.default_rng(n)
    ab = np.stack([rng.uniform(0.9, 1.0, n), rng.standard_normal(n)], 1).astype(np.float32)
    for exclusive in (False, True):
        got = kf.scan(kf.affine, torch.from_numpy(ab).to(dev), exclusive=exclusive).cpu().numpy()
        assert_mixed(got, oracle.scan(ab, "affine", exclusive=exclusive), 1e-5, what=f"affine n={n} excl={exclusive}")


def test_affine_is_order_sensitive(kf, oracle, dev):
    # a = 2 on even, 1/2 on odd positions with b = index: any reordering of
    # combines changes the result, exact in binary floating point
    n = 20000
    a = np.where(np.arange(n) % 2 == 0, 2.0, 0.5).astype(np.float32)
    b = (np.arange(n) % 7).astype(np.float32)
    ab = np.stack([a, b], 1)
    got = kf.scan(kf.affine, torch.from_numpy(ab).to(dev)).cpu().numpy()
    ref = oracle.scan(ab, "affine")
    assert np.array_equal(got[:, 0].astype(np.float64), ref[:, 0])
    assert_mixed(got, ref, 1e-6, what="alternating affine")


def test_reused_tmp_changing_data(kf, oracle, dev):
    # reference test/tests/scan/scan_test.jl:103-125: a stale descriptor from
    # the previous call would show up as an exact integer mismatch
    rng = np.random.default_rng(17)
    x0 = torch.zeros(1_000_000, dtype=torch.int32, device=dev)
    tmp = kf.get_allocation(kf.Scan1D, kf.identity, "+", x0)
    for call in range(12):
        n = [1_000_000, 1000, 100_000, 4097, 1_000_000, 65][call % 6]
        x = rng.integers(-4, 5, n).astype(np.int32)
        src = torch.from_numpy(x).to(dev)
        dst = torch.empty_like(src)
        kf.scan_("+", dst, src, tmp=tmp, exclusive=bool(call % 2))
        torch.cuda.synchronize()
        assert np.array_equal(dst.cpu().numpy(), oracle.scan(x, "+", exclusive=bool(call % 2))), call
    # the same buffer serves other element types and operators
    for dt in (np.int64, np.uint8):
        x = gen(rng, dt, 100_000)
        src = torch.from_numpy(x).to(dev)
        dst = torch.empty_like(src)
        kf.scan_("max", dst, src, tmp=tmp)
        assert np.array_equal(dst.cpu().numpy(), oracle.scan(x, "max"))
    # header word 1 is the lookback's give-up flag: never raised
    assert int(tmp.arr[8:16].cpu().numpy().view(np.uint64)[0]) == 0
    assert kf.scan_status(tmp) is False
    # the status query reads and clears the flag (set here from the host)
    tmp.arr[8] = 1
    assert kf.scan_status(tmp) is True
    assert kf.scan_status(tmp) is False
    with pytest.raises(kf.ArgumentError):
        kf.scan_status(kf.get_allocation(kf.MapReduce1D, kf.identity, "+", x0))


def test_views_offsets_strides_inplace(kf, oracle, dev):
    # reference test/tests/views/views_test.jl:1-42 (views of src/dst)
    rng = np.random.default_rng(19)
    n = 100_003
    x = rng.integers(0, 16, n).astype(np.int32)
    src = torch.from_numpy(x).to(dev)
    v = src[1:]                                       # view(src, 2:n): not 16-byte aligned
    out = kf.scan("+", v)
    assert np.array_equal(out.cpu().numpy(), oracle.scan(x[1:]))
    full = torch.zeros(n, dtype=torch.int32, device=dev)
    kf.scan_("+", full[2:], src[2:])                  # scan!(+, view(dst, 3:n), view(src, 3:n))
    got = full.cpu().numpy()
    assert np.array_equal(got[2:], oracle.scan(x[2:])) and np.all(got[:2] == 0)
    s = src[::3]                                      # strided source
    d = torch.zeros(2 * s.shape[0], dtype=torch.int32, device=dev)[::2]
    kf.scan_("+", d, s)
    assert np.array_equal(d.cpu().numpy(), oracle.scan(x[::3]))
    y = src.clone()                                   # in place
    kf.scan_("+", y, y)
    assert np.array_equal(y.cpu().numpy(), oracle.scan(x))


@pytest.mark.parametrize("dt", [np.float32, np.float64, np.int32, np.int64, np.uint8])
def test_tile_size_switchover(kf, oracle, dev, dt):
    # tiles are 1024 threads (512 for uint8; 768 x 8 vectors for 4- and
    # 8-byte types from 17 MiB on; uint8's own 12- and 16-vector shapes from 384 MiB and
    # 1 GiB are checked in test_gpu_large.py) x V 16-byte vectors, V in
    # (1, 2, 4, 8): the largest V that still makes >= 160 tiles (480 for
    # uint8), never below 2 except for uint8. The lookback polls 64 tiles
    # while every tile is resident, else 2, 4 or 8 by tile size (2 for
    # 128 KiB tiles from 4 generations on). Check both sides of every switch
    # (floats: sparse 0/1 values, so every partial sum is an integer and
    # exact in any order).
    epv = 16 // np.dtype(dt).itemsize
    block = {np.uint8: 512}.get(dt, 1024)
    min_tiles = 480 if dt == np.uint8 else 160
    rng = np.random.default_rng(23)
    edges = [min_tiles * block * v * epv for v in (2, 4, 8)] + [512 * block * 8 * epv]
    if dt != np.uint8:
        edges.append(4 * 512 * block * 8 * epv)        # window 2 from 4 generations of 128 KiB tiles
    if dt in (np.float32, np.float64, np.int32, np.int64):
        edges.append((17 << 20) // np.dtype(dt).itemsize)   # 768-thread tiles from 17 MiB on
    for e in edges:
        for n in (e - 1, e, e + 1):
            x = (rng.random(n) < 1 / 16).astype(dt) if np.dtype(dt).kind == "f" else gen(rng, dt, n)
            for exclusive in (False, True):
                assert np.array_equal(run(kf, dev, x, "+", exclusive=exclusive),
                                      oracle.scan(x, "+", exclusive=exclusive)), (n, exclusive)


@pytest.mark.parametrize("dt", [np.int32, np.int64, np.uint8])
def test_equally_misaligned_views_vector_path(kf, oracle, dev, dt):
    # src[k:] scanned into dst[k:]: both start k elements past a 16-byte
    # boundary, so the tile grid is shifted by k and interior tiles stay on
    # the vector path; results must be exact at every offset and size
    rng = np.random.default_rng(83)
    epv = 16 // np.dtype(dt).itemsize
    for n in (5, 4097, 8192 * 3 + 7, 512 * 32768 + 9, 1_000_003):
        x = gen(rng, dt, n + epv)
        src = torch.from_numpy(x).to(dev)
        for k in sorted({1, epv // 2, epv - 1}):
            for exclusive in (False, True):
                out = torch.zeros(n + epv, dtype=src.dtype, device=dev)
                kf.scan_("+", out[k:k + n], src[k:k + n], exclusive=exclusive)
                got = out.cpu().numpy()
                assert np.array_equal(got[k:k + n], oracle.scan(x[k:k + n], "+", exclusive=exclusive)), (n, k)
                assert not got[:k].any() and not got[k + n:].any()   # nothing written outside the view


def test_misaligned_affine_and_float(kf, oracle, dev):
    rng = np.random.default_rng(89)
    n = 300_001
    ab = np.stack([rng.uniform(0.9, 1.0, n + 1), rng.standard_normal(n + 1)], 1).astype(np.float32)
    t = torch.from_numpy(ab).to(dev)
    out = torch.zeros_like(t)
    kf.scan_(kf.affine, out[1:], t[1:])   # pairs offset by 8 bytes
    assert_mixed(out[1:].cpu().numpy(), oracle.scan(ab[1:], "affine"), 1e-5, what="misaligned affine")
    x = rng.random(n + 3)
    tx = torch.from_numpy(x).to(dev)
    y = torch.zeros_like(tx)
    kf.scan_("+", y[1:], tx[1:], exclusive=True)
    got = y[1:].cpu().numpy()
    assert got[0] == 0 and not np.signbit(got[0])
    assert_close(got, oracle.scan(x[1:], "+", exclusive=True), 1e-12, 1e-300, what="misaligned f64 excl")


def test_errors(kf, dev):
    a = torch.zeros(10, device=dev)
    with pytest.raises(kf.ArgumentError):
        kf.scan_("+", torch.zeros(9, device=dev), a)
    with pytest.raises(kf.ArgumentError):
        kf.scan_("+", torch.zeros(10, dtype=torch.float64, device=dev), a)
    with pytest.raises(kf.ArgumentError):
        kf.scan_("+", a[1:], a[:-1])  # partial overlap
    with pytest.raises(kf.ArgumentError):
        kf.scan(kf.affine, a)
    assert kf.scan("+", torch.zeros(0, device=dev)).numel() == 0


# ---- BASELINE.json configurations at full size -------------------------------
def test_config1_f32_inclusive_1e6(kf, oracle, dev):
    rng = np.random.default_rng(20261201 + 1)
    x = rng.random(10**6, dtype=np.float32)
    got = run(kf, dev, x, "+")
    assert_close(got, oracle.scan(x), 1e-5, what="config 1")  # rel tol 1e-5 vs Float64


@pytest.mark.parametrize("exclusive", [False, True])
def test_config2_int32_2pow28_exact(kf, oracle, dev, exclusive):
    rng = np.random.default_rng(20261201 + 2)
    n = 2**28
    x = rng.integers(0, 16, n, dtype=np.int32)
    print(f"config 2: Int32 n=2^28 exclusive={exclusive}", flush=True)
    got = run(kf, dev, x, "+", exclusive=exclusive)
    ref = oracle.scan(x, "+", exclusive=exclusive)
    assert np.array_equal(got, ref)
    # size-independent property: the last inclusive value is the total
    assert int(ref[-1]) + (int(x[-1]) if exclusive else 0) == int(x.sum(dtype=np.int64))


def test_config4_affine_2pow26(kf, oracle, dev):
    rng = np.random.default_rng(20261201 + 4)
    n = 2**26
    ab = np.empty((n, 2), np.float32)
    ab[:, 0] = rng.uniform(0.9, 1.0, n)
    ab[:, 1] = rng.standard_normal(n, dtype=np.float32)
    got = kf.scan(kf.affine, torch.from_numpy(ab).to(dev)).cpu().numpy()
    assert_mixed(got, oracle.scan(ab, "affine"), 1e-5, what="config 4")


def test_headline_f32_2pow28(kf, oracle, dev):
    # The bench workload, against the Float64 prefix sums. Bound per element:
    #   |y_i - s_i| <= lam * sqrt(D) * u * sum_{k<=i} |x_k|,   u = 2^-24,
    # the probabilistic rounding bound of Higham & Mary (SIAM J. Sci. Comput.
    # 41(5), 2019) for D roundings, with lam = 6 (each rounding set fails with
    # probability below 2e-8). Only the roundings of a running prefix are of
    # the size u * s_i; there are at most two per lookback hop (the window's
    # predecessor aggregates folded into the prefix found, then the tile's own
    # aggregate), and at most one hop per tile, so D = 2 * tiles; the tiles'
    # in-lane, wave and block sums round values a tile's total or smaller.
    # At 768 x 8 x 4 = 24576 elements per tile, 2^28 elements are 10923
    # tiles: bound 5.3e-5 relative. A dropped or doubled tile moves every
    # later prefix by about 12288 (a tile of U[0,1) values), which exceeds
    # the bound everywhere (at most 5.3e-5 * 1.34e8 = 7.1e3 at the end);
    # test_headline_exact_sparse checks the same size bit for bit.
    rng = np.random.default_rng(20261201 + 5)
    n = 2**28
    x = rng.random(n, dtype=np.float32)
    got = run(kf, dev, x, "+")
    ref = oracle.scan(x)                      # Float64, x >= 0: the sum of |x_k|
    tiles = -(-n // (768 * 8 * 4))
    bound = 6.0 * np.sqrt(2.0 * tiles) * 2.0**-24
    assert bound * ref[-1] < (768 * 8 * 4) * 0.5 * 0.999
    err = np.abs(got.astype(np.float64) - ref)
    worst = float(np.max(err / np.maximum(ref, 1.0)))
    print(f"headline F32 2^28: max relative error {worst:.3e}, bound {bound:.3e}", flush=True)
    assert np.all(err <= bound * np.maximum(ref, 1.0)), worst


def test_headline_exact_sparse(kf, oracle, dev):
    # 2^28 Float32 values in {0, 1} (one in 64): every prefix is an integer
    # below 2^24, so every rounding is exact and the scan must match the
    # integer prefix sums bit for bit; a wrong combine anywhere (a dropped,
    # doubled or reordered tile, window or row) is an integer mismatch
    rng = np.random.default_rng(20261201 + 6)
    n = 2**28
    x = (rng.random(n) < 2**-6).astype(np.float32)
    for exclusive in (False, True):
        got = run(kf, dev, x, "+", exclusive=exclusive)
        ref = np.cumsum(x, dtype=np.int64)
        if exclusive:
            ref = np.concatenate([[0], ref[:-1]])
        assert ref[-1] < 2**24
        assert np.array_equal(got.astype(np.int64), ref), exclusive


@pytest.mark.parametrize("exclusive", [False, True])
def test_post_map_g_in_the_store(kf, oracle, dev, exclusive):
    # reference src/scan/scan_kernel.jl:284-295: dst = g(prefix), g applied to
    # each stored value only (the running prefix stays un-mapped).
    # Integers: abs2 wraps, exact; floats: sqrt / abs2 of the Float64 prefix.
    rng = np.random.default_rng(131)
    for n in (1, 7, 4097, 100_003, 3 * 2**20 + 5):
        x = gen(rng, np.int32, n)
        src = torch.from_numpy(x).to(dev)
        ref = oracle.scan(x, "+", exclusive=exclusive).astype(np.uint32)
        got = kf.scan("+", src, exclusive=exclusive, g=kf.abs2).cpu().numpy()
        assert np.array_equal(got, (ref * ref).view(np.int32)), n
        # strided view: the strided kernel applies g the same way
        got = kf.scan("+", src[::2], exclusive=exclusive, g=kf.abs2).cpu().numpy()
        r2 = oracle.scan(x[::2], "+", exclusive=exclusive).astype(np.uint32)
        assert np.array_equal(got, (r2 * r2).view(np.int32)), n
        xf = rng.random(n).astype(np.float32)
        ref = oracle.scan(xf, "+", exclusive=exclusive)
        got = kf.scan("+", torch.from_numpy(xf).to(dev), exclusive=exclusive, g="sqrt").cpu().numpy()
        assert np.allclose(got, np.sqrt(ref), rtol=1e-5, atol=1e-6), n
        xd = rng.random(n)
        ref = oracle.scan(xd, "max", exclusive=exclusive)
        got = kf.scan("max", torch.from_numpy(xd).to(dev), exclusive=exclusive, g=kf.abs2).cpu().numpy()
        assert np.array_equal(got, ref * ref), n        # max selects an input: exact square
    with pytest.raises(kf.ArgumentError):
        kf.scan("+", torch.ones(10, dtype=torch.int32, device=dev), g="sqrt")


# ---- grids of 258..2049 resident tiles: the workgroup-wide lookback -----------
@pytest.mark.parametrize("dt,n", [(np.uint8, 3_000_007), (np.uint8, 10**7), (np.int32, 2_500_001),
                                  (np.int64, 10**6 + 3), (np.int64, 1_600_000), (np.float64, 2 * 10**6)])
def test_workgroup_wide_lookback(kf, oracle, dev, dt, n):
    rng = np.random.default_rng(n)
    x = gen(rng, dt, n)
    src = torch.from_numpy(x).to(dev)
    for excl in (False, True):
        got = kf.scan("+", src, exclusive=excl).cpu().numpy()
        ref = oracle.scan(x, "+", exclusive=excl)
        if dt == np.float64:
            assert np.allclose(got, ref, rtol=1e-12, atol=1e-9), (n, excl)
        else:
            assert np.array_equal(got, ref), (dt, n, excl)


@pytest.mark.parametrize("n", [10**6, 1_500_001])
def test_affine_workgroup_wide_lookback(kf, oracle, dev, n):
    # the affine pairs are not commutative: the waves' shares of the
    # predecessors must be combined in tile order
    rng = np.random.default_rng(n)
    ab = np.stack([rng.uniform(0.9, 1.0, n), rng.standard_normal(n)], 1).astype(np.float32)
    for exclusive in (False, True):
        got = kf.scan(kf.affine, torch.from_numpy(ab).to(dev), exclusive=exclusive).cpu().numpy()
        assert_mixed(got, oracle.scan(ab, "affine", exclusive=exclusive), 1e-5, what=f"affine n={n} excl={exclusive}")


# ---- source and destination misaligned differently ---------------------------
@pytest.mark.parametrize("dt", [np.int32, np.int64, np.uint8, np.float64])
def test_differently_misaligned_views(kf, oracle, dev, dt):
    # reference test/tests/views/views_test.jl:16-21 scans view(src, 2:n) into
    # a fresh dst: src and dst then sit at different offsets from a 16-byte
    # boundary, which the kernel streams with unaligned vector loads
    rng = np.random.default_rng(43)
    es = np.dtype(dt).itemsize
    for n in (5, 1000, 4097, 65536 * 4 + 3, 1_000_003):
        x = gen(rng, dt, n + 16)
        src = torch.from_numpy(x).to(dev)
        out = torch.empty(n + 16, dtype=src.dtype, device=dev)
        for si, di in ((1, 0), (0, 1), (3, 2), (16 // es - 1 if es < 16 else 0, 0), (2, 7)):
            if si + n > n + 16 or di + n > n + 16:
                continue
            d = out[di:di + n]
            kf.scan_("+" if dt != np.float64 else "max", d, src[si:si + n])
            ref = oracle.scan(x[si:si + n], "+" if dt != np.float64 else "max")
            assert np.array_equal(d.cpu().numpy(), ref), (n, si, di)


def test_misaligned_view_headline_size(kf, oracle, dev):
    # scan!(+, dst, src[2:end]) at 2^28 Float32 with an aligned dst: exact on
    # sparse 0/1 data (sums stay integers below 2^24)
    rng = np.random.default_rng(47)
    n = 2**28
    x = (rng.random(n + 1) < 2**-6).astype(np.float32)
    src = torch.from_numpy(x).to(dev)
    dst = torch.empty(n, dtype=torch.float32, device=dev)
    kf.scan_("+", dst, src[1:])
    got = dst.cpu().numpy()
    ref = np.cumsum(x[1:], dtype=np.float64)
    assert ref[-1] < 2**24
    assert np.array_equal(got.astype(np.float64), ref)


@pytest.mark.parametrize("dt", [np.int32, np.int64, np.uint8, np.float32, np.float64])
def test_launch_shape_keywords_every_compiled_shape(kf, oracle, dev, dt):
    # scan!(...; Nitem, workgroup) takes the nearest compiled tile shape;
    # run each shape of this element type at sizes around its tile and over
    # enough tiles to leave the all-resident lookback (floats: sparse 0/1
    # values, exact in any grouping)
    epv = 16 // np.dtype(dt).itemsize
    probe = torch.from_numpy(np.zeros(1, dt)).to(dev)
    shapes = sorted({kf.scan_shape(probe, "+", Nitem=epv * v, workgroup=b)
                     for b in (512, 768, 1024) for v in (1, 2, 4, 8, 12, 16)})
    want = {np.uint8: [(512, epv * v) for v in (1, 2, 4, 8, 12, 16)]}.get(
        dt, [(768, epv * 8)] + [(1024, epv * v) for v in (1, 2, 4, 8)])
    assert shapes == sorted(want)
    rng = np.random.default_rng(5)
    for threads, items in shapes:
        tile = threads * items
        for n in (1, tile - 1, tile + 1, 3 * tile + 5, 1200 * tile + 7):
            x = (rng.random(n) < 1 / 16).astype(dt) if np.dtype(dt).kind == "f" else gen(rng, dt, n)
            t = torch.from_numpy(x).to(dev)
            for exclusive in (False, True):
                y = kf.scan("+", t, exclusive=exclusive, Nitem=items, workgroup=threads)
                assert np.array_equal(y.cpu().numpy(), oracle.scan(x, "+", exclusive=exclusive)), \
                    (threads, items, n, exclusive)


def test_launch_shape_keywords_scratch(kf, oracle, dev):
    # get_allocation(Scan1D, f, op, src, workgroup, blocks) sizes for the
    # shape and tile count; a default-sized tmp is refused by a call whose
    # shape needs more tiles; the reference's get_allocation(..., blocks)
    rng = np.random.default_rng(6)
    n = 10**6
    x = gen(rng, np.int32, n)
    src = torch.from_numpy(x).to(dev)
    dst = torch.empty_like(src)
    small = kf.get_allocation(kf.Scan1D, kf.identity, "+", src)
    with pytest.raises(kf.ArgumentError, match="needs"):
        kf.scan_("+", dst, src, tmp=small, Nitem=4, workgroup=1024)
    tiles = -(-n // (1024 * 4))
    tmp = kf.get_allocation(kf.Scan1D, kf.identity, "+", src, 1024, tiles + 1)
    assert tmp.nbytes >= 256 + 128 * (tiles + 1)
    for _ in range(2):
        kf.scan_("+", dst, src, tmp=tmp, Nitem=4, workgroup=1024)
        assert np.array_equal(dst.cpu().numpy(), oracle.scan(x))
    big = kf.get_allocation(kf.Scan1D, kf.identity, "+", src, 100_000)
    assert big.nbytes >= 256 + 128 * 100_000
    kf.scan_("+", dst, src, tmp=big, Nitem=4)
    assert np.array_equal(dst.cpu().numpy(), oracle.scan(x))
    with pytest.raises(kf.ArgumentError, match="Nitem"):
        kf.scan_("+", dst, src, Nitem=0)
    with pytest.raises(kf.ArgumentError, match="unknown keyword"):
        kf.scan_("+", dst, src, Nitems=4)


@pytest.mark.parametrize("dt", [np.int32, np.int64, np.uint8, np.float32, np.float64])
@pytest.mark.parametrize("n", [1, 5, 1000, 8193, 100_003, 1_300_007, 6_000_001])
def test_strided_sources(kf, oracle, dev, dt, n):
    # a strided source into a contiguous, an offset and a strided destination:
    # interior tiles, boundary tiles (clamped loads) and every tile width that
    # n selects. Exact: integers, and max for the floats; the elements between
    # a strided destination's stay as they were.
    rng = np.random.default_rng(83)
    op = "max" if np.dtype(dt).kind == "f" else "+"
    for stride, off, exclusive in ((2, 0, False), (3, 1, True), (37, 0, False)):
        if n > 2_000_000 and stride == 37:
            continue
        x = gen(rng, dt, (n - 1) * stride + 1 + off)
        src = torch.from_numpy(x).to(dev)[off::stride]
        ref = oracle.scan(np.ascontiguousarray(x[off::stride]), op, exclusive=exclusive)
        out = torch.empty(n + 1, dtype=src.dtype, device=dev)
        for d in (out[:n], out[1:]):
            kf.scan_(op, d, src, exclusive=exclusive)
            assert np.array_equal(d.cpu().numpy(), ref), (n, stride, off)
        wide = torch.full((2 * n,), 7, dtype=src.dtype, device=dev)
        kf.scan_(op, wide[::2], src, exclusive=exclusive)
        assert np.array_equal(wide[::2].cpu().numpy(), ref) and bool((wide[1::2] == 7).all()), (n, stride)


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("n", [3, 4097, 500_003, 1_300_003])
def test_strided_quaternion_sources(kf, oracle, dev, dt, n):
    # every 2nd and 3rd quaternion through the transposed strided loads, at 2,
    # 4 and 8 quaternions a lane, into an aligned destination, one a
    # component off the 16-byte grid (element stores), and in place. Exact on
    # the group {+-1, +-i, +-j, +-k}, where any reordered factor shows.
    rng = np.random.default_rng(n)
    for stride, exclusive in ((2, False), (3, True)):
        q = q8_sequence(rng, (n - 1) * stride + 1, dt)
        t = torch.from_numpy(q).to(dev)
        ref = oracle.scan(q[::stride], "*", exclusive=exclusive)
        got = kf.scan("*", t[::stride], exclusive=exclusive)
        assert np.array_equal(got.cpu().numpy().astype(np.float64), ref), (stride, "aligned")
        off = torch.zeros(4 * n + 1, dtype=t.dtype, device=dev)[1:].view(n, 4)
        kf.scan_("*", off, t[::stride], exclusive=exclusive)
        assert np.array_equal(off.cpu().numpy().astype(np.float64), ref), (stride, "offset")
        kf.scan_("*", t[::stride], t[::stride], exclusive=exclusive)
        assert np.array_equal(t[::stride].cpu().numpy().astype(np.float64), ref), (stride, "in place")
        assert np.array_equal(t[1::stride].cpu().numpy(), q[1::stride]), stride


@pytest.mark.parametrize("n", [1, 2, 1025, 100_003, 1_000_001, 3_000_001])
def test_strided_affine_sources(kf, oracle, dev, n):
    # every 2nd, 3rd and 9th (a, b) pair into a contiguous, an 8-byte offset
    # and a strided destination, and in place, at every tile width. a = +-1
    # and small whole b: every composition is exact, and their order shows.
    rng = np.random.default_rng(n)
    for stride, exclusive in ((2, False), (3, True), (9, False)):
        m = (n - 1) * stride + 1
        ab = np.stack([rng.choice([1.0, -1.0], m), rng.integers(-3, 4, m)], 1).astype(np.float32)
        t = torch.from_numpy(ab).to(dev)
        ref = oracle.scan(ab[::stride], "affine", exclusive=exclusive)
        out = torch.empty(n + 1, 2, device=dev)
        for d in (out[:n], out[1:]):
            kf.scan_(kf.affine, d, t[::stride], exclusive=exclusive)
            assert np.array_equal(d.cpu().numpy().astype(np.float64), ref), stride
        wide = torch.full((2 * n, 2), 7.0, device=dev)
        kf.scan_(kf.affine, wide[::2], t[::stride], exclusive=exclusive)
        assert np.array_equal(wide[::2].cpu().numpy().astype(np.float64), ref) and bool((wide[1::2] == 7).all()), stride
        kf.scan_(kf.affine, t[::stride], t[::stride], exclusive=exclusive)
        assert np.array_equal(t[::stride].cpu().numpy().astype(np.float64), ref), (stride, "in place")


@pytest.mark.parametrize("dt", [np.int32, np.int64, np.uint8, np.float64])
@pytest.mark.parametrize("n", [5, 8193, 1_300_007, 6_000_001])
def test_strided_scans_in_place(kf, oracle, dev, dt, n):
    # source and destination the same strided view: each tile reads its
    # elements before it stores them, and boundary tiles drop what their
    # clamped loads read of others. Exact: integers, and max for the floats.
    rng = np.random.default_rng(n)
    op = "max" if np.dtype(dt).kind == "f" else "+"
    for stride, off, exclusive in ((2, 1, False), (3, 0, True)):
        x = gen(rng, dt, (n - 1) * stride + 1 + off)
        t = torch.from_numpy(x).to(dev)
        v = t[off::stride]
        kf.scan_(op, v, v, exclusive=exclusive)
        assert np.array_equal(v.cpu().numpy(), oracle.scan(np.ascontiguousarray(x[off::stride]), op, exclusive=exclusive))
        assert np.array_equal(t[off + 1::stride].cpu().numpy(), x[off + 1::stride])


@pytest.mark.parametrize("dt", [np.int32, np.int64, np.uint8, np.float32])
@pytest.mark.parametrize("n", [1, 17, 8193, 100_003, 1_300_007, 6_000_001])
def test_contiguous_sources_into_strided_destinations(kf, oracle, dev, dt, n):
    # a contiguous source of any alignment, mapped or not, into a strided
    # destination: vector loads in interior tiles, clamped ones at the ends.
    # Exact: integers, and max for the floats; the elements between the
    # destination's stay as they were.
    rng = np.random.default_rng(n)
    op, f = ("max", "identity") if dt == np.float32 else ("+", "abs2")
    x = gen(rng, dt, n + 3)
    t = torch.from_numpy(x).to(dev)
    for off, stride, exclusive in ((0, 2, False), (1, 3, True), (3, 2, False)):
        ref = oracle.scan(x[off:off + n], op, f, exclusive=exclusive)
        wide = torch.full((stride * n,), 7, dtype=t.dtype, device=dev)
        kf.scan_(kf.abs2 if f == "abs2" else kf.identity, op, wide[::stride], t[off:off + n], exclusive=exclusive)
        assert np.array_equal(wide[::stride].cpu().numpy(), ref.astype(dt)), (off, stride)
        assert bool((wide[1::stride] == 7).all())
