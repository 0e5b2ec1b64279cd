"""GPU parity: the hip engine's NTT and elementwise kernels against the oracle.

Mirrors modules/arith/c/test/test_ntt.c and test_mod.c (same sizes, prime
bit-widths and input formulas), calling through the C ABI, and adds the
benchmarked shapes (N = 2^12 .. 2^17, ~50-bit primes generated by Ring.gen_prime).
Every comparison is bit-exact.
"""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O
from vfhe_amd import runtime as rt

pytestmark = pytest.mark.gpu


def vp(a):
    return ctypes.c_void_p(a.ctypes.data)


def primes_for(n):
    ps = [int(O.lib().o_next_special_prime(1 << b, n, 1)) for b in (20, 30, 40, 50, 60, 62)]
    ps += [O.gen_prime(2 * n, 50), O.gen_prime(2 * n, 49)]
    return ps


@pytest.mark.parametrize("n", [16, 64, 256, 512, 1024, 2048, 4096, 8192, 16384, 32768, 65536, 131072])
def test_ntt_single_limb_matches_oracle(lib, n):
    """ntt_forward / ntt_reverse on host buffers (test_ntt.c:20-35), every prime width."""
    rng = np.random.default_rng(n)
    for q in primes_for(n):
        print(f"[ntt] n={n} q={q}", flush=True)
        proc = lib.ntt_new_proc(n, q)
        x = rng.integers(0, q, n, dtype=np.uint64)
        ref = x.copy()
        O.lib().o_ntt_forward(O.ptr(ref), n, q)
        fwd = np.zeros(n, dtype=np.uint64)
        lib.ntt_forward(vp(fwd), vp(x), proc)
        assert np.array_equal(fwd, ref), f"forward n={n} q={q}"
        back = np.zeros(n, dtype=np.uint64)
        lib.ntt_reverse(vp(back), vp(fwd), proc)
        assert np.array_equal(back, x), f"roundtrip n={n} q={q}"
        # inverse alone on arbitrary data
        y = rng.integers(0, q, n, dtype=np.uint64)
        refi = y.copy()
        O.lib().o_ntt_inverse(O.ptr(refi), n, q)
        inv = np.zeros(n, dtype=np.uint64)
        lib.ntt_reverse(vp(inv), vp(y), proc)
        assert np.array_equal(inv, refi), f"inverse n={n} q={q}"
        lib.ntt_free_proc(proc)


@pytest.mark.parametrize("N", [512, 1024, 2048, 4096])
def test_small_ntt_batch_register_kernel(lib, N):
    """k_ntt_small (whole transforms of 2^9..2^12 points in registers, 4096/N per workgroup)
    against the oracle and against the LDS radix-2 kernel (ntt.small = 0), on a batch whose row
    count leaves the last workgroup partly empty; the launch counter shows which kernel ran."""
    L, P = 3, 7   # 21 rows
    primes = O.gen_primes(N, [50, 49, 45])
    pool = rt.Pool(N, primes)
    octx = O.Ctx(N, primes)
    rng = np.random.default_rng(N + 5)
    xs = [rt.random_rows(rng, primes, N) for _ in range(P)]
    refs = []
    for x in xs:
        r = x.copy()
        octx.to_ntt(r, r, pool.full_mask())
        refs.append(r)
    saved = lib.vfhe_hip_get_option(b"ntt.small")
    try:
        for small in (1, 0):
            print(f"[small ntt] N={N} ntt.small={small}", flush=True)
            assert lib.vfhe_hip_set_option(b"ntt.small", small) == 0
            ps = [pool.poly(x) for x in xs]
            arr = rt._native.voidp_array(ps)
            n0 = lib.vfhe_hip_get_option(b"stat.ntt_small_launches")
            lib.vfhe_hip_ntt_batch(arr, P, 0)
            for p, r in zip(ps, refs):
                assert np.array_equal(pool.read(p), r), small
            lib.vfhe_hip_ntt_batch(arr, P, 1)
            for p, x in zip(ps, xs):
                assert np.array_equal(pool.read(p), x), small
            ran = lib.vfhe_hip_get_option(b"stat.ntt_small_launches") - n0
            assert (ran >= 2) if small else (ran == 0)
            for p in ps:
                pool.free(p)
    finally:
        lib.vfhe_hip_set_option(b"ntt.small", saved)


@pytest.mark.parametrize("per_cu_x2,small", [(0, False), (2, False), (3, False), (4, True)])
def test_integer_transforms_of_512_points(lib, cus, per_cu_x2, small):
    """Integer limbs at N = 512: few rows go to the radix-2 kernel (quicker there), more than 3 for 2 CUs to
    the register kernel, both directions against the oracle."""
    N, rows = 512, max(1, per_cu_x2 * cus // 2)
    primes = [int(O.lib().o_next_special_prime(1 << 60, N, 1))]
    pool, c, rng = rt.Pool(N, primes), O.Ctx(N, primes), np.random.default_rng(rows)
    xs = [rt.random_rows(rng, primes, N) for _ in range(rows)]
    ps = [pool.poly(x) for x in xs]
    arr = rt._native.voidp_array(ps)
    print(f"[512-point integer] rows={rows}", flush=True)
    n0 = lib.vfhe_hip_get_option(b"stat.ntt_small_launches")
    lib.vfhe_hip_ntt_batch(arr, rows, 0)
    for x, p in zip(xs, ps):
        ref = x.copy()
        c.to_ntt(ref, ref, 1)
        assert np.array_equal(pool.read(p), ref)
    lib.vfhe_hip_ntt_batch(arr, rows, 1)
    assert all(np.array_equal(pool.read(p), x) for p, x in zip(ps, xs))
    assert lib.vfhe_hip_get_option(b"stat.ntt_small_launches") - n0 == (2 if small else 0)
    for p in ps:
        pool.free(p)


def test_block_cache_cap_and_release(lib):
    """The device block cache keeps at most cache.max_mb parked, evicting the least recently parked
    blocks (results unchanged), and vfhe_hip_release_cached empties it."""
    saved = lib.vfhe_hip_get_option(b"cache.max_mb")
    N = 1 << 14
    primes = O.gen_primes(N, [50] * 6)
    pool = rt.Pool(N, primes)
    rng = np.random.default_rng(7)
    try:
        assert lib.vfhe_hip_set_option(b"cache.max_mb", 8) == 0
        for rows in (1, 3, 6, 2, 5):            # polynomials of several sizes: 128 KiB .. 768 KiB
            xs = [rt.random_rows(rng, primes[:rows], N) for _ in range(4)]
            sub = rt.Pool(N, primes[:rows])
            ps = [sub.poly(x) for x in xs]
            arr = rt._native.voidp_array(ps)
            lib.vfhe_hip_ntt_batch(arr, len(ps), 0)
            lib.vfhe_hip_ntt_batch(arr, len(ps), 1)
            for p, x in zip(ps, xs):
                assert np.array_equal(sub.read(p), x)
            for p in ps:
                sub.free(p)
            assert lib.vfhe_hip_get_option(b"stat.cache_parked_bytes") <= 8 << 20
        lib.vfhe_hip_synchronize()
        lib.vfhe_hip_release_cached()
        assert lib.vfhe_hip_get_option(b"stat.cache_parked_bytes") == 0
    finally:
        lib.vfhe_hip_set_option(b"cache.max_mb", saved)
    del pool


def test_ntt_and_eltwise_match_golden_vectors(lib):
    """The reference kernels' own outputs (tests/golden/ref_ntt_mod.npz) through the hip engine."""
    from conftest import golden_ntt_mod_cases
    for n, q, x, y, exp in golden_ntt_mod_cases():
        print(f"[golden] n={n} q={q}", flush=True)
        proc = lib.ntt_new_proc(n, q)
        out = np.zeros(n, dtype=np.uint64)
        lib.ntt_forward(vp(out), vp(x), proc)
        assert np.array_equal(out, exp["fwd"]), (n, q)
        lib.ntt_reverse(vp(out), vp(y), proc)
        assert np.array_equal(out, exp["rev"]), (n, q)
        for name in ("mul", "add", "sub"):
            getattr(lib, f"mod_eltwise_{name}")(vp(out), vp(x), vp(y), n, proc)
            assert np.array_equal(out, exp[name]), (name, n, q)
        lib.ntt_free_proc(proc)


def test_ntt_roundtrip_matrix_and_30bit(lib):
    """test_ntt.c:37-49: sizes {64..4096} x bits {20..62}, in[i] = (0x123456789ABCDEF + i) % q."""
    for n in (64, 256, 1024, 4096):
        qs = [int(lib.next_special_prime(1 << b, n, True)) for b in (20, 30, 40, 50, 60, 62)]
        if n == 1024:
            qs.append(1073643521)
        for q in qs:
            proc = lib.ntt_new_proc(n, q)
            x = np.array([(0x123456789ABCDEF + i) % q for i in range(n)], dtype=np.uint64)
            f = np.zeros(n, dtype=np.uint64)
            b = np.zeros(n, dtype=np.uint64)
            lib.ntt_forward(vp(f), vp(x), proc)
            lib.ntt_reverse(vp(b), vp(f), proc)
            assert np.array_equal(b, x)
            lib.ntt_free_proc(proc)


def negacyclic(a, b, q):
    n = len(a)
    out = [0] * n
    for i in range(n):
        ai = int(a[i])
        for j in range(n):
            p = ai * int(b[j]) % q
            k = i + j
            if k < n:
                out[k] = (out[k] + p) % q
            else:
                out[k - n] = (out[k - n] - p) % q
    return np.array(out, dtype=np.uint64)


def test_negacyclic_convolution(lib):
    """test_ntt.c:51-104: INTT(NTT(a) * NTT(b)) equals the schoolbook product."""
    for n in (64, 256):
        for b in (20, 40, 60, 62):
            q = int(lib.next_special_prime(1 << b, n, True))
            proc = lib.ntt_new_proc(n, q)
            a = np.array([(i + 123) % q for i in range(n)], dtype=np.uint64)
            bb = np.array([(2 * i + 456) % q for i in range(n)], dtype=np.uint64)
            na, nb, nr, res = (np.zeros(n, dtype=np.uint64) for _ in range(4))
            lib.ntt_forward(vp(na), vp(a), proc)
            lib.ntt_forward(vp(nb), vp(bb), proc)
            lib.mod_eltwise_mul(vp(nr), vp(na), vp(nb), n, proc)
            lib.ntt_reverse(vp(res), vp(nr), proc)
            assert np.array_equal(res, negacyclic(a, bb, q)), (n, q)
            lib.ntt_free_proc(proc)


@pytest.mark.parametrize("bits", [10, 20, 30, 40, 49, 50, 60, 62])
def test_mod_eltwise_sweep(lib, bits):
    """test_mod.c:89-185 inputs, every op, against the oracle's exact arithmetic."""
    n = 1024
    q = int(lib.next_special_prime(1 << bits, n, True)) if bits != 49 else O.gen_prime(2 * n, 50)
    proc = lib.ntt_new_proc(n, q)
    i = np.arange(n, dtype=np.uint64)
    in1 = ((np.uint64(0x123456789ABCDEF) ^ (i * np.uint64(0x1337BEEF))) % np.uint64(q)).astype(np.uint64)
    in2 = ((np.uint64(0xFEDCBA987654321) ^ (i * np.uint64(0xDEADBEEF))) % np.uint64(q)).astype(np.uint64)
    scale, scalar = 0x123456789ABCDEF, 0x9876543210ABCDEF

    def both(op, name, a, b=None, s=0, start=None):
        ref = np.zeros(n, dtype=np.uint64) if start is None else start.copy()
        out = np.zeros(n, dtype=np.uint64) if start is None else start.copy()
        O.lib().o_eltwise(op, O.ptr(ref), O.ptr(a), O.ptr(b if b is not None else a), s, n, q)
        f = getattr(lib, name)
        if name in ("mod_eltwise_scale", "mod_eltwise_fma", "mod_eltwise_add_scalar", "mod_eltwise_sub_scalar"):
            f(vp(out), vp(a), s, n, proc)
        elif b is not None:
            f(vp(out), vp(a), vp(b), n, proc)
        else:
            f(vp(out), vp(a), n, proc)
        assert np.array_equal(out, ref), (name, q)

    both(O.O_ADD, "mod_eltwise_add", in1, in2)
    both(O.O_SUB, "mod_eltwise_sub", in1, in2)
    both(O.O_MUL, "mod_eltwise_mul", in1, in2)
    both(O.O_SCALE, "mod_eltwise_scale", in1, s=scale)
    both(O.O_FMA, "mod_eltwise_fma", in1, s=scale, start=(i % np.uint64(q)).astype(np.uint64))
    both(O.O_MUL_ADDTO, "mod_eltwise_mul_addto", in1, in2, start=in2.copy())
    both(O.O_MUL_SUBTO, "mod_eltwise_mul_subto", in1, in2, start=in2.copy())
    both(O.O_ADD_SCALAR, "mod_eltwise_add_scalar", in1, s=scalar)
    both(O.O_SUB_SCALAR, "mod_eltwise_sub_scalar", in1, s=scalar)
    both(O.O_NEGATE, "mod_eltwise_negate", in1)
    large = (np.uint64(0xFFFFFFFFFFFFFFFF) ^ (i * np.uint64(0x12345678))).astype(np.uint64)
    both(O.O_REDUCE, "mod_eltwise_reduce", large)
    sig = np.array([0, -(2**63), -1, 1] + [(1 if k % 2 else -1) * k * 0x12345678 for k in range(4, n)], dtype=np.int64)
    sig_u = sig.view(np.uint64)
    both(O.O_REDUCE_SIGNED, "mod_eltwise_reduce_signed", sig_u)
    hi = (np.uint64(0xAAAAAAAAAAAAAAAA) ^ (i * np.uint64(0x11111111))).astype(np.uint64)
    lo = (np.uint64(0x5555555555555555) ^ (i * np.uint64(0x22222222))).astype(np.uint64)
    ref = np.zeros(n, dtype=np.uint64)
    O.lib().o_reduce_mp(O.ptr(ref), O.ptr(hi), O.ptr(lo), n, q)
    out = np.zeros(n, dtype=np.uint64)
    lib.mod_reduce_array_mp(vp(out), vp(hi), vp(lo), n, proc)
    assert np.array_equal(out, ref)
    lib.ntt_free_proc(proc)


@pytest.mark.parametrize("N,L,split", [(4096, 4, 1), (4096, 4, 4), (8192, 3, 1), (65536, 24, 1), (131072, 3, 1)])
def test_poly_domain_conversion(lib, N, L, split):
    """polynomial_RNSc_to_RNS / RNS_to_RNSc on masked multi-limb polynomials vs the oracle."""
    primes = O.gen_primes(N, [50] * L, split)
    pool = rt.Pool(N, primes, split)
    octx = O.Ctx(N, primes, split)
    rng = np.random.default_rng(N + L + split)
    mask = pool.full_mask() & ~0b10  # one inactive limb
    x = rt.random_rows(rng, primes, N, mask)
    p = pool.poly(x, mask)
    lib.polynomial_RNSc_to_RNS(p, p)
    ref = x.copy()
    octx.to_ntt(ref, ref, mask)
    got = pool.read(p)
    for i in range(L):
        if (mask >> i) & 1:
            assert np.array_equal(got[i], ref[i]), f"limb {i}"
    assert pool.mask(p) == mask
    lib.polynomial_RNS_to_RNSc(p, p)
    back = pool.read(p)
    for i in range(L):
        if (mask >> i) & 1:
            assert np.array_equal(back[i], x[i])
    pool.free(p)


def test_empty_batches_and_masks(lib):
    """Zero-length batches are no-ops, and a polynomial whose limb mask is empty passes through
    domain conversion and products untouched (the reference's per-limb loops run zero times,
    rns_polynomial.c:582-614); the product's mask is the intersection, here empty."""
    N, L = 4096, 3
    primes = O.gen_primes(N, [50] * L)
    pool = rt.Pool(N, primes)
    rng = np.random.default_rng(5)
    x = rt.random_rows(rng, primes, N)
    y = rt.random_rows(rng, primes, N)
    p = pool.poly(x)
    none = rt._native.voidp_array([])
    print("[empty] zero-length batches", flush=True)
    lib.vfhe_hip_ntt_batch(none, 0, 0)
    lib.vfhe_hip_ntt_batch(none, 0, 1)
    lib.vfhe_hip_ntt_mul_intt_batch(none, none, none, 0)
    assert np.array_equal(pool.read(p), x)
    print("[empty] empty limb mask", flush=True)
    e = pool.poly(y, 0)
    lib.polynomial_RNSc_to_RNS(e, e)
    lib.polynomial_RNS_to_RNSc(e, e)
    assert pool.mask(e) == 0 and np.array_equal(pool.read(e), y)
    out = pool.poly(None)
    lib.polynomial_mul_RNS_polynomial(out, p, e)
    assert pool.mask(out) == 0
    for h in (p, e, out):
        pool.free(h)


def test_batched_ntt_equals_per_poly(lib):
    """vfhe_hip_ntt_batch over 16 polynomials (N = 4096, 4 limbs: the smallest benchmarked batch) == one call per polynomial."""
    N, L, P = 4096, 4, 16
    primes = O.gen_primes(N, [50] * L)
    pool = rt.Pool(N, primes)
    octx = O.Ctx(N, primes)
    rng = np.random.default_rng(7)
    xs = [rt.random_rows(rng, primes, N) for _ in range(P)]
    a = [pool.poly(x) for x in xs]
    b = [pool.poly(x) for x in xs]
    lib.vfhe_hip_ntt_batch(rt._native.voidp_array(a), P, 0)
    for p in b:
        lib.polynomial_RNSc_to_RNS(p, p)
    for k in range(P):
        ref = xs[k].copy()
        octx.to_ntt(ref, ref, pool.full_mask())
        assert np.array_equal(pool.read(a[k]), ref)
        assert np.array_equal(pool.read(b[k]), ref)
    lib.vfhe_hip_ntt_batch(rt._native.voidp_array(a), P, 1)
    for k in range(P):
        assert np.array_equal(pool.read(a[k]), xs[k])
    for p in a + b:
        pool.free(p)


@pytest.mark.parametrize("N", [8192, 16384, 32768, 65536])
def test_ntt_schedules_agree(lib, N):
    """Every NTT schedule for N = 2^13..2^16 (two launches of the pipelined pass kernel, persistent or
    one tile per workgroup per pass, 256- or 512-thread column passes, or of the plain pass kernel,
    with and without sub-batching; the persistent per-XCD kernel at each occupancy and queue lag)
    matches the oracle bit for bit."""
    L, P = 3, 11   # 33 rows: uneven over the 8 XCD queues
    primes = O.gen_primes(N, [50] * L)
    pool = rt.Pool(N, primes)
    octx = O.Ctx(N, primes)
    rng = np.random.default_rng(N)
    xs = [rt.random_rows(rng, primes, N) for _ in range(P)]
    refs = []
    for x in xs:
        r = x.copy()
        octx.to_ntt(r, r, pool.full_mask())
        refs.append(r)
    print("xcd available:", lib.vfhe_hip_get_option(b"ntt.xcd_available"),
          [lib.vfhe_hip_get_option(f"probe.xcd{k}".encode()) for k in range(8)], flush=True)
    keys = (b"ntt.mode", b"ntt.chunk_mb", b"ntt.xcd_lag", b"ntt.xcd_occupancy", b"ntt.tile_grid", b"ntt.col_wide",
            b"ntt.xcd_l2")
    saved = {k: lib.vfhe_hip_get_option(k) for k in keys}
    # col_wide = 2 forces the 512-thread column instances at this small batch (33 rows would
    # otherwise stay below the two-workgroups-per-CU rule); the launch counter shows they ran
    # (the last column: the persistent kernel keeps its intermediate in the L2, 1, or streams it, 0)
    settings = [(2, 0, 3, 2, 15, 1, 1), (2, 0, 3, 2, 15, 2, 1), (2, 0, 3, 2, 0, 2, 1), (2, 0, 3, 2, 6, 0, 1),
                (2, 0, 3, 2, 0, 0, 1), (2, 4, 3, 2, 15, 2, 1), (0, 0, 3, 2, 6, 0, 1), (0, 4, 3, 2, 6, 0, 1),
                (1, 0, 0, 2, 6, 0, 1), (1, 0, 3, 2, 6, 0, 1), (1, 0, 6, 4, 6, 0, 1), (1, 0, 3, 2, 6, 0, 0),
                (1, 0, 2, 4, 6, 0, 0)]
    try:
        for setting in settings:
            print(f"[schedule] N={N} mode/chunk/lag/occ/tile_grid/col_wide/xcd_l2={setting}", flush=True)
            for k, v in zip(keys, setting):
                assert lib.vfhe_hip_set_option(k, v) == 0
            ps = [pool.poly(x) for x in xs]
            arr = rt._native.voidp_array(ps)
            wide0 = lib.vfhe_hip_get_option(b"stat.col_wide_launches")
            lib.vfhe_hip_ntt_batch(arr, P, 0)
            for p, r in zip(ps, refs):
                assert np.array_equal(pool.read(p), r), setting
            lib.vfhe_hip_ntt_batch(arr, P, 1)
            for p, x in zip(ps, xs):
                assert np.array_equal(pool.read(p), x), setting
            wide = lib.vfhe_hip_get_option(b"stat.col_wide_launches") - wide0
            if setting[0] == 2 and setting[5] == 2:
                assert wide >= 2, setting         # forward and inverse column passes ran 512-thread
            elif setting[5] == 0:
                assert wide == 0, setting
            for p in ps:
                pool.free(p)
    finally:
        for k, v in saved.items():
            lib.vfhe_hip_set_option(k, v)


@pytest.mark.parametrize("N,L,count", [(4096, 4, 16), (8192, 3, 4), (16384, 2, 3), (32768, 2, 3), (65536, 24, 2)])
def test_ntt_mul_intt_batch(lib, N, L, count):
    """z = INTT(NTT(x) * NTT(y)) (the fused product) against the oracle's NTT, product and inverse."""
    primes = O.gen_primes(N, [50] * L)
    pool = rt.Pool(N, primes)
    c = O.Ctx(N, primes)
    rng = np.random.default_rng(N + count)
    m = (1 << L) - 1
    xs = [rt.random_rows(rng, primes, N) for _ in range(count)]
    ys = [rt.random_rows(rng, primes, N) for _ in range(count)]
    px, py = [pool.poly(x) for x in xs], [pool.poly(y) for y in ys]
    pz = [pool.poly() for _ in range(count)]
    print(f"[fused product] N={N} L={L} count={count}", flush=True)
    lib.vfhe_hip_ntt_mul_intt_batch(rt._native.voidp_array(pz), rt._native.voidp_array(px),
                                    rt._native.voidp_array(py), count)
    for k in range(count):
        a, b, z = np.zeros_like(xs[k]), np.zeros_like(xs[k]), np.zeros_like(xs[k])
        c.to_ntt(a, xs[k], m)
        c.to_ntt(b, ys[k], m)
        c.mul(z, a, m, b, m, 0)
        c.to_coeff(z, z, m)
        assert np.array_equal(pool.read(pz[k]), z), k
        assert np.array_equal(pool.read(px[k]), xs[k]) and np.array_equal(pool.read(py[k]), ys[k])
    for p in px + py + pz:
        pool.free(p)


@pytest.mark.parametrize("N,widths,split", [
    (256, (50, 60), 1),                  # below the register sizes: separate transforms
    (512, (50,), 1), (512, (60, 49, 51), 1), (1024, (60,), 1), (2048, (50, 60), 1), (4096, (60, 50, 40), 1),
    (8192, (60,), 1), (16384, (60, 50), 1), (32768, (51, 60), 1), (65536, (60, 50), 1),
    (4096, (60, 62), 1), (8192, (62, 50), 1),   # a limb above 2^62: separate transforms
    (4096, (49, 60), 4),                 # split degree 4: the wrap-aware product
])
def test_ntt_mul_intt_prime_widths(lib, N, widths, split):
    """The product over every arithmetic and size class, limbs of one ring in different classes, an odd
    batch (the last workgroup of small rows partly empty), largest residues in one pair, a limb mask
    with a gap in another, against the oracle."""
    n2, primes = 2 * N // split, []
    for b in widths:   # above 2^50: the first prime past 2^b; else below
        q = int(O.lib().o_next_special_prime(1 << b, N // split, 1)) if b > 50 else O.gen_prime(n2, b, primes)
        primes.append(q)
    count, L = 3, len(primes)
    pool, c = rt.Pool(N, primes, split), O.Ctx(N, primes, split)
    rng = np.random.default_rng(N + sum(widths))
    masks = [(1 << L) - 1] * count
    xs = [rt.random_rows(rng, primes, N) for _ in range(count)]
    ys = [rt.random_rows(rng, primes, N) for _ in range(count)]
    for i, q in enumerate(primes):
        xs[1][i], ys[1][i] = q - 1, q - 1
    if L > 2:
        masks[2] = 0b101
    px = [pool.poly(x, m) for x, m in zip(xs, masks)]
    py, pz = [pool.poly(y) for y in ys], [pool.poly() for _ in range(count)]
    print(f"[product] N={N} widths={widths} split={split}", flush=True)
    lib.vfhe_hip_ntt_mul_intt_batch(rt._native.voidp_array(pz), rt._native.voidp_array(px),
                                    rt._native.voidp_array(py), count)
    for k in range(count):
        a, b, z = np.zeros_like(xs[k]), np.zeros_like(xs[k]), np.zeros_like(xs[k])
        c.to_ntt(a, xs[k], masks[k])
        c.to_ntt(b, ys[k], masks[k])
        c.mul(z, a, masks[k], b, masks[k], 0)
        c.to_coeff(z, z, masks[k])
        assert pool.mask(pz[k]) == masks[k]
        got = pool.read(pz[k])
        for i in range(L):
            if (masks[k] >> i) & 1:
                assert np.array_equal(got[i], z[i]), (k, i)
    for p in px + py + pz:
        pool.free(p)


@pytest.mark.parametrize("split", [1, 2, 4, 8])
@pytest.mark.parametrize("rows", [1, 16, 17, 32, 33, 64, 65])
def test_work_lists_by_length(lib, rows, split):
    """Transforms, products and wrap-aware products whose row lists are just within and just past the
    sizes passed in kernel arguments, limbs of both arithmetics, against the oracle (exact)."""
    N, L = 512 * split, 2 if rows % 2 == 0 else 1
    count, primes = rows // L, []
    for b in (50, 60)[:L]:
        primes.append(int(O.lib().o_next_special_prime(1 << b, 512, 1)) if b > 50
                      else O.gen_prime(2 * N // split, b, primes))
    pool, c, m = rt.Pool(N, primes, split), O.Ctx(N, primes, split), (1 << L) - 1
    rng = np.random.default_rng(rows * 8 + split)
    print(f"[lists] rows={rows} split={split}", flush=True)
    xs = [rt.random_rows(rng, primes, N) for _ in range(count)]
    ys = [rt.random_rows(rng, primes, N) for _ in range(count)]
    px, py = [pool.poly(x) for x in xs], [pool.poly(y) for y in ys]
    pz = [pool.poly() for _ in range(count)]
    arr = rt._native.voidp_array
    lib.vfhe_hip_ntt_mul_intt_batch(arr(pz), arr(px), arr(py), count)
    lib.vfhe_hip_ntt_batch(arr(px), count, 0)
    lib.vfhe_hip_ntt_batch(arr(py), count, 0)
    for k in range(count):
        a, b, z = np.zeros_like(xs[k]), np.zeros_like(xs[k]), np.zeros_like(xs[k])
        c.to_ntt(a, xs[k], m)
        c.to_ntt(b, ys[k], m)
        c.mul(z, a, m, b, m, 0)
        assert np.array_equal(pool.read(px[k]), a), k
        for mode, fn in enumerate((lib.polynomial_mul_RNS_polynomial, lib.polynomial_mul_addto_RNS_polynomial,
                                   lib.polynomial_mul_subto_RNS_polynomial)):
            if k or split == 1:   # one polynomial is enough for the single products
                break
            out, ref = pool.poly(xs[0]), xs[0].copy()
            fn(out, px[0], py[0])
            c.mul(ref, a, m, b, m, mode)
            assert np.array_equal(pool.read(out), ref), mode
            pool.free(out)
        c.to_coeff(z, z, m)
        assert np.array_equal(pool.read(pz[k]), z), k
    lib.vfhe_hip_ntt_batch(arr(px), count, 1)
    assert all(np.array_equal(pool.read(p), x) for p, x in zip(px, xs))
    for p in px + py + pz:
        pool.free(p)


@pytest.mark.parametrize("rows", [1, 31, 32, 33])
def test_two_pass_lists_by_length(lib, rows):
    """Two-pass transforms (N = 8192) of row lists just within and past the 32 rows passed in kernel
    arguments, both directions, against the oracle (exact)."""
    N = 8192
    primes = O.gen_primes(N, [50])
    pool, c, rng = rt.Pool(N, primes), O.Ctx(N, primes), np.random.default_rng(rows)
    print(f"[lists] two passes, rows={rows}", flush=True)
    xs = [rt.random_rows(rng, primes, N) for _ in range(rows)]
    ps = [pool.poly(x) for x in xs]
    lib.vfhe_hip_ntt_batch(rt._native.voidp_array(ps), rows, 0)
    for p, x in zip(ps, xs):
        ref = np.zeros_like(x)
        c.to_ntt(ref, x, 1)
        assert np.array_equal(pool.read(p), ref)
    lib.vfhe_hip_ntt_batch(rt._native.voidp_array(ps), rows, 1)
    for p, x in zip(ps, xs):
        assert np.array_equal(pool.read(p), x)
        pool.free(p)


@pytest.mark.slow
def test_ntt_mul_intt_batch64_config2(lib):
    """The benchmarked fused-product batch: 64 pairs at N = 2^16, L = 24 in one call.  Every product
    equals the same pair computed alone (a batch of one), and two pairs -- the first and the last --
    equal the oracle's NTT, pointwise product and inverse bit for bit."""
    import concurrent.futures as cf
    N, L, count = 65536, 24, 64
    primes = O.gen_primes(N, [50] * L)
    pool = rt.Pool(N, primes)
    c = O.Ctx(N, primes)
    rng = np.random.default_rng(6464)
    m = (1 << L) - 1
    xs = [rt.random_rows(rng, primes, N) for _ in range(count)]
    ys = [rt.random_rows(rng, primes, N) for _ in range(count)]
    px, py = [pool.poly(x) for x in xs], [pool.poly(y) for y in ys]
    pz = [pool.poly() for _ in range(count)]

    def oracle_product(k):
        a, b, z = np.zeros_like(xs[k]), np.zeros_like(xs[k]), np.zeros_like(xs[k])
        c.to_ntt(a, xs[k], m)
        c.to_ntt(b, ys[k], m)
        c.mul(z, a, m, b, m, 0)
        c.to_coeff(z, z, m)
        return z

    print(f"[fused product] N={N} L={L} count={count}", flush=True)
    lib.vfhe_hip_ntt_mul_intt_batch(rt._native.voidp_array(pz), rt._native.voidp_array(px),
                                    rt._native.voidp_array(py), count)
    with cf.ThreadPoolExecutor(2) as ex:
        futs = {k: ex.submit(oracle_product, k) for k in (0, count - 1)}
        one = pool.poly()
        for k in range(count):
            lib.vfhe_hip_ntt_mul_intt_batch(rt._native.voidp_array([one]), rt._native.voidp_array([px[k]]),
                                            rt._native.voidp_array([py[k]]), 1)
            assert np.array_equal(pool.read(pz[k]), pool.read(one)), k
        for k, f in futs.items():
            assert np.array_equal(pool.read(pz[k]), f.result()), k
    for p in px + py + pz + [one]:
        pool.free(p)


@pytest.mark.parametrize("N", [16384, 65536])
def test_ntt_mul_intt_ragged_masks(lib, N):
    """The fused product over pairs with different limb masks: z takes the common limbs
    (rns_mask of x AND y) and each of them matches the oracle; items of a batch mix limbs."""
    L = 5
    primes = O.gen_primes(N, [50] * L)
    pool = rt.Pool(N, primes)
    c = O.Ctx(N, primes)
    rng = np.random.default_rng(N + 7)
    mx = [0b11111, 0b10101, 0b01110, 0b00001]
    my = [0b11111, 0b11100, 0b01111, 0b10001]
    xs = [rt.random_rows(rng, primes, N) for _ in mx]
    ys = [rt.random_rows(rng, primes, N) for _ in my]
    px = [pool.poly(x, m) for x, m in zip(xs, mx)]
    py = [pool.poly(y, m) for y, m in zip(ys, my)]
    pz = [pool.poly() for _ in mx]
    print(f"[fused product, ragged masks] N={N}", flush=True)
    lib.vfhe_hip_ntt_mul_intt_batch(rt._native.voidp_array(pz), rt._native.voidp_array(px),
                                    rt._native.voidp_array(py), len(mx))
    for k in range(len(mx)):
        m = mx[k] & my[k]
        assert pool.mask(pz[k]) == m
        a, b, z = np.zeros_like(xs[k]), np.zeros_like(xs[k]), np.zeros_like(xs[k])
        c.to_ntt(a, xs[k], m)
        c.to_ntt(b, ys[k], m)
        c.mul(z, a, m, b, m, 0)
        c.to_coeff(z, z, m)
        got = pool.read(pz[k])
        for li in range(L):
            if (m >> li) & 1:
                assert np.array_equal(got[li], z[li]), (k, li)
    for p in px + py + pz:
        pool.free(p)


@pytest.mark.parametrize("split", [2, 4])
def test_split_products_bound_their_temporaries(lib, split):
    """A batch of products on a split ring holds no more temporary memory than its y operands and one pair
    more (what the engine parks afterwards), and every product equals the one of its pair alone."""
    N, L, count = 65536, 11, 13
    primes = O.gen_primes(N, [50] * L, split)
    pool = rt.Pool(N, primes, split)
    rng = np.random.default_rng(split)
    x, y, z, one = ([pool.poly() for _ in range(count)] for _ in range(4))
    for p in x + y:
        pool.write(p, rt.random_rows(rng, primes, N))
    arr = rt._native.voidp_array
    lib.vfhe_hip_ntt_batch(arr(x + y), 2 * count, 0)   # operands on the device
    lib.vfhe_hip_release_cached()
    print(f"[split products] S={split}", flush=True)
    lib.vfhe_hip_ntt_mul_intt_batch(arr(z), arr(x), arr(y), count)
    assert 0 < lib.vfhe_hip_get_option(b"stat.cache_parked_bytes") <= (count + 1) * L * N * 8 + (1 << 20)
    for k in range(count):
        lib.vfhe_hip_ntt_mul_intt_batch(arr([one[k]]), arr([x[k]]), arr([y[k]]), 1)
        assert np.array_equal(pool.read(z[k]), pool.read(one[k])), k
    for p in x + y + z + one:
        pool.free(p)


@pytest.mark.parametrize("N", [8192, 16384, 32768, 65536])
@pytest.mark.parametrize("tile_grid,col_wide", [(0, 0), (31, 2), (16, 0), (15, 2)])
def test_ntt_mul_intt_grid_shapes(lib, N, tile_grid, col_wide):
    """The fused product under each grid shape of its three launches (persistent or one tile per
    workgroup, 256- or 512-thread column passes; col_wide = 2 forces the 512-thread instances at this
    batch size and the launch counter shows they ran) matches the oracle bit for bit."""
    L, count = 3, 5
    primes = O.gen_primes(N, [50] * L)
    pool = rt.Pool(N, primes)
    c = O.Ctx(N, primes)
    rng = np.random.default_rng(tile_grid * 7 + col_wide)
    m = (1 << L) - 1
    keys = (b"ntt.tile_grid", b"ntt.col_wide")
    saved = {k: lib.vfhe_hip_get_option(k) for k in keys}
    try:
        for k, v in zip(keys, (tile_grid, col_wide)):
            assert lib.vfhe_hip_set_option(k, v) == 0
        xs = [rt.random_rows(rng, primes, N) for _ in range(count)]
        ys = [rt.random_rows(rng, primes, N) for _ in range(count)]
        px, py = [pool.poly(x) for x in xs], [pool.poly(y) for y in ys]
        pz = [pool.poly() for _ in range(count)]
        print(f"[fused product] N={N} tile_grid={tile_grid} col_wide={col_wide}", flush=True)
        wide0 = lib.vfhe_hip_get_option(b"stat.col_wide_launches")
        lib.vfhe_hip_ntt_mul_intt_batch(rt._native.voidp_array(pz), rt._native.voidp_array(px),
                                        rt._native.voidp_array(py), count)
        wide = lib.vfhe_hip_get_option(b"stat.col_wide_launches") - wide0
        assert (wide >= 2) if col_wide == 2 else (wide == 0)
        for k in range(count):
            a, b, z = np.zeros_like(xs[k]), np.zeros_like(xs[k]), np.zeros_like(xs[k])
            c.to_ntt(a, xs[k], m)
            c.to_ntt(b, ys[k], m)
            c.mul(z, a, m, b, m, 0)
            c.to_coeff(z, z, m)
            assert np.array_equal(pool.read(pz[k]), z), k
        for p in px + py + pz:
            pool.free(p)
    finally:
        for k, v in saved.items():
            lib.vfhe_hip_set_option(k, v)


def test_autotune_picks_a_schedule_and_stays_exact(lib):
    """The NTT schedule autotuner times every candidate and leaves a schedule that is still bit-exact."""
    import ctypes
    N = 8192
    primes = O.gen_primes(N, [50] * 4)
    pool = rt.Pool(N, primes)
    us = (ctypes.c_double * 9)()
    saved = {k: lib.vfhe_hip_get_option(k)
             for k in (b"ntt.mode", b"ntt.chunk_mb", b"ntt.xcd_lag", b"ntt.xcd_occupancy", b"ntt.tile_grid",
                       b"ntt.col_wide")}
    try:
        best = lib.vfhe_hip_autotune_ntt(pool.h, 64, 2, us)
        assert 0 <= best < 9 and us[best] > 0
        assert all(us[k] > 0 for k in range(6))               # the two-launch candidates always run
        assert all(us[best] <= x for x in us if x > 0)
        x = rt.random_rows(np.random.default_rng(1), primes, N)
        p = pool.poly(x)
        lib.vfhe_hip_ntt_batch(rt._native.voidp_array([p]), 1, 0)
        ref = x.copy()
        for i, q in enumerate(primes):
            O.lib().o_ntt_forward(O.ptr(ref[i]), N, q)
        assert np.array_equal(pool.read(p), ref)
        pool.free(p)
    finally:
        for k, v in saved.items():
            lib.vfhe_hip_set_option(k, v)


def test_mul_modq_against_bigint(lib):
    """mul_modq (mod.c:64-67): a*b mod q through an NTT_proc, every prime width, edge values."""
    import random
    rnd = random.Random(64)
    for q in primes_for(1024):
        proc = lib.ntt_new_proc(1024, q)
        vals = [0, 1, q - 1, q // 2] + [rnd.randrange(q) for _ in range(300)]
        for a in vals:
            b = rnd.choice(vals)
            assert lib.mul_modq(a, b, proc) == (a * b) % q, (q, a, b)
        lib.ntt_free_proc(proc)


def test_product_autotuner_adopts_a_timed_schedule(lib):
    """vfhe_hip_autotune_product times its three schedules (two candidate indexes each), adopts the fastest
    (ntt.col_wide; ntt.tile_grid stays), and the fused product afterwards equals the oracle."""
    N, L, P = 16384, 3, 4
    primes = O.gen_primes(N, [50] * L)
    pool = rt.Pool(N, primes)
    octx = O.Ctx(N, primes)
    rng = np.random.default_rng(33)
    xs = [rt.random_rows(rng, primes, N) for _ in range(P)]
    ys = [rt.random_rows(rng, primes, N) for _ in range(P)]
    px, py, pz = [pool.poly(x) for x in xs], [pool.poly(y) for y in ys], [pool.poly() for _ in range(P)]
    ax, ay, az = (rt._native.voidp_array(v) for v in (px, py, pz))
    keys = (b"ntt.tile_grid", b"ntt.col_wide", b"ntt.mode")
    before = {k: lib.vfhe_hip_get_option(k) for k in keys}
    us = (ctypes.c_double * 6)()
    try:
        best = lib.vfhe_hip_autotune_product(az, ax, ay, P, 2, us)
        print("[autotune product] best", best, [round(u, 1) for u in us], flush=True)
        assert 0 <= best < 6 and all(u > 0 for u in us)
        assert lib.vfhe_hip_get_option(b"ntt.col_wide") == best >> 1
        assert (lib.vfhe_hip_get_option(b"ntt.tile_grid") >> 4) & 1 == (0 if best & 1 else 1)
        assert lib.vfhe_hip_get_option(b"ntt.mode") == before[b"ntt.mode"]
        lib.vfhe_hip_ntt_mul_intt_batch(az, ax, ay, P)
        m = pool.full_mask()
        for k in range(P):
            x, y = xs[k].copy(), ys[k].copy()
            octx.to_ntt(x, x, m)
            octx.to_ntt(y, y, m)
            z = np.zeros_like(x)
            octx.mul(z, x, m, y, m, 0)
            octx.to_coeff(z, z, m)
            assert np.array_equal(pool.read(pz[k]), z), k
    finally:
        for k, v in before.items():
            lib.vfhe_hip_set_option(k, v)


def test_dropped_tile_grid_bit(lib):
    """ntt.tile_grid bit 4 chooses nothing: it is dropped where the option is set (so that graph plans do not
    differ by it), and the product tuner gives both indexes of a pair the one time it measured."""
    N, count = 8192, 2
    pool = rt.Pool(N, O.gen_primes(N, [50]))
    x, y, z = ([pool.poly() for _ in range(count)] for _ in range(3))
    keys = (b"ntt.tile_grid", b"ntt.col_wide")
    before = {k: lib.vfhe_hip_get_option(k) for k in keys}
    us = (ctypes.c_double * 6)()
    arr = rt._native.voidp_array
    try:
        for value, kept in ((31, 15), (16, 0), (15, 15)):
            assert lib.vfhe_hip_set_option(b"ntt.tile_grid", value) == 0
            assert lib.vfhe_hip_get_option(b"ntt.tile_grid") == kept
        print("[autotune product] pairs", flush=True)
        best = lib.vfhe_hip_autotune_product(arr(z), arr(x), arr(y), count, 2, us)
        assert best in (1, 3, 5) and all(u > 0 for u in us)
        assert all(us[2 * c] == us[2 * c + 1] for c in range(3)) and us[best] == min(us)
        assert lib.vfhe_hip_get_option(b"ntt.tile_grid") == 15
        lib.vfhe_hip_autotune_product(arr(z), arr(x), arr(y), count, 1, None)
    finally:
        for k, v in before.items():
            lib.vfhe_hip_set_option(k, v)
    for p in x + y + z:
        pool.free(p)


def test_alu_rate_probe(lib):
    """vfhe_hip_probe_alu_rates: six finite positive device-wide rates; the engine keeps working after."""
    rates = (ctypes.c_double * 6)()
    lib.vfhe_hip_probe_alu_rates(rates)
    print("[alu rates Gop/s]", [round(r / 1e9, 1) for r in rates], flush=True)
    assert all(np.isfinite(r) and r > 0 for r in rates)
    q = O.gen_prime(2048, 50)
    proc = lib.ntt_new_proc(1024, q)
    assert lib.mul_modq(q - 1, q - 1, proc) == 1
    lib.ntt_free_proc(proc)
