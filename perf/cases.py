"""Work that users of the engine have it do, as cases that a timing program can run.

A case is a dict of plain values.  prepare() makes what a program has in hand before the
call (inputs, keys and output buffers on the GPU), run() is one pass through the public
entry points, work() the bytes and operations a pass cannot do without.  Sizes follow the
repository's own configurations (bench.py, the serving mix, the tests).

Residues, ciphertexts and evaluation keys are uniform modulo their primes, as real ones
are; the bootstrapping keys and LWE samples are real encryptions.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from vfhe_amd import _native, arith, cggi, fhe, params, runtime, torus

KINDS = ("ring_product", "transform", "product", "multiply", "rotate", "torus", "cggi")


def listed():
    return [
        # one product of two polynomials of the arith layer's default ring (49-bit primes, split
        # degree 4) and its way back to coefficients: the smallest call, all latency
        {"name": "ring_product_4096", "kind": "ring_product", "N": 4096, "limbs": 7},
        # the headline transform: 64 polynomials x 24 limbs of 2^16 coefficients, forward
        {"name": "ntt_forward_65536", "kind": "transform", "N": 65536, "limbs": 24, "count": 64, "bits": 50,
         "inverse": False},
        # the plain configuration's inverse: 16 polynomials x 4 limbs of 4096 coefficients
        {"name": "ntt_inverse_4096", "kind": "transform", "N": 4096, "limbs": 4, "count": 16, "bits": 50,
         "inverse": True},
        # negacyclic products z = INTT(NTT(x) NTT(y)) of an odd batch on a small bootstrapping-size ring
        {"name": "product_2048_odd", "kind": "product", "N": 2048, "limbs": 3, "count": 37, "bits": 50},
        # the fused product configuration: 64 pairs x 24 limbs of 2^16
        {"name": "product_65536", "kind": "product", "N": 65536, "limbs": 24, "count": 64, "bits": 50},
        # products modulo 60-bit primes (above the 50 bits of the FP64 path), as wide-prime chains need
        {"name": "product_wide_16384", "kind": "product", "N": 16384, "limbs": 6, "count": 9, "bits": 60},
        # CKKS multiply + relinearize + rescale, the 32-pair configuration at 24 + 4 limbs
        {"name": "multiply_65536_b32", "kind": "multiply", "N": 65536, "limbs": 24, "special": 4, "count": 32},
        # one request of the serving mix alone: a multiply at a middle level
        {"name": "multiply_16384_b1", "kind": "multiply", "N": 16384, "limbs": 11, "special": 4, "count": 1},
        # rotations (automorphism + key-switch) of a small odd batch
        {"name": "rotate_32768_b5", "kind": "rotate", "N": 32768, "limbs": 13, "special": 4, "count": 5},
        # functional bootstraps over the 32-bit torus, the 1024-sample configuration, results read back
        {"name": "torus_bootstrap_1024", "kind": "torus", "count": 1024, "n": 630, "ell": 3, "base_log": 7},
        # the same for a handful of samples, where latency counts
        {"name": "torus_bootstrap_3", "kind": "torus", "count": 3, "n": 630, "ell": 3, "base_log": 7},
        # CGGI16 bootstraps over RNS primes (the NTT variant), 1024 samples, extracted to the host
        {"name": "cggi_bootstrap_1024", "kind": "cggi", "count": 1024, "n": 630},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(KINDS)
    if kind == "ring_product":
        return {"kind": kind, "N": 1 << rng.randint(8, 14), "limbs": rng.randint(1, 12)}
    if kind == "transform":
        return {"kind": kind, "N": 1 << rng.randint(10, 16), "limbs": rng.randint(1, 24),
                "count": _log_int(rng, 1, 64), "bits": rng.choice((50, 50, 60)), "inverse": rng.random() < 0.5}
    if kind == "product":
        bits = rng.choice((50, 50, 60))
        return {"kind": kind, "N": 1 << rng.randint(10, 16), "limbs": rng.randint(1, 24 if bits == 50 else 8),
                "count": _log_int(rng, 1, 64 if bits == 50 else 16), "bits": bits}
    if kind in ("multiply", "rotate"):
        return {"kind": kind, "N": 1 << rng.randint(13, 16), "limbs": rng.randint(4, 24), "special": 4,
                "count": _log_int(rng, 1, 32)}
    if kind == "torus":
        ell, base_log = rng.choice(((3, 7), (3, 7), (2, 10)))
        return {"kind": kind, "count": _log_int(rng, 1, 1024), "n": rng.randint(450, 630), "ell": ell,
                "base_log": base_log}
    return {"kind": kind, "count": _log_int(rng, 1, 1024), "n": rng.randint(450, 630)}


# ---------------------------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------------------------
class _DeviceRows:
    """The rows of an engine polynomial as a torch-readable array (no copy); holds `owner`."""

    def __init__(self, handle, rows, N, owner):
        ptr = ctypes.cast(_native.load().polynomial_device_row(handle, 0), ctypes.c_void_p).value
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (rows, N), "typestr": "<i8", "data": (ptr, False), "version": 2}


def _rows(handle, rows, N, owner=None):
    return torch.as_tensor(_DeviceRows(handle, rows, N, owner), device="cuda")


_pools = {}


def _pool(N, bits, limbs):
    """The prime pool of a ring: a program makes it once and keeps it."""
    key = (N, bits, limbs)
    if key not in _pools:
        _pools[key] = runtime.Pool(N, params.gen_primes(N, [bits] * limbs))
    return _pools[key]


class _State:
    """Handles and buffers of one case; frees its engine objects when it goes."""

    def __init__(self, case):
        self.case = case
        self.polys, self.samples = [], []

    def __del__(self):
        try:
            lib = _native.load()
            lib.vfhe_hip_synchronize()
            for p in self.polys:
                lib.free_RNS_polynomial(p)
            for c in self.samples:
                lib.free_mlwe_RNS_sample(c)
        except Exception:
            pass


def _fill(pool, gen, handle):
    """Uniform residues in every row of the pool (once the engine has cleared them)."""
    _native.load().vfhe_hip_synchronize()
    q = torch.tensor(pool.primes, dtype=torch.int64, device="cuda")[:, None]
    _rows(handle, pool.l, pool.N).copy_(torch.randint(0, 1 << 62, (pool.l, pool.N), generator=gen, device="cuda") % q)


def _poly(st, pool, gen=None):
    p = pool.poly()
    st.polys.append(p)
    if gen is not None:
        _fill(pool, gen, p)
    return p


def _sample(st, pool, mask, gen=None):
    c = pool.sample(1, mask)
    st.samples.append(c)
    if gen is not None:
        for p in pool.comps(c):
            _fill(pool, gen, p)
    return c


def _switch_key(st, pool, gen, limbs):
    """One digit per level limb, each a sample on the extended ring."""
    return _native.voidp_array([_sample(st, pool, pool.full_mask(), gen) for _ in range(limbs)])


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def run(state):
    return globals()["_run_" + state.case["kind"]](state)


def _gen(seed):
    torch.cuda.synchronize()
    return torch.Generator(device="cuda").manual_seed(seed)


# -- products in the arith layer's default ring
_rings = {}


def _ring(N, limbs):
    if N not in _rings:   # the pool of this N, with every prime a program will use
        _rings[N] = arith.Ring(N, prime_size=[49] * 12)
    return _rings[N].quotient_ring(ell=limbs)


def _prepare_ring_product(case, seed):
    st = _State(case)
    st.ring = _ring(case["N"], case["limbs"])
    gen = _gen(seed)
    st.ab = []
    for _ in range(2):
        p = arith.Polynomial(st.ring, arith.repr.ntt)
        q = torch.tensor(st.ring.primes, dtype=torch.int64, device="cuda")[:, None]
        _native.load().vfhe_hip_synchronize()
        _rows(p.obj, case["limbs"], case["N"]).copy_(
            torch.randint(0, 1 << 62, (case["limbs"], case["N"]), generator=gen, device="cuda") % q)
        st.ab.append(p)
    torch.cuda.synchronize()
    return st


def _run_ring_product(st):
    c = st.ab[0] * st.ab[1]
    c.to_coeff()
    return _rows(c.obj, st.case["limbs"], st.case["N"], c)


# -- batched transforms, in place
def _prepare_transform(case, seed):
    st, pool = _State(case), _pool(case["N"], case["bits"], case["limbs"])
    gen = _gen(seed)
    hs = [_poly(st, pool, gen) for _ in range(case["count"])]
    st.handles = _native.voidp_array(hs)
    st.out = [_rows(p, pool.l, pool.N) for p in hs]
    torch.cuda.synchronize()
    return st


def _run_transform(st):
    _native.load().vfhe_hip_ntt_batch(st.handles, st.case["count"], 1 if st.case["inverse"] else 0)
    return st.out


# -- batched negacyclic products
def _prepare_product(case, seed):
    st, pool = _State(case), _pool(case["N"], case["bits"], case["limbs"])
    gen = _gen(seed)
    x, y = ([_poly(st, pool, gen) for _ in range(case["count"])] for _ in range(2))
    z = [_poly(st, pool) for _ in range(case["count"])]
    st.x, st.y, st.z = (_native.voidp_array(v) for v in (x, y, z))
    st.out = [_rows(p, pool.l, pool.N) for p in z]
    torch.cuda.synchronize()
    return st


def _run_product(st):
    _native.load().vfhe_hip_ntt_mul_intt_batch(st.z, st.x, st.y, st.case["count"])
    return st.out


# -- CKKS multiply + relinearize + rescale
def _prepare_multiply(case, seed):
    L, K, B = case["limbs"], case["special"], case["count"]
    st, pool = _State(case), _pool(case["N"], 50, L + K)
    level = (1 << L) - 1
    gen = _gen(seed)
    c1, c2 = ([_sample(st, pool, level, gen) for _ in range(B)] for _ in range(2))
    outs = [_sample(st, pool, pool.full_mask()) for _ in range(B)]
    st.key = _switch_key(st, pool, gen, L)
    st.rlk = _native.voidp_array([st.key, None])
    st.c1, st.c2, st.outs = (_native.voidp_array(v) for v in (c1, c2, outs))
    st.out = [_rows(p, L - 1, pool.N) for c in outs for p in pool.comps(c)]
    torch.cuda.synchronize()
    return st


def _run_multiply(st):
    _native.load().vfhe_hip_mlwe_multiply_batch(st.outs, st.c1, st.c2, st.case["count"], st.rlk,
                                                1 << (st.case["limbs"] - 1))
    return st.out


# -- rotations
def _prepare_rotate(case, seed):
    L, K, B = case["limbs"], case["special"], case["count"]
    st, pool = _State(case), _pool(case["N"], 50, L + K)
    gen = _gen(seed)
    ins = [_sample(st, pool, (1 << L) - 1, gen) for _ in range(B)]
    outs = [_sample(st, pool, pool.full_mask()) for _ in range(B)]
    st.key = _switch_key(st, pool, gen, L)
    st.ksk = _native.voidp_array([st.key])
    st.ins, st.outs = _native.voidp_array(ins), _native.voidp_array(outs)
    st.gen = pow(5, 1 + seed % 31, 2 * case["N"])
    st.out = [_rows(p, L, pool.N) for c in outs for p in pool.comps(c)]
    torch.cuda.synchronize()
    return st


def _run_rotate(st):
    _native.load().vfhe_hip_mlwe_automorphism_batch(st.outs, st.ins, st.case["count"], st.gen, st.ksk)
    return st.out


# -- functional bootstraps over the 32-bit torus
def _prepare_torus(case, seed):
    st = _State(case)
    p = torus.TorusParams(n=case["n"], ell=case["ell"], base_log=case["base_log"])
    keys = torus.TorusKeys(p, seed=seed)
    st.boot = torus.TorusBootstrapper(keys.bootstrap_key(), p)
    st.tv = torus.TorusBatch.upload(torus.pack_lut(list(range(16)), 16, 5))
    st.lwes = torus.TorusBatch.upload(keys.encrypt(keys.rng.integers(0, 16, case["count"]), 5))
    st.samples_out = torus.TorusBatch.zeros(case["count"], p.N + 1)
    return st


def _run_torus(st):
    return st.boot.bootstrap(st.lwes, st.tv, 16, out=st.samples_out).read().view(np.int32)


# -- CGGI16 bootstraps over RNS primes
class _Lwe(ctypes.Structure):   # struct _LWE of include/vfhe_hip.h
    _fields_ = [("a", ctypes.POINTER(ctypes.c_void_p)), ("b", ctypes.c_void_p), ("n", ctypes.c_uint64),
                ("l", ctypes.c_uint64), ("ntt", ctypes.c_void_p)]


_cggi_ring = []


def _prepare_cggi(case, seed):
    st, N = _State(case), 1024
    rng = np.random.default_rng(seed)
    _native.load().vfhe_prng_set_deterministic_seed(seed)
    if not _cggi_ring:
        _cggi_ring.append(arith.Ring(N, prime_size=[50, 50, 50], split_degree=1))
    ring = _cggi_ring[0]
    in_ring = ring.quotient_ring(ell=2)
    st.lwe_key = cggi.LweKey(in_ring, [int(b) for b in rng.integers(0, 2, case["n"])])
    chain = fhe.Chain.nested(ring, special=1, levels=1)
    sk = [0] * N
    for k in rng.choice(N, size=64, replace=False):
        sk[int(k)] = 1
    st.out_key = fhe.SecretKey(chain, [sk], 3.2)
    st.boot = cggi.Bootstrapper(chain, cggi.BootstrapKey(chain, st.lwe_key, st.out_key))
    st.tv = cggi.pack_lut(chain, list(range(16)), 16, 5)
    q = in_ring.q_l
    st.lwes = cggi.LweBatch.encrypt(st.lwe_key, [round(int(v) * q / 32) % q for v in rng.integers(0, 16, case["count"])])
    _native.load().vfhe_hip_synchronize()
    return st


def _run_cggi(st):
    out = st.boot.bootstrap(st.tv, st.lwes, 16)
    parts = []
    for h in out.handles:
        s = _Lwe.from_address(h)
        parts += [ctypes.string_at(s.a[j], 8 * s.n) for j in range(s.l)]
        parts.append(ctypes.string_at(s.b, 8 * s.l))
    return np.frombuffer(b"".join(parts), dtype=np.int64).reshape(len(out), -1)


# ---------------------------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------------------------
def _ntt_flops(n, rows):
    return rows * n / 2 * math.log2(n) * 7   # a butterfly: a modular product of 5 operations, two sums


def work(case):
    kind = case["kind"]
    if kind == "torus":
        n, M, rows, B = case["n"], 512, 2 * case["ell"], case["count"]
        fft = 5 * M * math.log2(M)
        return {"bytes": 16.0 * M * n * rows * 2 + B * 4.0 * (n + 1 + 2 * M + 1),
                "flops": 1.0 * B * n * ((rows + 2) * fft + rows * 2 * M * 8)}
    if kind == "cggi":
        n, N, B = case["n"], 1024, case["count"]
        return {"bytes": n * 4 * 2 * 3 * N * 8.0 + B * 8.0 * 2 * (n + 1 + N + 1),
                "flops": 1.0 * B * n * (_ntt_flops(N, 4 * 3 + 2 * 3) + 4 * 2 * 3 * N * 6)}
    N, L, B = case["N"], case["limbs"], case.get("count", 1)
    row = 8.0 * N
    if kind == "ring_product":
        return {"bytes": 3 * L * row, "flops": _ntt_flops(N // 4, 4 * L) + L * N * 4 * 6.0}
    if kind == "transform":
        return {"bytes": 2 * L * B * row, "flops": _ntt_flops(N, L * B)}
    if kind == "product":
        return {"bytes": 3 * L * B * row, "flops": 3 * _ntt_flops(N, L * B) + L * B * N * 6.0}
    ext, digits = L + case["special"], L
    key = digits * 2 * ext * row
    switch = B * (_ntt_flops(N, digits * ext + 2 * ext) + digits * ext * 2 * N * 6.0)
    if kind == "multiply":
        return {"bytes": key + B * (4 * L + 2 * (L - 1)) * row,
                "flops": switch + B * (_ntt_flops(N, L) + L * N * 4 * 6.0)}
    return {"bytes": key + B * 4 * L * row, "flops": switch}


# ---------------------------------------------------------------------------------------------
# Values
# ---------------------------------------------------------------------------------------------
def _negacyclic(x, y, N, q):
    """x * y mod X^N + 1 mod q with Python integers (one big product of packed coefficients)."""
    width = 8 * ((2 * q.bit_length() + N.bit_length() + 7) // 8)
    pack = lambda v: int.from_bytes(b"".join(int(c).to_bytes(width // 8, "little") for c in v), "little")  # noqa: E731
    z = (pack(x) * pack(y)).to_bytes(2 * N * width // 8 + 8, "little")
    c = [int.from_bytes(z[i * width // 8:(i + 1) * width // 8], "little") for i in range(2 * N)]
    return [(c[i] - c[i + N]) % q for i in range(N)]


def exact(case, seed):
    """Every output is whole numbers; the products also have a direct value."""
    if case["kind"] != "product" or case["N"] * case["limbs"] * case["count"] > 1 << 18:
        return None
    st, pool = prepare(case, seed), _pool(case["N"], case["bits"], case["limbs"])
    xs, ys = ([_rows(h, pool.l, pool.N).cpu().numpy() for h in v] for v in (st.x, st.y))
    return [np.array([_negacyclic(x[i], y[i], pool.N, q) for i, q in enumerate(pool.primes)], dtype=np.int64)
            for x, y in zip(xs, ys)]
