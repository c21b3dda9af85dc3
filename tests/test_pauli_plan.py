"""The passes that a Pauli sum is cut into (qcsim_amd/csrc/pauli_plan.cpp), on
the CPU: each term is in one pass, whose masks say of it what the term's say,
and planning takes time in proportion."""
import ctypes as C
import os
import subprocess
import time

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SLOTS, TERMS = 12, 64


class Tile(C.Structure):
    _fields_ = [("t", C.c_uint32), ("ns", C.c_uint32), ("nt", C.c_uint32), ("im", C.c_uint32), ("pos", C.c_uint32 * 12),
                ("tile_bits", C.c_uint64), ("step", C.c_uint64), ("x", C.c_uint32 * SLOTS), ("zt", C.c_uint32 * (2 * SLOTS)),
                ("first", C.c_uint32 * (SLOTS + 1)), ("z", C.c_uint32 * TERMS)]


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("pauli") / "libpauli_host.so")
    src = [os.path.join(ROOT, p) for p in ("tests/cpp/pauli_host.cpp", "qcsim_amd/csrc/pauli_plan.cpp")]
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-shared", "-fPIC", *src, "-o", lib], check=True)
    L = C.CDLL(lib)
    L.pauli_new.restype, L.pauli_new.argtypes = C.c_void_p, [C.c_uint32, C.c_uint64, C.c_uint32, C.c_void_p, C.c_void_p]
    L.pauli_free.restype, L.pauli_free.argtypes = None, [C.c_void_p]
    L.pauli_step.restype, L.pauli_step.argtypes = C.c_uint32, [C.c_void_p, C.POINTER(Tile), C.c_void_p]
    L.pauli_wide.restype, L.pauli_wide.argtypes = C.c_uint32, [C.c_void_p, C.c_void_p]
    return L


def unpack(v, bits):
    """The low bits of v at the given places."""
    return sum(1 << b for i, b in enumerate(bits) if v >> i & 1)


def plan(host, n, x, z, amp_bytes=16):
    """[(tile, pairs, terms)] and the terms of wide masks."""
    x, z = np.array(x, dtype=np.uint64), np.array(z, dtype=np.uint64)
    h = host.pauli_new(n, amp_bytes, len(x), x.ctypes.data, z.ctypes.data)
    out = []
    while True:
        tile, terms = Tile(), np.zeros(TERMS, dtype=np.uint32)
        k = host.pauli_step(h, C.byref(tile), terms.ctypes.data)
        if not k:
            break
        count = k % 1000
        assert 0 < count <= TERMS and tile.nt == count
        out.append((tile, k >= 1000, terms[:count].copy()))
    wide = np.zeros(len(x), dtype=np.uint32)
    wide = wide[: host.pauli_wide(h, wide.ctypes.data)]
    host.pauli_free(h)
    return out, wide


def check(n, x, z, passes, wide):
    t = max(2, min(n, 12))
    seen = list(wide)
    for tile, pairs, terms in passes:
        inside = list(tile.pos)[:t]
        outside = [q for q in range(n) if q not in inside]
        assert tile.t == t and inside == sorted(set(inside)) and tile.tile_bits == sum(1 << q for q in inside)
        assert tile.step == unpack(min(2 ** len(outside), 256), [*outside, n, n + 1] if n >= t else [2])
        assert tile.ns <= SLOTS and tile.first[0] == 0
        seen += list(terms)
        for e, i in enumerate(terms):
            X, Z = int(x[i]), int(z[i])
            j = sum(e >= tile.first[k + 1] for k in range(tile.ns))
            zl = tile.z[e]
            if j == tile.ns:  # x = 0 and z within the tile
                assert X == 0 and unpack(zl, inside) == Z
            elif pairs:
                assert X and unpack(tile.x[j], inside) == X
                assert unpack(zl, inside) | unpack(tile.zt[j], outside) == Z
                assert tile.im >> j & 1 == bin(X & Z).count("1") & 1
            else:
                s = 2 * j + (zl >> 15)
                zl &= 0x7FFF
                assert X == 0 and tile.zt[s] >> 30 == zl >> (t - 2)
                assert unpack(zl, inside) | unpack(tile.zt[s] & 0x3FFFFFFF, outside) == Z
        if not pairs:  # a sum holds one term
            used = [2 * sum(e >= tile.first[k + 1] for k in range(tile.ns)) + (tile.z[e] >> 15)
                    for e in range(tile.first[tile.ns])]
            assert len(set(used)) == len(used)
    assert sorted(seen) == list(range(len(x)))


def random_terms(rng, n, masks, terms, weight=4):
    xs = {0}
    for _ in range(20 * masks):
        if len(xs) == masks:
            break
        xs.add(sum(1 << int(q) for q in rng.choice(n, min(n, int(rng.integers(1, weight + 1))), replace=False)))
    xs = list(xs)
    x = [xs[i % len(xs)] for i in range(terms)]
    z = [int(rng.integers(1 << n)) & (v if v and rng.random() < 0.5 else (1 << n) - 1) for v in x]
    return x, z


def chain(n):
    x, z = [], []
    for q in range(n - 1):
        x, z = x + [3 << q, 3 << q, 0], z + [0, 3 << q, 3 << q]
    return x + [0] * n, z + [1 << q for q in range(n)]


@pytest.mark.parametrize("n", [1, 2, 3, 5, 11, 12, 13, 16, 21, 30])
def test_every_term_once(host, n):
    rng = np.random.default_rng(n)
    full = (1 << n) - 1
    for x, z in (chain(n), random_terms(rng, n, min(2**n // 2 + 1, 60), 400),
                 ([0] * 300, [int(v) for v in rng.integers(0, full + 1, 300)]),
                 ([int(v) for v in rng.integers(0, full + 1, 90)], [int(v) for v in rng.integers(0, full + 1, 90)]),
                 ([full, 0, 1] * 50, [int(v) for v in rng.integers(0, full + 1, 150)])):
        for amp_bytes in (8, 16):
            passes, wide = plan(host, n, x, z, amp_bytes)
            check(n, x, z, passes, wide)


def test_passes_are_few(host):
    """A Heisenberg chain's pairs in three tiles, its fields and bonds with
    them; and terms that differ in z alone in as many passes as they need."""
    x, z = chain(26)
    assert len(plan(host, 26, x, z)[0]) == 3
    rng = np.random.default_rng(1)
    z = [int(v) | 1 << 25 for v in rng.integers(0, 1 << 26, 32)]
    passes, _ = plan(host, 26, [0] * 32, z)
    assert [p[0].nt for p in passes] == [16, 16]  # 24 and 8 sums take longer
    x, z = random_terms(rng, 12, 100, 1280)
    assert len(plan(host, 12, x, z)[0]) <= 25  # 20 hold as many terms


def test_planning_grows_with_the_terms(host):
    """Ten times the masks and terms take at most fifty times as long, where
    gathering the masks for every pass made it a thousand."""
    rng = np.random.default_rng(2)

    def best(masks, terms):
        x, z = (np.array(v, dtype=np.uint64) for v in random_terms(rng, 20, masks, terms))
        tile, out, times = Tile(), np.zeros(TERMS, dtype=np.uint32), []
        for _ in range(3):
            t = time.perf_counter()
            h = host.pauli_new(20, 16, terms, x.ctypes.data, z.ctypes.data)
            while host.pauli_step(h, C.byref(tile), out.ctypes.data):
                pass
            host.pauli_free(h)
            times.append(time.perf_counter() - t)
        return min(times)

    assert best(2500, 30000) < 50 * best(250, 3000)
