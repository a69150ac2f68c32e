"""The choice of tile and K split (csrc/tile_choice.h), compiled for the host: no GPU needed."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

from chatrwkv_amd import build as _build

WS = 64 << 20   # scratch for slabs that the models' launches have

SOURCE = r"""
#include "tile_choice.h"
#include <chrono>

// the definition, product by product, tile by tile and split by split
static TilePick one_by_one(bool w_u8, int64_t T, int nk, int n, const int64_t *M, uint64_t ws) {
    TilePick best = {TILE_S, 1, NEVER};
    for (int tile = 0; tile < TILES; ++tile) {
        const TileDim d = tile_dim[tile];
        const TilePrice &p = tile_price[w_u8][tile];
        int64_t tiles = 0, outs = 0;
        for (int i = 0; i < n; ++i) { tiles += ((T + d.tm - 1) / d.tm) * ((M[i] + d.tn - 1) / d.tn); outs += T * M[i]; }
        if (!tile_offered(tile, T, (float)tiles)) continue;
        for (int c = 1; c <= 8; ++c) {
            if (nk % c || (c > 1 && (nk / c < 8 || 4 * (uint64_t)outs * c > ws || tile >= TILE_96x128))) continue;
            const int64_t wgs = tiles * c, full = wgs / 256;
            const float depth = (float)(nk / c), last = (float)(wgs % 256) / 256.f;
            float us = p.launch + (float)(full + (last > 0.f)) * (c > 1 ? p.split_round : p.round) + depth * p.step_1 * ((float)full + last);
            if (last > 0.f) us += depth * p.step_0 * (1.f - last);
            if (wgs > 256) us += depth * p.extra * ((float)wgs / 256.f - 1.f);
            if (c > 1) us += SECOND_LAUNCH + (float)c * (p.split + p.slab * (float)(4 * outs) / (float)(16 << 20));
            if (us < best.us) best = {tile, c, us};
        }
    }
    return best;
}
struct Out { int tile, ks, tm, tn; float us; };
static Out out(const TilePick &p) { return {p.tile, p.ks, tile_dim[p.tile].tm, tile_dim[p.tile].tn, p.us}; }
extern "C" Out pick(int u8, int64_t T, int nk, int n, const int64_t *M, uint64_t ws) { return out(Launch(T, nk, n, M, ws).best(u8)); }
extern "C" Out slow_pick(int u8, int64_t T, int nk, int n, const int64_t *M, uint64_t ws) { return out(one_by_one(u8, T, nk, n, M, ws)); }
extern "C" Out with(int u8, int tile, int64_t T, int nk, int64_t M, uint64_t ws) { return out(Launch(T, nk, 1, &M, ws).with(u8, tile)); }
// how often each tile is chosen, over single launches of 17 to 2048 rows with and without scratch
extern "C" int chosen(int u8, int *count) {
    for (int t = 0; t < TILES; ++t) count[t] = 0;
    for (int64_t T = 17; T <= 2048; T += T < 128 ? 1 : T < 600 ? 31 : 181)
        for (int nk = 1; nk <= 320; nk += nk < 16 ? 1 : 5)
            for (int64_t M = 64; M <= 24576; M += M < 4096 ? 40 : 672)
                for (uint64_t ws = 0; ws <= 64u << 20; ws += 64 << 20) ++count[Launch(T, nk, 1, &M, ws).best(u8).tile];
    return TILES;
}
// ns a choice, over launches of many sizes
extern "C" double time_choice(int slow, int reps) {
    volatile int sink = 0;
    const auto t0 = std::chrono::steady_clock::now();
    for (int i = 0; i < reps; ++i) {
        const int64_t T = 17 + i * 37 % 500, M = 64 * (1 + i * 13 % 200);
        const int nk = 4 * (1 + i * 7 % 32);
        sink = sink + (slow ? one_by_one(i & 1, T, nk, 1, &M, 64 << 20) : Launch(T, nk, 1, &M, 64 << 20).best(i & 1)).tile;
    }
    return std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count() / reps * 1e9;
}
"""


class Out(ctypes.Structure):
    _fields_ = [("tile", ctypes.c_int), ("ks", ctypes.c_int), ("tm", ctypes.c_int), ("tn", ctypes.c_int), ("us", ctypes.c_float)]

    def key(self):
        return self.tile, self.ks, self.us


@pytest.fixture(scope="module")
def choice(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if not cxx:
        pytest.skip("no C++ compiler for the host")
    d = tmp_path_factory.mktemp("choice")
    (d / "choice.cpp").write_text(SOURCE)
    subprocess.run([cxx, "-O3", "-std=c++17", "-shared", "-fPIC", "-I", _build.CSRC, str(d / "choice.cpp"), "-o", str(d / "choice.so")],
                   check=True)
    lib = ctypes.CDLL(os.fspath(d / "choice.so"))
    for f in (lib.pick, lib.slow_pick):
        f.restype = Out
        f.argtypes = [ctypes.c_int, ctypes.c_int64, ctypes.c_int, ctypes.c_int, ctypes.POINTER(ctypes.c_int64), ctypes.c_uint64]
    lib.with_ = getattr(lib, "with")
    lib.with_.restype = Out
    lib.with_.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int64, ctypes.c_int, ctypes.c_int64, ctypes.c_uint64]
    lib.time_choice.restype = ctypes.c_double
    return lib


def _pick(lib, u8, T, nk, M, ws=WS, f="pick"):
    return getattr(lib, f)(u8, T, nk, len(M), (ctypes.c_int64 * len(M))(*M), ws)


def test_choice_is_the_one_of_least_cost(choice):
    """Against the definition in 64-bit divisions, one tile and one split after the other: the same tile, split and price, bit for bit,
    for 1 to 4 products, at the edges of every side and of what a tile is offered for, and far past the models' sizes."""
    rng = np.random.default_rng(1)
    edges = [1, 2, 16, 17, 63, 64, 65, 80, 96, 97, 128, 129, 223, 225, 256, 257, 1024, 65535, 1 << 20]
    for i in range(20000):
        T = int(rng.choice(edges)) if i % 3 == 0 else int(np.exp(rng.uniform(0, np.log(70000))))
        M = [int(rng.choice([16, 97, 255, 257, 50277, 64 * int(rng.integers(1, 400)), 8 * int(rng.integers(1, 9000))]))
             for _ in range(int(rng.integers(1, 5)))]
        nk, ws, u8 = int(rng.integers(1, 330)), int(rng.choice([0, 16 << 20, WS])), i & 1
        assert _pick(choice, u8, T, nk, M, ws).key() == _pick(choice, u8, T, nk, M, ws, "slow_pick").key(), (u8, T, nk, M, ws)


def test_choice_takes_little_host_time(choice):
    """A choice is made for every launch, up to ten times a layer.  One tile and split after the other it took 0.9 us and more, which made
    products of 11 to 20 us by the operators up to 8 % slower; well under that here (0.33 of it as measured)."""
    ratio = min(choice.time_choice(0, 20000) / choice.time_choice(1, 20000) for _ in range(5))
    assert ratio < 0.6, ratio


@pytest.mark.parametrize("u8,N,M,Ts", [(1, 3072, 768, (17, 24, 32)), (1, 4096, 2048, (17, 24, 32)), (1, 3072, 1280, (17,)),
                                       (1, 4096, 4096, (45,)), (1, 3072, 768, (513,)), (0, 3072, 768, (17, 24))])
def test_a_split_pays_for_its_second_launch(choice, u8, N, M, Ts):
    """Products that are as fast or up to 0.9 us faster at full depth in a chain of launches, and one launch less for the host."""
    for T in Ts:
        assert _pick(choice, u8, T, N // 64, [M]).ks == 1, T
    # and one that gains by it
    assert _pick(choice, 0, 513, 48, [768]).ks == 2


@pytest.mark.parametrize("u8", [1, 0])
@pytest.mark.parametrize("N,M", [(4096, [4096, 16384]), (4096, [4096, 14336]), (5120, [20480]), (2048, [18432]), (4096, [24576])])
def test_tiles_of_96_rows_in_calls_of_65_to_96(choice, u8, N, M):
    """Launches of 192 to 256 workgroups take them, so that 65 to 96 rows cost no more than 97; others, where they are slower by up to a
    factor of two, do not."""
    more = _pick(choice, u8, 97, N // 64, M).us
    for T in (65, 72, 80, 95, 96):
        p = _pick(choice, u8, T, N // 64, M)
        assert p.tm == 96 and p.us <= more, (T, p.key(), more)
    for T in (64, 65, 80, 96):
        for few in ([M[0] // 2], [12288], [16384], [4096] * 3, [50304], [65536]):
            p = _pick(choice, u8, T, N // 64, few)
            assert p.tm != 96 and (p.tm, p.tn) != (128, 96), (T, few, p.key())


@pytest.mark.parametrize("u8", [1, 0])
def test_every_tile_is_chosen_somewhere(choice, u8):
    """No kernel is built for nothing, but the uint8 64 x 16 tile."""
    count = (ctypes.c_int * 64)()
    n = choice.chosen(u8, count)
    never = [(d.tm, d.tn) for d in (choice.with_(u8, t, 1024, 64, 4096, WS) for t in range(n)) if not count[d.tile]]
    assert never == ([(64, 16)] if u8 else [])
