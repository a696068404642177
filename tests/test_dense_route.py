"""The rules of dense_route.hpp, compiled for the CPU: which kernel a dense
GEMM runs on and its tile.

* every tile that the rules choose over the shapes of the models here and over
  generic ones is one the kernels are built for;
* the exact GPU tests of gemm_tile.hip run every tile that is chosen over the
  models' shapes, with fewer, as many and more K steps than its stages;
* calls measured on both kernels (one MI355X, us) go to the faster one,
  wherever the two are 5 % apart or more."""
import ctypes
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "pih_amd", "csrc")

# (N, K): Qwen3-8B, the Qwen3 MLP blocks and the LM heads; DeepSeek FP8
QWEN = [(4096, 4096), (1024, 4096), (12288, 4096), (4096, 12288)]
MLP = [(3 * h, h) for h in (1024, 2048, 2560)] + [(h, 3 * h) for h in (1024, 2048, 2560)]
HEADS = [(129280, 4096), (151936, 1024), (151936, 2560), (151936, 4096)]
DEEPSEEK = [(1024, 4096), (32768, 1024), (4096, 8192), (2048, 4096), (4096, 2048)]
ROWS = sorted(set(range(1, 129)) | set(range(129, 2049, 7)) | {256, 512, 1024, 1500, 2047, 2048, 4096})


@pytest.fixture(scope="module")
def route(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    lib = str(tmp_path_factory.mktemp("route") / "route.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-Wall", "-Werror", "-I", CSRC,
                    os.path.join(HERE, "dense_route_check.cpp"), "-o", lib], check=True)
    return ctypes.CDLL(lib)


def _tile(route, bf16, m, n, k, problems=1):
    v = route.pick_tile(int(bf16), m, n, k, problems)
    return v & 0xFF, v >> 8 & 0xFF, v >> 16


def _built(bf16):
    one = {(mb, nb, 0) for mb in (1, 2, 3, 4, 5, 6, 8) for nb in (1, 2, 3, 4, 8)
           if (bf16 or nb != 3) and (nb != 8 or mb <= 4)}
    return one | {(8, 8, 1), (12, 8, 1)} | ({(16, 8, 1)} if bf16 else set())


@pytest.mark.parametrize("bf16", [True, False])
def test_only_built_tiles_are_chosen(route, bf16):
    step = 16 if bf16 else 128
    generic = [(n, k) for n in (step, 3 * step, 128, 384, 640, 1280, 5120, 28672)
               for k in ((128, 256, 384, 640, 5120, 17408) if bf16 else (512, 1024, 1536, 7168, 8192))]
    for n, k in generic + (QWEN + MLP + HEADS if bf16 else DEEPSEEK):
        for m in ROWS:
            for problems in (1,) if bf16 else (1, 4, 8):
                tile = _tile(route, bf16, m, n, k, problems)
                assert tile in _built(bf16), (m, n, k, problems, tile)
                # a walked tile has at least 8 K steps; a tile's columns divide n
                assert n % (16 * tile[1]) == 0 and (not tile[2] or (2 * k if bf16 else k) >= 1024)


def _stages(bf16, tile):
    """LDS stages of a tile and its K steps per 1024 row bytes, as the kernels
    size them"""
    mb, nb, grid = tile
    lds, step = 160 * 1024 - 512, 128 if grid else 256
    panel = 0 if bf16 else 256 + 16 * mb * 64
    loads = (mb + nb) * step // 256
    room = lds - (2 * panel + 4 * 16 * 144 if grid else panel)
    return min(room // (16 * (mb + nb) * step), 8, 63 // loads + 1), 1024 // step


@pytest.mark.parametrize("bf16", [True, False])
def test_gpu_tests_run_every_tile_of_the_models(route, bf16):
    import test_gpu_tile as gpu

    used = {}
    for n, k in QWEN + MLP + HEADS if bf16 else DEEPSEEK:
        for m in (r for r in ROWS if r <= 2048):
            taken = route.bf16_on_tiles(m, n, k, 0, 1) if bf16 else route.fp8_on_tiles(m, n, k, 1, 0, 1)
            if taken:
                used.setdefault(_tile(route, bf16, m, n, k), (m, n, k))
    tested = {}
    for m, n, k in gpu.BF16 + gpu.BF16_TILES if bf16 else gpu.FP8 + gpu.FP8_TILES:
        if route.bf16_on_tiles(m, n, k, 0, 0) if bf16 else k % 512 == 0 and k <= 8192 and route.fp8_on_tiles(m, n, k, 1, 0, 1):
            tile = _tile(route, bf16, m, n, k)
            st, per_kb = _stages(bf16, tile)
            steps = (2 * k if bf16 else k) * per_kb // 1024
            tested.setdefault(tile, set()).add((steps > st) - (steps < st))
    missing = {t: used[t] for t in used if t not in tested}
    assert not missing, missing
    for t in used:  # (a walked tile has 8 steps or more and at most 5 stages)
        assert tested[t] >= ({1} if t[2] else {-1, 1}), (t, tested[t], used[t])
    assert sum(0 in s for s in tested.values()) >= len(used) // 3


# (m, n, k, us on the other kernel, us on the tiles)
FP8_MEASURED = [
    (1, 128, 512, 2.67, 2.98), (2, 256, 512, 2.75, 3.15), (8, 2048, 512, 3.07, 3.31), (1, 4096, 1024, 3.45, 3.72),
    (1, 129280, 1024, 27.2, 33.8), (8, 7168, 512, 3.9, 3.5), (4, 1024, 4096, 5.77, 4.27), (4, 32768, 1024, 10.0, 8.1),
    (64, 4096, 8192, 30.4, 13.2), (301, 32768, 1024, 33.1, 22.2), (2048, 1024, 4096, 27.2, 15.5),
    (4096, 32768, 512, 169.6, 313.0), (2048, 16384, 512, 46.6, 78.8), (4096, 7168, 512, 46.1, 66.9),
    (4096, 2048, 7168, 66.7, 80.8), (4096, 2048, 4096, 44.3, 50.7), (2048, 4096, 8192, 76.1, 80.2),
    (2048, 4096, 6144, 60.1, 64.9), (4096, 8192, 8192, 284.6, 309.6), (2048, 12288, 4096, 121.6, 128.5),
    (512, 4096, 8192, 50.5, 29.3), (1024, 2048, 7168, 47.5, 26.0), (2048, 32768, 1024, 127.0, 101.0)]
BF16_MEASURED = [
    (8, 1024, 128, 2.08, 2.77), (8, 256, 512, 2.5, 3.0), (8, 1024, 768, 3.7, 3.1), (2, 12288, 4096, 20.3, 17.7),
    (17, 12288, 4096, 21.6, 18.7), (57, 1024, 4096, 11.0, 6.4), (200, 4096, 4096, 25.0, 17.3),
    (200, 28672, 4096, 87.0, 78.0), (2048, 12288, 4096, 183.0, 163.0), (2048, 4096, 12288, 175.0, 160.0),
    (4096, 1024, 16384, 119.4, 257.1), (2048, 1024, 16384, 68.9, 121.5), (2048, 256, 16384, 42.5, 77.0),
    (4096, 512, 7168, 41.2, 66.7), (1024, 2560, 7680, 52.4, 72.0), (256, 4096, 12288, 49.9, 59.4),
    (1024, 4096, 12288, 103.0, 118.3), (200, 8192, 28672, 130.5, 189.7), (128, 5120, 17408, 52.0, 69.2),
    (4096, 4096, 256, 22.3, 36.4), (1000, 5120, 5120, 90.7, 52.4), (2048, 2560, 7680, 125.3, 82.7)]
# without a workspace: the 128 x 256 tiles unsplit, in 64- and 32-row M tiles
BF16_NO_WORKSPACE = [
    (2048, 1024, 4096, 43.1, 29.4), (1024, 1024, 4096, 42.9, 21.0), (301, 4096, 12288, 130.5, 61.9),
    (512, 4096, 4096, 43.7, 27.7), (1024, 4096, 12288, 134.1, 117.2), (301, 12288, 4096, 52.5, 44.8),
    (2048, 2048, 6144, 69.5, 61.4), (96, 2048, 6144, 70.8, 16.4)]


def test_measured_calls_go_to_the_faster_kernel(route):
    for m, n, k, other, tiles in FP8_MEASURED:
        assert bool(route.fp8_on_tiles(m, n, k, 1, 0, 1)) == (tiles < other), ("fp8", m, n, k)
    for m, n, k, other, tiles in BF16_MEASURED:
        assert bool(route.bf16_on_tiles(m, n, k, 0, 1)) == (tiles < other), ("bf16", m, n, k)
    for m, n, k, other, tiles in BF16_NO_WORKSPACE:
        assert bool(route.bf16_on_tiles(m, n, k, 0, 0)) == (tiles < other), ("bf16 unsplit", m, n, k)


def test_grouped_calls_stay_off_the_128_x_256_tiles(route):
    """Without a code check those read blocks under a 0xFF weight scale."""
    for m in (64, 257, 700, 2048, 4096):
        for n, k in ((1024, 4096), (128, 512), (4096, 8192)):
            for problems in (1, 4, 8, 16):
                assert route.fp8_on_tiles(m, n, k, problems, 0, 0)


def test_w4a16_rule(route):
    def blocks(m, k, *n):
        return route.w4a16_blocks(m, k, (ctypes.c_uint32 * len(n))(*n), len(n))

    # Qwen3-8B: [q, k, v], o, [gate, up], down
    qkv, o, gu, down = (4096, (4096, 1024, 1024)), (4096, (4096,)), (4096, (12288, 12288)), (12288, (4096,))
    taken = {1: (), 2: (gu,), 4: (gu,), 8: (qkv, gu), 12: (qkv, gu, down), 16: (qkv, o, gu, down),
             32: (qkv, o, gu, down)}
    for m, groups in taken.items():
        for k, n in (qkv, o, gu, down):
            assert bool(blocks(m, k, *n)) == ((k, n) in groups), (m, k, n)
    assert blocks(33, 4096, 12288) == 0
    assert blocks(2, 2048, 6144, 6144) == 0  # 5.54 us on the GEMV, 6.10 on the tiles
    assert blocks(32, 1024, 3072) == 0 and blocks(32, 1536, 3072)  # 4.1 us on the GEMV, 4.7 on the tiles
    for m in range(2, 33):
        for n in ((16,), (48, 96), (16, 32, 4096), (2560,), (9728, 9728)):
            for k in (512, 1536, 4096, 12288):
                c = blocks(m, k, *n)
                assert c in (0, 1, 2, 3, 4, 6) and (not c or all(v % (16 * c) == 0 for v in n))
