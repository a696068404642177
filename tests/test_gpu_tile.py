"""GPU parity of the per-shape tiles (gemm_tile.hip): BF16 and e4m3 (UE8M0)
dense GEMMs at the edges of their tiles.

Operands are small integers (e4m3: integers times power-of-two scales within
a factor of 8), so every product and every partial sum is an integer multiple
of one power of two below 2^24 of it: exact in fp32 in any order.  The fp32
output must therefore equal the float64 product bit for bit, and the bf16
output its rounding, whatever tile, K split or order the kernel uses."""
import numpy as np
import pytest

from pih_amd import abi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    import torch

    from pih_amd.device import engine_stream

    with engine_stream() as s:
        yield s
        torch.cuda.synchronize()


def _ints(shape, seed, high=3):
    import torch

    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randint(-high, high + 1, shape, device="cuda", generator=g).float()


# m, n, k around: two rows, whole and ragged 16-row blocks, n / 16 not even,
# one K step (k 128), several rounds, the tile-walking kernel (128 x 128, 192 x
# 128 and 256 x 128 tiles, more tiles than CUs and fewer), and calls that stay
# on the GEMV, the 128 x 256 and the 128 x 128 kernel
BF16 = [(2, 16, 128), (3, 64, 256), (16, 1024, 384), (17, 4096, 128), (33, 48, 1152), (48, 768, 512),
        (57, 12288, 512), (64, 1024, 4096), (65, 256, 640), (80, 4096, 256), (127, 512, 1024), (200, 12288, 512),
        (301, 1024, 2048), (600, 9216, 512), (1000, 4096, 1024), (2048, 4096, 512), (2047, 12288, 512)]
# every tile that the Qwen3 projections, MLP blocks and LM heads get, with a
# ragged last tile and fewer, as many and more K steps than its LDS stages
# (test_dense_route.py checks that none is left out)
BF16_TILES = [
    (2, 16, 256), (2, 16, 1024), (2, 16, 1152), (2, 5120, 256), (2, 5120, 1024), (2, 5120, 1152), (33, 1536, 128),
    (17, 2560, 1024), (17, 2560, 1152), (33, 3072, 128), (17, 5120, 1024), (17, 5120, 1152), (97, 3072, 128),
    (17, 9216, 1024), (33, 5120, 128), (33, 5120, 1024), (33, 9216, 128), (33, 9216, 768), (33, 9216, 1024),
    (193, 2560, 128), (193, 2560, 640), (193, 2560, 768), (49, 5120, 128), (49, 5120, 768), (49, 5120, 1024),
    (49, 9216, 128), (49, 9216, 640), (49, 9216, 768), (600, 1280, 128), (600, 1280, 512), (600, 1280, 640),
    (150, 9216, 128), (150, 9216, 384), (150, 9216, 512), (65, 9216, 128), (65, 9216, 512), (65, 9216, 640),
    (193, 5120, 128), (193, 5120, 512), (193, 5120, 640), (81, 9216, 128), (81, 9216, 512), (81, 9216, 640),
    (1000, 1280, 128), (1000, 1280, 384), (1000, 1280, 512), (97, 9216, 128), (97, 9216, 384), (97, 9216, 512),
    (600, 2560, 128), (600, 2560, 384), (600, 2560, 512), (129, 12288, 512), (257, 12288, 512), (390, 12288, 512)]


@pytest.mark.parametrize("m,n,k", BF16 + BF16_TILES)
def test_bf16_exact(eng, m, n, k):
    import torch

    from pih_amd.linear import bf16_gemm

    a, w = _ints((m, k), m + k), _ints((n, k), n + k + 1)
    ref = a.double() @ w.double().T
    f32 = bf16_gemm(a.bfloat16(), w.bfloat16(), abi.OUTPUT_F32, out=torch.full((m, n), float("nan"), device="cuda"))
    b16 = bf16_gemm(a.bfloat16(), w.bfloat16())
    torch.cuda.synchronize()
    assert torch.equal(f32.double(), ref)
    assert torch.equal(b16, ref.float().bfloat16())


# 16 x 16 (four accumulator sets in each of four waves), 48 x 64 and 80 x 64
# (two in each) and the walked 128 x 128 (two)
@pytest.mark.parametrize("m,n,k,chains,limit", [(3, 1024, 4096, 16, 1.2e-7), (130, 4096, 4096, 8, 1.6e-7),
                                                (300, 4096, 4096, 8, 1.6e-7), (1024, 4096, 4096, 2, 3.3e-7)])
def test_bf16_rounding_of_the_sums(eng, m, n, k, chains, limit):
    """Normwise error of fp32 outputs against 64 bits.  A chain of c MFMAs
    rounds each time by up to 2^-24 of what it has reached, in sum about
    2^-24 sqrt(c / 6) of its result (c = k / 32 / chains); measured 1.03e-7,
    1.34e-7 and 2.7e-7, and sqrt(2) times that with half the chains, which the
    limits leave out."""
    import torch

    from pih_amd.linear import bf16_gemm

    g = torch.Generator(device="cuda")
    g.manual_seed(m)
    a = torch.randn(m, k, device="cuda", generator=g).bfloat16()
    w = (torch.randn(n, k, device="cuda", generator=g) * 0.02).bfloat16()
    got = bf16_gemm(a, w, abi.OUTPUT_F32)
    torch.cuda.synchronize()
    ref = a.double() @ w.double().T
    err = ((got.double() - ref).norm() / ref.norm()).item()
    assert 2.0 ** -24 * (k / 32 / chains / 6) ** 0.5 * 0.5 < err < limit


@pytest.mark.parametrize("m,n,k", [(5, 64, 256), (40, 128, 384)])
def test_bf16_unaligned_operand(eng, m, n, k):
    """W 8 bytes off a 16-byte boundary: the GEMV the call took before."""
    import torch

    from pih_amd.linear import bf16_gemm

    a, w = _ints((m, k), 1).bfloat16(), _ints((n, k), 2).bfloat16()
    buf = torch.empty(n * k + 8, dtype=torch.bfloat16, device="cuda")
    off = buf[4:4 + n * k].view(n, k)
    off.copy_(w)
    got = bf16_gemm(a, off, abi.OUTPUT_F32)
    torch.cuda.synchronize()
    assert off.data_ptr() % 16 == 8 and torch.equal(got.double(), a.double() @ w.double().T)


def _fp8(m, n, k, seed):
    """e4m3 codes of integers in [-3, 3] and scale bytes 126..128, with the
    float64 operands they stand for."""
    import torch

    a, w = _ints((m, k), seed), _ints((n, k), seed + 1)
    sa = 127 + _ints((m, k // 128), seed + 2, 1).to(torch.uint8)
    sw = 127 + _ints((n // 128, k // 128), seed + 3, 1).to(torch.uint8)
    code = lambda v: v.to(torch.float8_e4m3fn).view(torch.uint8).clone()  # noqa: E731
    return code(a), sa, code(w), sw


def _values(c):
    import torch

    v = c.view(torch.float8_e4m3fn).double()
    return torch.where(torch.isnan(v), torch.zeros_like(v), v)


def _scales(s):
    import torch

    return torch.where(s == 255, torch.zeros_like(s, dtype=torch.float64), torch.exp2(s.double() - 127))


def _product(av, w, sw):
    """av (float64 rows) times W, its NaN codes and 0xFF-scaled blocks as 0"""
    n, k = w.shape
    wv = (_values(w).view(n // 128, 128, k // 128, 128) * _scales(sw)[:, None, :, None]).view(n, k)
    return av @ wv.T


def _expect(a, sa, w, sw):
    """(float64 product with NaN codes and 0xFF-scaled blocks as 0)"""
    m, k = a.shape
    return _product((_values(a).view(m, k // 128, 128) * _scales(sa)[:, :, None]).view(m, k), w, sw)


def _run_fp8(a, sa, w, sw, out_type):
    import torch

    from pih_amd.device import ptr, stream_handle

    m, k = a.shape
    n = w.shape[0]
    out = torch.full((m, n), float("nan"), device="cuda", dtype=torch.float32 if out_type == 2 else torch.bfloat16)
    flag = torch.zeros(1, dtype=torch.int32, device="cuda")
    r = abi.request(abi.DS["fp8_gemm"], activation_e4m3=ptr(a), activation_scale_bits=ptr(sa), weight_e4m3=ptr(w),
                    weight_scale_bits=ptr(sw), output=ptr(out), error_flag=ptr(flag), stream=stream_handle(), m=m, n=n,
                    k=k, output_type=out_type)
    st = abi.deepseek_pack().call("launch_fp8_gemm", r)
    assert st.code == abi.OK, st
    torch.cuda.synchronize()
    return out, int(flag.item())


# k 8192 is the deepest scale panel; 768 (not a multiple of 512) and 8704
# (deeper), and some of the smallest calls, stay on other kernels
FP8 = [(1, 128, 512), (3, 1024, 1024), (4, 4096, 8192), (16, 2048, 512), (17, 128, 1536), (40, 256, 768),
       (50, 4096, 512), (75, 1024, 2048), (129, 4096, 1024), (33, 128, 8704), (301, 2048, 1024), (301, 32768, 1024),
       (700, 4096, 2048), (2048, 1024, 1024), (2047, 8192, 1024)]
# every tile that the DeepSeek projections get, as BF16_TILES
FP8_TILES = [
    (2, 128, 1536), (2, 128, 2048), (2, 128, 2560), (2, 32768, 512), (2, 32768, 1024), (2, 32768, 1536),
    (17, 2560, 512), (17, 2560, 2048), (17, 2560, 2560), (17, 5120, 512), (17, 5120, 2048), (17, 5120, 2560),
    (17, 32768, 512), (17, 32768, 1024), (33, 5120, 512), (33, 5120, 2048), (33, 9216, 512), (33, 9216, 1536),
    (97, 9216, 512), (97, 9216, 1024), (49, 5120, 512), (49, 5120, 1536), (49, 5120, 2048), (49, 9216, 512),
    (49, 9216, 1024), (49, 9216, 1536), (150, 9216, 512), (150, 9216, 1024), (65, 9216, 512), (65, 9216, 1024),
    (65, 9216, 1536), (81, 9216, 512), (81, 9216, 1024), (97, 12288, 512), (97, 12288, 1024), (129, 12288, 1024),
    (257, 12288, 1024)]


@pytest.mark.parametrize("m,n,k", FP8 + FP8_TILES)
def test_fp8_exact(eng, m, n, k):
    import torch

    a, sa, w, sw = _fp8(m, n, k, 7 * m + n + k)
    ref = _expect(a, sa, w, sw)
    for out_type in (1, 2):
        got, flag = _run_fp8(a, sa, w, sw, out_type)
        assert flag == 0
        assert torch.equal(got, ref.float().bfloat16() if out_type == 1 else ref.float())


@pytest.mark.parametrize("m,n,k", [(20, 256, 1024), (301, 2048, 1024), (301, 4096, 1024), (700, 8192, 1024)])
def test_fp8_codes_and_invalid_scales(eng, m, n, k):
    """NaN codes count as 0 and raise bit 1, 0xFF scales leave their block out
    and raise bit 2, in one-tile-per-block and in walked tiles; a code in a
    block that a 0xFF scale leaves out raises bit 2 alone."""
    import torch

    a, sa, w, sw = _fp8(m, n, k, m)
    a[m - 1, 5], w[n - 1, k - 1] = 0x7F, 0xFF
    got, flag = _run_fp8(a, sa, w, sw, 2)
    assert flag == 1 and torch.equal(got, _expect(a, sa, w, sw).float())
    a, sa, w, sw = _fp8(m, n, k, m)
    sa[m // 2, 3], sw[n // 128 - 1, 1] = 255, 255
    got, flag = _run_fp8(a, sa, w, sw, 2)
    assert flag == 2 and torch.equal(got, _expect(a, sa, w, sw).float())
    a[m // 2, 3 * 128 + 7] = 0x7F
    w[n - 1, 128 + 9] = 0xFF
    got, flag = _run_fp8(a, sa, w, sw, 2)
    assert flag == 2 and torch.equal(got, _expect(a, sa, w, sw).float())
    # a W code that the row's 0xFF scale leaves out, but no other row's
    w[5, 3 * 128 + 1] = 0x7F
    got, flag = _run_fp8(a, sa, w, sw, 2)
    assert flag == 3 and torch.equal(got, _expect(a, sa, w, sw).float())


def _run_grouped(t, g, n, k, w, sw, seed):
    """launch_grouped_fp8_gemm on integer rows: (output, flag, the float64
    activations [t, g, k] its quantised rows stand for)."""
    import torch

    from pih_amd.device import ptr, stream_handle

    x = _ints((t * g, k), seed, 100).bfloat16()
    aq = torch.empty(t * g, k, dtype=torch.uint8, device="cuda")
    sa = torch.empty(t * g, k // 128, dtype=torch.uint8, device="cuda")
    out = torch.full((t, g * n), float("nan"), dtype=torch.bfloat16, device="cuda")
    flag = torch.zeros(1, dtype=torch.int32, device="cuda")
    r = abi.request(abi.DS["grouped_fp8_gemm"], input_bf16=ptr(x), activation_e4m3=ptr(aq),
                    activation_scale_bits=ptr(sa), weight_e4m3=ptr(w), weight_scale_bits=ptr(sw), output_bf16=ptr(out),
                    error_flag_u32=ptr(flag), stream=stream_handle(), token_count=t, group_count=g,
                    output_per_group=n, input_per_group=k)
    st = abi.deepseek_pack().call("launch_grouped_fp8_gemm", r)
    assert st.code == abi.OK, st
    torch.cuda.synchronize()
    av = (aq.view(torch.float8_e4m3fn).double().view(t, g, k // 128, 128) *
          torch.exp2(sa.double() - 127).view(t, g, k // 128, 1)).view(t, g, k)
    return out, int(flag.item()), av


def _check_grouped(out, av, w, sw, g, n):
    """fp32 sums of codes up to 448 are not exact, so k terms' rounding bounds
    the error (k x 2^-24 of the sum of magnitudes) beside bf16's half ulp."""
    k = w.shape[1]
    for q in range(g):
        wq, sq = w[q * n:(q + 1) * n], sw[q * n // 128:(q + 1) * n // 128]
        ref = _product(av[:, q], wq, sq)
        mag = _product(av[:, q].abs(), wq & 0x7F, sq)
        err = (out[:, q * n:(q + 1) * n].double() - ref).abs()
        assert bool((err <= ref.abs() * 2.0 ** -8 + mag * k * 2.0 ** -24).all())


# tiles of 16 x 16, 48 x 16, 80 x 64 (an odd number of row blocks, walked in
# pairs of waves) and the walked 128 x 128
@pytest.mark.parametrize("m,n,k", [(4, 1024, 512), (40, 1024, 2048), (301, 4096, 1024), (130, 32768, 1024)])
def test_fp8_many_codes(eng, m, n, k):
    """A whole A row and a whole W row of NaN codes and scattered ones: every
    element that a wave sums again, and those beside them, are exact."""
    import torch

    a, sa, w, sw = _fp8(m, n, k, 3 * m)
    a[m - 1], w[n // 2 + 1] = 0xFF, 0x7F
    g = torch.Generator(device="cuda")
    g.manual_seed(m)
    for t, rows in ((a, m), (w, n)):
        at = torch.randint(0, rows * k, (5,), device="cuda", generator=g)
        t.view(-1)[at] = 0x7F
    for out_type in (1, 2):
        got, flag = _run_fp8(a, sa, w, sw, out_type)
        ref = _expect(a, sa, w, sw).float()
        assert flag == 1 and torch.equal(got, ref.bfloat16() if out_type == 1 else ref)


@pytest.mark.parametrize("m,n,k", [(4, 1024, 4096), (64, 1024, 4096)])
def test_fp8_code_costs_no_scan_per_element(eng, m, n, k):
    """One NaN code in an A row makes its n sums start over: n / 16 blocks of
    them.  Shared by the waves that is a few clean calls; a lane walking K
    alone for each took 300 to 600 of them."""
    import torch

    a, sa, w, sw = _fp8(m, n, k, 1)
    bad = a.clone()
    bad[m // 2, 5] = 0xFF

    def best(rows):
        times = []
        for _ in range(8):
            start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            _run_fp8(rows, sa, w, sw, 1)
            stop.record()
            stop.synchronize()
            times.append(start.elapsed_time(stop))
        return min(times)

    best(a)
    assert best(bad) < best(a) + 0.5


@pytest.mark.parametrize("t", [1, 7, 65, 130])
def test_grouped_fp8_exact(eng, t):
    """Strided problems: 4 groups of 256 x 512 over interleaved rows."""
    g, n, k = 4, 256, 512
    _, _, w, sw = _fp8(1, g * n, k, t)
    out, flag, av = _run_grouped(t, g, n, k, w, sw, t)
    assert flag == 0
    _check_grouped(out, av, w, sw, g, n)


# one-tile-per-block tiles (16 x 16 and 48 x 64) and walked tiles (192 x 128)
@pytest.mark.parametrize("t,n,k", [(1, 256, 512), (7, 256, 512), (65, 2048, 1024), (700, 2048, 1024)])
def test_grouped_fp8_codes_under_an_invalid_scale(eng, t, n, k):
    """The grouped entry checks no codes; a W block under a 0xFF scale is left
    out unseen all the same, NaN codes included: bit 1024 alone, and every
    column finite."""
    g = 4
    _, _, w, sw = _fp8(1, g * n, k, t)
    sw[1, 2] = 255  # W rows 128..255 of group 0, k 256..383
    w[130, 256], w[255, 383] = 0x7F, 0xFF
    sw[-1, 0] = 255
    w[-1, 0:128] = 0xFF
    out, flag, av = _run_grouped(t, g, n, k, w, sw, t)
    assert flag == 1024
    _check_grouped(out, av, w, sw, g, n)


def test_lm_head_nonfinite_bits_many_rows(eng):
    """Above 128 rows the DeepSeek head runs on the per-shape tiles: a
    non-finite logit is stored and raises 128, the element behind it 64."""
    import torch

    from pih_amd.device import flag_value
    from pih_amd.linear import deepseek_lm_head

    x, w = _ints((150, 4096), 3).bfloat16(), _ints((129280, 4096), 4).bfloat16()
    out, flag = deepseek_lm_head(x, w)
    torch.cuda.synchronize()
    ref = torch.cat([(x.double() @ v.double().T).float() for v in w.split(16160)], dim=1)
    assert flag_value(flag) == 0 and torch.equal(out, ref)
    w[70000, 9] = float("inf")
    out, flag = deepseek_lm_head(x, w)
    torch.cuda.synchronize()
    assert flag_value(flag) == 128 | 64
    keep = np.arange(129280) != 70000
    assert torch.equal(out[:, keep], ref[:, keep]) and not bool(torch.isfinite(out[:, 70000]).any())
