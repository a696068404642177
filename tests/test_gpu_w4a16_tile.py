"""GPU parity of the W4A16 tiles (w4a16_tile.hip), 2-32 rows, one problem and
groups, both formats.

x holds integers in [-3, 3] and the scales are powers of two within a factor
of 4: every product and partial sum is a multiple of one power of two below
2^24 of it, exact in fp32 in any order, so the output must equal the float64
product rounded to bf16, bit for bit."""
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


def _weights(n, k, sym, seed):
    """(qweight, scales, zeros or None, float64 [n, k] values)"""
    import torch

    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    s = torch.exp2(torch.randint(-2, 1, (n, k // 128), device="cuda", generator=g).float())
    if sym:
        q = torch.randint(-7, 8, (n, k), device="cuda", generator=g)
        u = (q & 15).to(torch.uint8)
        packed, scales, zeros, v = u[:, 0::2] | (u[:, 1::2] << 4), s.half(), None, q
    else:
        q = torch.randint(0, 16, (n, k), device="cuda", generator=g)
        z = torch.randint(0, 16, (n, -(-k // 1024) * 8), device="cuda", generator=g)
        shift = torch.arange(0, 32, 4, device="cuda")
        packed = (q.view(n, k // 8, 8) << shift).sum(2).to(torch.int32)
        zeros = (z.view(n, -1, 8) << shift).sum(2).to(torch.int32)
        scales, v = s.bfloat16(), q - z[:, :k // 128].repeat_interleave(128, 1)
    return packed.contiguous(), scales, zeros, v.double() * s.double().repeat_interleave(128, 1)


def _run(x, ws, sym, flag=None):
    import torch

    from pih_amd.device import ptr, stream_handle

    m, k = x.shape
    flag = torch.zeros(1, dtype=torch.int32, device="cuda") if flag is None else flag
    out = [torch.full((m, w[1].shape[0]), float("nan"), dtype=torch.bfloat16, device="cuda") for w in ws]
    probs = (abi.W4A16_PROBLEM * len(ws))()
    for p, (q, s, z, _), o in zip(probs, ws, out):
        p.input_bf16, p.qweight, p.scales, p.zeros, p.output_bf16, p.n = ptr(x), ptr(q), ptr(s), ptr(z), ptr(o), o.shape[1]
    r = abi.request(abi.LN["w4a16_grouped"], problems=abi.C.addressof(probs), error_flag_u32=ptr(flag),
                    stream=stream_handle(), problem_count=len(ws), m=m, k=k,
                    format=abi.W4A16_SYMMETRIC if sym else abi.W4A16_ASYMMETRIC)
    st = abi.linear_pack().call("launch_w4a16_grouped", r)
    assert st.code == abi.OK, st
    torch.cuda.synchronize()
    return out, int(flag.item())


def _x(m, k, seed):
    import torch

    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randint(-3, 4, (m, k), device="cuda", generator=g).bfloat16()


# 1, 2, 3, 4 and 6 weight blocks a tile; one K step, fewer steps than stages,
# many; rows at the edges of the 16- and 32-row operands; k 640 (not a
# multiple of 512), 12800 (past the panels), 2 rows of 512 blocks, 9 and 17
# rows of few blocks and short K stay on the GEMV
@pytest.mark.parametrize("sym", [False, True])
@pytest.mark.parametrize("m,ns,k", [(2, (8192,), 512), (4, (12288, 12288), 1024), (5, (4096, 1024, 1024), 1536),
                                    (9, (48,), 512), (15, (16, 32, 4096), 2560), (16, (12288, 12288), 4096),
                                    (16, (6144,), 12288), (17, (64,), 4096), (31, (9216, 96), 1024),
                                    (32, (4096, 4096), 2048), (8, (4096,), 640), (20, (256,), 12800),
                                    (2, (16384,), 512), (9, (48,), 1536), (14, (4096,), 4096), (15, (4096,), 512),
                                    (17, (1024,), 1024), (17, (1024,), 1536)])
def test_exact(eng, m, ns, k, sym):
    import torch

    x = _x(m, k, m + k)
    ws = [_weights(n, k, sym, n + k + i) for i, n in enumerate(ns)]
    out, flag = _run(x, ws, sym)
    assert flag == 0
    for o, w in zip(out, ws):
        assert torch.equal(o, (x.double() @ w[3].T).float().bfloat16())


@pytest.mark.parametrize("m,n", [(16, 256), (32, 768)])
def test_error_codes(eng, m, n):
    """12 a reserved nibble, 13 a scale not finite and positive, 14 a
    non-finite output; the first code stays."""
    import torch

    x = _x(m, 1024, 1)
    w = _weights(n, 1024, True, 2)
    w[0][n - 1, 500] = 0x18  # low nibble 8
    assert _run(x, [w], True)[1] == 12
    for bad in (0.0, float("inf")):
        w = _weights(n, 1024, False, 3)
        w[1][n // 2, 7] = bad
        assert _run(x, [w], False)[1] == 13
    w = _weights(n, 1024, False, 4)
    x[m - 1, 1000] = float("inf")
    out, flag = _run(x, [w], False)
    assert flag == 14 and bool(torch.isfinite(out[0][:m - 1]).all())
    flag = torch.full((1,), 99, dtype=torch.int32, device="cuda")
    assert _run(x, [w], False, flag)[1] == 99
