"""The calls a model host makes through the gfx950 packs, as measurable cases.

Six kinds of work, each over the range of batch rows it meets in use:

  qwen_mlp   the Qwen3 BF16 MLP block (``QwenMlpBlock``), decode batches
  bf16       the seven Qwen3-8B BF16 projections of one layer
             (``launch_bf16_gemm`` with the queried workspace), one decode
             row up to a 2048-row prefill
  w4a16      the same seven projections with INT4 weights, as a decode step
             issues them (``launch_w4a16_grouped``: [q, k, v], o, [gate, up],
             down), asymmetric or symmetric format
  fp8        the five DeepSeek dense FP8 projections (``launch_fp8_gemm`` of
             the DeepSeek table, UE8M0 scales), decode to prefill
  moe        one MoE expert layer (``MoeLayer``): FP8 experts with fp32
             scales, or MXFP4 experts with e4m3 or bf16 activations, at the
             hidden 7168 / top-8 and the hidden 4096 / top-6 geometry
  lm_head    the DeepSeek LM head (``launch_lm_head``), fp32 logits

Weights, buffers and request structs are made in ``prepare``, as a host holds
them; ``run`` only makes the calls.  Routing follows a Zipf(1.1) expert skew.
"""
import math

import torch

from pih_amd import abi
from pih_amd.device import engine_stream, error_flag, ptr, stream_handle
from pih_amd.linear import MoeLayer, QwenMlpBlock, bf16_gemm_workspace

# Qwen3-8B projections as (N, K): q, k, v, o, gate, up, down
QWEN8B = ((4096, 4096), (1024, 4096), (1024, 4096), (4096, 4096), (12288, 4096), (12288, 4096), (4096, 12288))
# which of them a grouped W4A16 launch takes together (one input each)
W4A16_GROUPS = ((0, 1, 2), (3,), (4, 5), (6,))
# DeepSeek-V4-Flash dense FP8 projections as (N, K)
DS_FP8 = ((1024, 4096), (32768, 1024), (4096, 8192), (2048, 4096), (4096, 2048))
# MoE geometries: hidden, intermediate, top-k, SwiGLU clamp
MOE = {"h7168": (7168, 2048, 8, 0.0), "h4096": (4096, 2048, 6, 10.0)}
EXPERTS = 256
VOCAB, VOCAB_HIDDEN = 129280, 4096
E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


def listed():
    return [
        # Qwen3-0.6B MLP block on a 16-row decode batch: the smallest call,
        # four short launches
        {"name": "qwen_mlp_m16", "kind": "qwen_mlp", "hidden": 1024, "inter": 3072, "m": 16},
        # one decode step of one Qwen3-8B layer, single request
        {"name": "bf16_m1", "kind": "bf16", "m": 1},
        # a decode step for a ragged batch of concurrent requests
        {"name": "bf16_m57", "kind": "bf16", "m": 57},
        # prefill of a 2048-token prompt
        {"name": "bf16_m2048", "kind": "bf16", "m": 2048},
        # INT4 decode, single request and a batch of 16
        {"name": "w4a16_m1", "kind": "w4a16", "m": 1, "symmetric": False},
        {"name": "w4a16_m16", "kind": "w4a16", "m": 16, "symmetric": False},
        # DeepSeek dense FP8 projections: a decode step and a ragged
        # chunked-prefill batch
        {"name": "fp8_m4", "kind": "fp8", "m": 4},
        {"name": "fp8_m301", "kind": "fp8", "m": 301},
        # MoE expert layer: 4096-token prefill with FP8 experts (the largest
        # call), decode batches of 64 and 512 tokens with MXFP4 experts
        {"name": "moe_fp8_t4096", "kind": "moe", "geometry": "h7168", "weights": "fp8", "act": "e4m3", "tokens": 4096},
        {"name": "moe_mxfp4_t64", "kind": "moe", "geometry": "h7168", "weights": "mxfp4", "act": "e4m3", "tokens": 64},
        {"name": "moe_mxfp4_t512", "kind": "moe", "geometry": "h7168", "weights": "mxfp4", "act": "bf16",
         "tokens": 512},
        # logits of a 33-request decode batch
        {"name": "lm_head_m33", "kind": "lm_head", "m": 33},
    ]


def _log_int(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    shapes = [{k: v for k, v in c.items() if k != "name"} for c in listed()]
    while True:
        case = _draw(rng)
        if case not in shapes:
            return case


def _draw(rng):
    kind = rng.choice(("qwen_mlp", "bf16", "bf16", "w4a16", "fp8", "fp8", "moe", "moe", "lm_head"))
    if kind == "qwen_mlp":
        hidden = rng.choice((1024, 2048, 2560))
        return {"kind": kind, "hidden": hidden, "inter": 3 * hidden, "m": _log_int(rng, 1, 64)}
    if kind == "bf16":
        return {"kind": kind, "m": _log_int(rng, 1, 2048)}
    if kind == "w4a16":
        return {"kind": kind, "m": _log_int(rng, 1, 32), "symmetric": rng.random() < 0.3}
    if kind == "fp8":
        return {"kind": kind, "m": _log_int(rng, 1, 2048)}
    if kind == "lm_head":
        return {"kind": kind, "m": _log_int(rng, 1, 256)}
    geometry = rng.choice(("h7168", "h4096"))
    if geometry == "h7168" and rng.random() < 0.4:
        return {"kind": kind, "geometry": geometry, "weights": "fp8", "act": "e4m3", "tokens": _log_int(rng, 32, 4000)}
    act = "e4m3" if geometry == "h4096" else rng.choice(("e4m3", "bf16"))
    return {"kind": kind, "geometry": geometry, "weights": "mxfp4", "act": act, "tokens": _log_int(rng, 16, 1024)}


# ------------------------------------------------------------------ inputs
def _gen(seed, device="cuda"):
    g = torch.Generator(device=device)
    g.manual_seed(0x5049_4800 + int(seed))
    return g


def _normal(g, shape, std=1.0):
    return (torch.randn(shape, device=g.device, generator=g) * std).to(torch.bfloat16)


def _route(g, tokens, topk):
    """Softmax top-k over logits N(0, 1) with a Zipf(1.1) bias over a seeded
    expert permutation, weights renormalised."""
    rank = torch.randperm(EXPERTS, device=g.device, generator=g)
    z = torch.randn(tokens, EXPERTS, device=g.device, generator=g) - 1.1 * torch.log1p(rank.float())
    top, ids = torch.topk(z, topk, dim=1)
    return ids.to(torch.int32).contiguous(), torch.softmax(top, dim=1).contiguous()


def _fp8_rows(v):
    """[R, K] values -> (e4m3 codes, UE8M0 bytes [R, K/128])."""
    r, k = v.shape
    x = v.view(r, k // 128, 128)
    e = torch.ceil(torch.log2(x.abs().amax(2).clamp_min(1e-4).double() / 448.0)).float()
    q = (x / torch.exp2(e)[:, :, None]).clamp(-448, 448).to(torch.float8_e4m3fn)
    return q.view(torch.uint8).view(r, k), (e + 127).to(torch.uint8)


def _fp8_blocks(v, ue8m0):
    """[N, K] values -> (e4m3 codes, scales [N/128, K/128]), UE8M0 or fp32."""
    n, k = v.shape
    x = v.view(n // 128, 128, k // 128, 128)
    s = x.abs().amax(dim=(1, 3)).clamp_min(1e-12) / 448.0
    if ue8m0:
        e = torch.ceil(torch.log2(s.double())).float()
        s, stored = torch.exp2(e), (e + 127).to(torch.uint8)
    else:
        stored = s
    q = (x / s[:, None, :, None]).clamp(-448, 448).to(torch.float8_e4m3fn)
    return q.view(torch.uint8).view(n, k), stored


def _mxfp4(g, n, k):
    """e2m1 codes of normal weights (std about 0.02) and UE8M0 scales."""
    z = (torch.randn(n, k, device=g.device, generator=g) * 2.0).to(torch.bfloat16)
    edges = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=g.device, dtype=torch.bfloat16)
    c = torch.bucketize(z.abs(), edges).to(torch.uint8) | ((z < 0).to(torch.uint8) << 3)
    return c[:, 0::2] | (c[:, 1::2] << 4), torch.randint(119, 122, (n, k // 32), device=g.device, generator=g,
                                                         dtype=torch.uint8)


def _tensors(case, seed):
    g = _gen(seed)
    dev = g.device
    kind = case["kind"]
    t = {}
    if kind == "qwen_mlp":
        h, i = case["hidden"], case["inter"]
        t.update(x=_normal(g, (case["m"], h)), wg=_normal(g, (i, h), 0.02), wu=_normal(g, (i, h), 0.02),
                 wd=_normal(g, (h, i), 0.02))
    elif kind == "bf16":
        t.update(x={k: _normal(g, (case["m"], k)) for k in (4096, 12288)},
                 w=[_normal(g, s, 0.02) for s in QWEN8B])
    elif kind == "w4a16":
        t["x"] = {k: _normal(g, (case["m"], k)) for k in (4096, 12288)}
        t["w"] = []
        for n, k in QWEN8B:
            s = torch.rand(n, k // 128, device=dev, generator=g) * 0.019 + 0.001
            if case["symmetric"]:
                q = torch.randint(-7, 8, (n, k), device=dev, generator=g, dtype=torch.int8).view(torch.uint8) & 15
                t["w"].append((q[:, 0::2] | (q[:, 1::2] << 4), s.to(torch.float16), None))
            else:
                q = torch.randint(-2 ** 31, 2 ** 31, (n, k // 8), device=dev, generator=g, dtype=torch.int64)
                z = torch.randint(-2 ** 31, 2 ** 31, (n, -(-k // 1024)), device=dev, generator=g, dtype=torch.int64)
                t["w"].append((q.to(torch.int32), s.to(torch.bfloat16), z.to(torch.int32)))
    elif kind == "fp8":
        t["a"] = [_fp8_rows(torch.randn(case["m"], k, device=dev, generator=g)) for _, k in DS_FP8]
        t["w"] = [_fp8_blocks(torch.randn(n, k, device=dev, generator=g) * 0.02, True) for n, k in DS_FP8]
    elif kind == "lm_head":
        t["x"] = _normal(g, (case["m"], VOCAB_HIDDEN))
        t["w"] = _normal(g, (VOCAB, VOCAB_HIDDEN), 0.02)
    else:
        h, i, topk, _ = MOE[case["geometry"]]
        t["x"] = _normal(g, (case["tokens"], h))
        t["ids"], t["wts"] = _route(g, case["tokens"], topk)
        for name, n, k in (("w13", 2 * i, h), ("w2", h, i)):
            fp8 = case["weights"] == "fp8"
            w = torch.empty(EXPERTS, n, k if fp8 else k // 2, dtype=torch.uint8, device=dev)
            s = (torch.empty(EXPERTS, n // 128, k // 128, dtype=torch.float32, device=dev) if fp8 else
                 torch.empty(EXPERTS, n, k // 32, dtype=torch.uint8, device=dev))
            for e in range(EXPERTS):
                if fp8:
                    w[e], s[e] = _fp8_blocks(torch.randn(n, k, device=dev, generator=g) * 0.02, False)
                else:
                    w[e], s[e] = _mxfp4(g, n, k)
            t[name], t[name + "_scale"] = w, s
    return t


def _checked(pack, entry, request):
    fn = getattr(pack.table, entry)
    byref = abi.C.byref(request)

    def call():
        st = fn(byref)
        if st.code != abi.OK:
            raise RuntimeError(f"{entry}: {st!r}")
    return call


def prepare(case, seed):
    t = _tensors(case, seed)
    kind = case["kind"]
    torch.cuda.synchronize()  # the inputs were made on torch's default stream, the calls use the engine's
    with engine_stream():
        s = stream_handle()
        flag = error_flag()
        state = {"keep": (t, flag)}
        new = lambda m, n, dt=torch.bfloat16: torch.empty(m, n, dtype=dt, device="cuda")  # noqa: E731
        if kind == "qwen_mlp":
            block = QwenMlpBlock(t["wg"], t["wu"], t["wd"], case["m"])
            state.update(calls=[lambda: block.forward(t["x"])], out=block.out, block=block)
        elif kind == "bf16":
            m, L = case["m"], abi.linear_pack()
            need = [bf16_gemm_workspace(m, n, k) for n, k in QWEN8B]
            ws = torch.empty(max(max(need), 16), dtype=torch.uint8, device="cuda")
            out = [new(m, n) for n, _ in QWEN8B]
            reqs = [abi.request(abi.LN["bf16_gemm"], a_bf16=ptr(t["x"][k]), w_bf16=ptr(t["w"][j]), output=ptr(out[j]),
                                workspace=ptr(ws) if need[j] else 0, workspace_bytes=need[j], stream=s, m=m, n=n, k=k,
                                output_type=abi.OUTPUT_BF16) for j, (n, k) in enumerate(QWEN8B)]
            state.update(calls=[_checked(L, "launch_bf16_gemm", r) for r in reqs], out=out, ws=ws)
        elif kind == "w4a16":
            m, L = case["m"], abi.linear_pack()
            out = [new(m, n) for n, _ in QWEN8B]
            calls = []
            for group in W4A16_GROUPS:
                probs = (abi.W4A16_PROBLEM * len(group))()
                k = QWEN8B[group[0]][1]
                for p, j in zip(probs, group):
                    q, sc, z = t["w"][j]
                    p.input_bf16, p.qweight, p.scales, p.zeros = ptr(t["x"][k]), ptr(q), ptr(sc), ptr(z)
                    p.output_bf16, p.n = ptr(out[j]), QWEN8B[j][0]
                r = abi.request(abi.LN["w4a16_grouped"], problems=abi.C.addressof(probs), error_flag_u32=ptr(flag),
                                stream=s, problem_count=len(group), m=m, k=k,
                                format=abi.W4A16_SYMMETRIC if case["symmetric"] else abi.W4A16_ASYMMETRIC)
                calls.append(_checked(L, "launch_w4a16_grouped", r))
                state.setdefault("problems", []).append(probs)
            state.update(calls=calls, out=out)
        elif kind == "fp8":
            m, D = case["m"], abi.deepseek_pack()
            out = [new(m, n) for n, _ in DS_FP8]
            reqs = [abi.request(abi.DS["fp8_gemm"], activation_e4m3=ptr(t["a"][j][0]),
                                activation_scale_bits=ptr(t["a"][j][1]), weight_e4m3=ptr(t["w"][j][0]),
                                weight_scale_bits=ptr(t["w"][j][1]), output=ptr(out[j]), error_flag=ptr(flag),
                                stream=s, m=m, n=n, k=k, output_type=1) for j, (n, k) in enumerate(DS_FP8)]
            state.update(calls=[_checked(D, "launch_fp8_gemm", r) for r in reqs], out=out)
        elif kind == "lm_head":
            m = case["m"]
            out = new(m, VOCAB, torch.float32)
            r = abi.request(abi.DS["lm_head"], input_bf16=ptr(t["x"]), weight_bf16=ptr(t["w"]), logits_f32=ptr(out),
                            error_flag_u32=ptr(flag), stream=s, output_rows=m, vocab_size=VOCAB,
                            hidden_size=VOCAB_HIDDEN)
            state.update(calls=[_checked(abi.deepseek_pack(), "launch_lm_head", r)], out=out)
        else:
            _, _, topk, limit = MOE[case["geometry"]]
            layer = MoeLayer(t["w13"], t["w13_scale"], t["w2"], t["w2_scale"], case["tokens"], topk,
                             weight_format=abi.WEIGHT_FP8 if case["weights"] == "fp8" else abi.WEIGHT_MXFP4,
                             scale_format=abi.SCALE_F32 if case["weights"] == "fp8" else abi.SCALE_UE8M0,
                             activation_type=abi.ACTIVATION_E4M3 if case["act"] == "e4m3" else abi.ACTIVATION_BF16,
                             swiglu_limit=limit)
            state.update(calls=[lambda: layer.forward(t["x"], t["ids"], t["wts"])], out=layer.out, layer=layer)
    return state


def run(state):
    with engine_stream():
        for call in state["calls"]:
            call()
    return state["out"]


# ------------------------------------------------------------------ floors
def work(case):
    kind = case["kind"]
    if kind == "qwen_mlp":
        m, h, i = case["m"], case["hidden"], case["inter"]
        return {"bytes": 3 * h * i * 2 + 2 * m * h * 2, "flops": 6 * m * h * i}
    if kind == "bf16":
        m = case["m"]
        return {"bytes": sum(n * k * 2 + m * n * 2 for n, k in QWEN8B) + 2 * m * (3 * 4096 + 12288),
                "flops": sum(2 * m * n * k for n, k in QWEN8B)}
    if kind == "w4a16":
        m = case["m"]
        zeros = 0 if case["symmetric"] else sum(n * -(-k // 1024) * 4 for n, k in QWEN8B)
        return {"bytes": sum(n * k // 2 + n * k // 64 + m * n * 2 for n, k in QWEN8B) + zeros
                + 2 * m * (3 * 4096 + 12288), "flops": sum(2 * m * n * k for n, k in QWEN8B)}
    if kind == "fp8":
        m = case["m"]
        return {"bytes": sum(n * k + n * k // 16384 + m * k + m * k // 128 + m * n * 2 for n, k in DS_FP8),
                "flops": sum(2 * m * n * k for n, k in DS_FP8)}
    if kind == "lm_head":
        m = case["m"]
        return {"bytes": VOCAB * VOCAB_HIDDEN * 2 + m * VOCAB_HIDDEN * 2 + m * VOCAB * 4,
                "flops": 2 * m * VOCAB * VOCAB_HIDDEN}
    h, i, topk, _ = MOE[case["geometry"]]
    ids, _ = _route(_gen(0, "cpu"), case["tokens"], topk)
    touched = int(torch.unique(ids).numel())  # of one routing; another seed's differs by a few experts
    per = 3 * h * i + 3 * h * i // 16384 * 4 if case["weights"] == "fp8" else 3 * h * i * 17 // 32
    return {"bytes": touched * per + case["tokens"] * (h * 4 + topk * 8),
            "flops": 6 * case["tokens"] * topk * h * i}


def tolerance(case):
    # measured against exact(): bf16 results are 1.7e-3 off by their own
    # rounding, the MoE layers (an intermediate rounded to bf16, and to e4m3
    # where a code may flip) and the MLP block 2e-3 to 3e-3, the fp32 logits
    # 3e-7 (sums of 4096 products)
    if case["kind"] == "lm_head":
        return {"rel": 2e-6, "max": 1e-4}
    if case["kind"] in ("moe", "qwen_mlp"):
        return {"rel": 1e-2, "max": 0.2}
    return {"rel": 7e-3, "max": 0.05}


# ------------------------------------------------------------- 64-bit form
def _e4m3(codes):
    return codes.view(torch.float8_e4m3fn).to(torch.float64)


def _e8m0(bits):
    return torch.exp2(bits.to(torch.float64) - 127)


def _dequant_rows(codes, s):
    r, k = codes.shape
    return (_e4m3(codes).view(r, k // 128, 128) * s[:, :, None]).view(r, k)


def _dequant_blocks(codes, s):
    n, k = codes.shape
    return (_e4m3(codes).view(n // 128, 128, k // 128, 128) * s.to(torch.float64)[:, None, :, None]).view(n, k)


def _dequant_mxfp4(packed, s):
    n, half = packed.shape
    table = torch.tensor(E2M1 + tuple(-v for v in E2M1), dtype=torch.float64, device=packed.device)
    v = torch.stack((table[(packed & 15).long()], table[(packed >> 4).long()]), dim=2).view(n, half // 16, 32)
    return (v * _e8m0(s)[:, :, None]).view(n, 2 * half)


def _act(x, case):
    """The activation values a MoE GEMM multiplies: e4m3 per 128 columns with
    an fp32 or UE8M0 scale, or bf16 as they are."""
    if case["act"] == "bf16":
        return x.to(torch.float64)
    if case["weights"] == "mxfp4":
        q, s = _fp8_rows(x.float())
        return _dequant_rows(q, _e8m0(s))
    r, k = x.shape
    v = x.float().view(r, k // 128, 128)
    # a tensor divisor: by a Python number torch multiplies with the rounded reciprocal
    s = v.abs().amax(2).clamp_min(1e-4) / torch.full((), 448.0, device=v.device)
    q = (v / s[:, :, None]).clamp(-448, 448).to(torch.float8_e4m3fn)
    return (q.to(torch.float64) * s.to(torch.float64)[:, :, None]).view(r, k)


def _silu_mul(g, u):
    return g / (1 + torch.exp(-g)) * u


def _exact_moe(case, t):
    h, i, topk, limit = MOE[case["geometry"]]
    tokens = case["tokens"]
    dequant = _dequant_blocks if case["weights"] == "fp8" else _dequant_mxfp4
    x = _act(t["x"], case)
    out = torch.zeros(tokens, h, dtype=torch.float64, device=x.device)
    for e in range(EXPERTS):
        tok, slot = torch.nonzero(t["ids"] == e, as_tuple=True)
        if not tok.numel():
            continue
        # the rounding points of the path: gate, up, the weighted product and
        # the expert's output are bf16
        gu = (x[tok] @ dequant(t["w13"][e], t["w13_scale"][e]).T).to(torch.bfloat16).to(torch.float64)
        gate, up = gu[:, :i], gu[:, i:]
        if limit:
            gate, up = gate.clamp(max=limit), up.clamp(-limit, limit)
        mid = (_silu_mul(gate, up) * t["wts"][tok, slot].to(torch.float64)[:, None]).to(torch.bfloat16)
        y = _act(mid, case) @ dequant(t["w2"][e], t["w2_scale"][e]).T
        out.index_add_(0, tok, y.to(torch.bfloat16).to(torch.float64))
    return out


def exact(case, seed):
    t = _tensors(case, seed)
    kind = case["kind"]
    d = lambda v: v.to(torch.float64)  # noqa: E731
    if kind == "qwen_mlp":
        g, u = ((d(t["x"]) @ d(t[w]).T).to(torch.bfloat16) for w in ("wg", "wu"))
        return d(_silu_mul(d(g), d(u)).to(torch.bfloat16)) @ d(t["wd"]).T
    if kind == "bf16":
        return [d(t["x"][k]) @ d(t["w"][j]).T for j, (_, k) in enumerate(QWEN8B)]
    if kind == "w4a16":
        out = []
        for (n, k), (q, s, z) in zip(QWEN8B, t["w"]):
            if case["symmetric"]:
                v = torch.stack((q & 15, q >> 4), dim=2).view(n, k).to(torch.int32)
                v = torch.where(v > 7, v - 16, v).view(n, k // 128, 128)
            else:
                shift = torch.arange(0, 32, 4, device=q.device, dtype=torch.int32)
                zero = ((z[:, :, None] >> shift) & 15).view(n, -1)[:, :k // 128]
                v = ((q[:, :, None] >> shift) & 15).view(n, k // 128, 128) - zero[:, :, None]
            out.append(d(t["x"][k]) @ (d(v) * d(s)[:, :, None]).view(n, k).T)
        return out
    if kind == "fp8":
        return [_dequant_rows(a, _e8m0(sa)) @ _dequant_blocks(w, _e8m0(sw)).T
                for (a, sa), (w, sw) in zip(t["a"], t["w"])]
    if kind == "lm_head":
        x = d(t["x"])
        return torch.cat([x @ d(w).T for w in t["w"].split(16160)], dim=1)
    return _exact_moe(case, t)
