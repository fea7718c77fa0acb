"""The work that a user of this library has it do, as cases to be timed and compared.

A served model of hidden size 5120 calls the library in two regimes, and the cases cover both over their range:

* up to 80 rows at once (a decode step, a verified draft tree, a batch of those): the weight-streaming GEMMs;
* more rows than that (a prompt, or a chunk of one): the prefill GEMMs, behind the quantizer that feeds them.

Each case is one block of a layer, called as a program calls it: the activations come in as the layer before left
them, the weights are in the tiled layout already, and the outputs are the block's.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ling-engine_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import ling_gemm as L  # noqa: E402

DEV = "cuda:0"
EPS = 1e-6
MAX_ROWS = 80

# widths of the matrices (out, in): the benchmark's hybrid model and its neighbours, with ragged ones among them
ROWS_SHAPES = ((5120, 5120), (7168, 5120), (12352, 5120), (5120, 6144), (5120, 17408), (2048, 4096), (1040, 2688),
               (8208, 1152), (32000, 5120))
PREFILL_SHAPES = ((5120, 5120), (7168, 5120), (5120, 6144), (5120, 17408), (17408, 5120), (34816, 5120), (2048, 4096),
                  (1152, 2688), (4224, 7552))


def listed():
    return [
        # one token through a square projection: the smallest call a decode step makes, latency and launch bound
        {"name": "decode_linear_m1", "kind": "rows_linear", "M": 1, "N": 5120, "K": 5120, "residual": False},
        # a 1 + 16 draft tree verified: the MLP of a layer, gate|up with SiLU*mul, then down onto the residual
        {"name": "verify_mlp_m17", "kind": "rows_mlp", "M": 17, "H": 5120, "F": 17408},
        # four sequences of 17 rows share one read of the MLP's weights
        {"name": "batch_mlp_m68", "kind": "rows_mlp", "M": 68, "H": 5120, "F": 17408},
        # the drafter's input projection: five hidden states of 16 draft rows, NVFP4 weights
        {"name": "drafter_fc_nvfp4_m16", "kind": "rows_nvfp4", "M": 16, "N": 5120, "K": 25600, "coded": False},
        # the FP16-copy interface: a norm, then two matrices in one launch; NVFP4 with coded scales, a few rows
        {"name": "norm_multi_nvfp4_m5", "kind": "rows_multi", "M": 5, "N": 17408, "K": 5120, "nvfp4": True},
        # the drafter's sparse head: some rows of a large vocabulary's matrix
        {"name": "sparse_head_m17", "kind": "gather", "M": 17, "N": 151936, "K": 5120, "cap": 2048},
        # a short prompt's QKV projection, block-scaled FP8
        {"name": "prompt_qkv_m200", "kind": "prefill_block", "M": 200, "N": 7168, "K": 5120},
        # an ordinary prompt's down projection, a ragged number of tokens
        {"name": "prompt_down_m1000", "kind": "prefill_block", "M": 1000, "N": 5120, "K": 17408},
        # a full prefill chunk's gate|up: the largest call
        {"name": "chunk_gate_up_m4096", "kind": "prefill_block", "M": 4096, "N": 34816, "K": 5120},
        # per-tensor FP8 into FP32: the attention's output projection of a prompt
        {"name": "prompt_out_fp8_m777", "kind": "prefill_tensor", "M": 777, "N": 5120, "K": 6144},
        # NVFP4 down projection of a short prompt, added to the residual
        {"name": "prompt_down_nvfp4_m300", "kind": "prefill_nvfp4", "M": 300, "N": 5120, "K": 17408},
        # NVFP4 FFN entry of a long prompt: norm and quantizer, gate and up with SwiGLU into the down projection's codes
        {"name": "chunk_swiglu_nvfp4_m2048", "kind": "prefill_swiglu", "M": 2048, "N": 17408, "K": 5120},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["rows_linear", "rows_mlp", "rows_nvfp4", "rows_multi", "gather", "prefill_block", "prefill_tensor",
                       "prefill_nvfp4", "prefill_swiglu", "prefill_block", "prefill_nvfp4"])
    if kind.startswith("rows") or kind == "gather":
        M = min(MAX_ROWS, _log_int(rng, 1, MAX_ROWS + 1))
        N, K = rng.choice(ROWS_SHAPES)
        if kind == "rows_mlp":
            H, F = rng.choice(((5120, 17408), (5120, 13824), (2048, 6144), (1152, 3072)))
            return {"kind": kind, "M": M, "H": H, "F": F}
        if kind == "rows_linear":
            return {"kind": kind, "M": M, "N": N, "K": K, "residual": rng.random() < 0.5}
        if kind == "rows_nvfp4":
            return {"kind": kind, "M": M, "N": N, "K": K, "coded": rng.random() < 0.3}
        if kind == "rows_multi":
            return {"kind": kind, "M": M, "N": N, "K": K, "nvfp4": rng.random() < 0.5}
        return {"kind": kind, "M": M, "N": rng.choice((32000, 65536, 151936)), "K": rng.choice((2048, 4096, 5120)),
                "cap": 32 * _log_int(rng, 8, 128)}
    M = _log_int(rng, MAX_ROWS + 1, 4096)
    N, K = rng.choice(PREFILL_SHAPES)
    if kind == "prefill_swiglu":
        N, K = rng.choice(((17408, 5120), (13824, 5120), (3072, 1024)))
    flops = 2.0 * M * N * K * (4.0 if kind == "prefill_swiglu" else 2.0 if kind == "prefill_nvfp4" else 1.0)
    if flops > 1.4e12:
        M = int(M * 1.4e12 / flops)
    return {"kind": kind, "M": M, "N": N, "K": K}


# ---------------- inputs ----------------
def _randn(gen, *shape, scale=1.0):
    return torch.randn(shape, device=DEV, generator=gen) * scale


def _fp8_channel(gen, N, K):
    """Weights N(0, 0.02) as FP8 with one scale per output channel: codes [N][K], scales [N]."""
    w = _randn(gen, N, K, scale=0.02)
    s = w.abs().amax(1) / 448.0
    return (w / s[:, None]).to(torch.float8_e4m3fn).view(torch.uint8), s


def _fp8_block(gen, N, K):
    """The same in 128 x 128 blocks: scales [N/128][K/128]."""
    w = _randn(gen, N, K, scale=0.02).view(N // 128, 128, K // 128, 128)
    s = w.abs().amax((1, 3)) / 448.0
    q = (w / s[:, None, :, None]).to(torch.float8_e4m3fn).view(torch.uint8)
    return q.view(N, K), s


def _nvfp4(gen, N, K):
    """The same as NVFP4: packed E2M1 codes [N][K/2], E4M3 scales [N][K/16], the global scale."""
    w = _randn(gen, N, K, scale=0.02)
    g = float(w.abs().max()) / (448.0 * 6.0)
    w = w.view(N, K // 16, 16)
    sc = (w.abs().amax(2) / 6.0 / g).clamp(2.0 ** -9, 448.0).to(torch.float8_e4m3fn)
    edges = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=DEV)
    w = w / (sc.float() * g)[:, :, None]
    code = torch.bucketize(w.abs(), edges, out_int32=True).to(torch.uint8)
    code = code | ((w < 0) & (code > 0)).to(torch.uint8) * 8
    code = code.view(N, K // 2, 2)
    return code[:, :, 0] | (code[:, :, 1] << 4), sc.view(torch.uint8).view(N, K // 16), g


def _e4m3(codes):
    return codes.view(torch.float8_e4m3fn).double()


_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0)


def _nvfp4_values(q, sc):
    """E2M1 code times E4M3 block scale, in 64 bits."""
    table = torch.tensor(_E2M1, dtype=torch.float64, device=DEV)
    rows, half = q.shape
    v = table[torch.stack((q & 15, q >> 4), 2).view(rows, 2 * half).int()]
    return (v.view(rows, half // 8, 16) * _e4m3(sc)[:, :, None]).view(rows, 2 * half)


def _inputs(case, seed):
    """What the seed gives, before the weights are laid out: codes row by row, scales, activations."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(int(seed))
    kind, M = case["kind"], case["M"]
    d = {}
    if kind == "rows_mlp":
        H, F = case["H"], case["F"]
        d["x"] = _randn(gen, M, H).to(torch.bfloat16)
        d["resid"] = _randn(gen, M, H).to(torch.bfloat16)
        for name, n, k in (("gate", F, H), ("up", F, H), ("down", H, F)):
            d[name], d["s_" + name] = _fp8_channel(gen, n, k)
        return d
    N, K = case["N"], case["K"]
    if kind == "rows_linear":
        d["x"] = _randn(gen, M, K).to(torch.bfloat16)
        d["w"], d["s"] = _fp8_channel(gen, N, K)
        d["resid"] = _randn(gen, M, N).to(torch.bfloat16) if case["residual"] else None
    elif kind == "rows_nvfp4":
        d["x"] = _randn(gen, M, K).to(torch.bfloat16)
        d["w"], d["sc"], d["g"] = _nvfp4(gen, N, K)
    elif kind == "rows_multi":
        d["x"] = _randn(gen, M, K)
        d["norm"] = _randn(gen, K, scale=0.1).to(torch.bfloat16)
        d["mats"] = [_nvfp4(gen, N, K) if case["nvfp4"] else _fp8_block_one(gen, N, K) for _ in range(2)]
    elif kind == "gather":
        d["x"] = _randn(gen, M, K).to(torch.bfloat16)
        d["w"], d["sc"], d["g"] = _nvfp4(gen, N, K)
        rows = torch.randperm(N, device=DEV, generator=gen)[: case["cap"]].to(torch.int32)
        d["rows"] = rows.contiguous()
        d["count"] = case["cap"] - 37  # the drafter keeps fewer than the buffer holds
    elif kind == "prefill_block":
        d["x"] = _randn(gen, M, K).to(torch.bfloat16)
        d["w"], d["s"] = _fp8_block(gen, N, K)
    elif kind == "prefill_tensor":
        d["x"] = _randn(gen, M, K).to(torch.bfloat16)
        d["w"], d["s"], _ = _fp8_block_one(gen, N, K)
        d["in_scale"] = 4.5 / 448.0
    elif kind == "prefill_nvfp4":
        d["x"] = _randn(gen, M, K)
        d["resid"] = _randn(gen, M, N)
        d["w"], d["sc"], d["g"] = _nvfp4(gen, N, K)
        d["in_scale"] = 4.5 / (448.0 * 6.0)
    else:
        d["x"] = _randn(gen, M, K)
        d["norm"] = _randn(gen, K, scale=0.1).to(torch.bfloat16)
        d["gate"], d["up"] = _nvfp4(gen, N, K), _nvfp4(gen, N, K)
        d["in_scale"], d["out_scale"] = 4.5 / (448.0 * 6.0), 10.0 / (448.0 * 6.0)
    return d


def _fp8_block_one(gen, N, K):
    """FP8 with one scale for the whole matrix."""
    w = _randn(gen, N, K, scale=0.02)
    s = float(w.abs().max()) / 448.0
    return (w / s).to(torch.float8_e4m3fn).view(torch.uint8), s, None


def _coded(values, scales):
    """The blob with 6-bit scale codes where the matrix has few enough scales, as a loader chooses: (blob, table, raw)."""
    ok, table, code_of = L.scale_code_table(scales.cpu().numpy())
    if not ok:
        return L.retile_nvfp4(values, scales), None, None
    blob, raw = L.retile_nvfp4_coded(values, scales, torch.from_numpy(code_of).to(DEV))
    return blob, torch.from_numpy(table).to(DEV), raw


def prepare(case, seed):
    """The layer's weights in the tiled layout and its input, as a program holds them between calls."""
    L.init()
    kind, d = case["kind"], _inputs(case, seed)
    s = dict(case)
    if kind == "rows_mlp":
        s.update(x=d["x"], resid=d["resid"])
        for name in ("gate", "up", "down"):
            s[name], s["s_" + name] = L.retile_fp8(d[name]), d["s_" + name]
    elif kind == "rows_linear":
        s.update(x=d["x"], w=L.retile_fp8(d["w"]), s=d["s"], resid=d["resid"])
    elif kind == "rows_nvfp4":
        blob, table, _ = _coded(d["w"], d["sc"]) if case["coded"] else (L.retile_nvfp4(d["w"], d["sc"]), None, None)
        s.update(x=d["x"], w=blob, table=table, g=d["g"])
    elif kind == "rows_multi":
        targets = []
        for q, sc, g in d["mats"]:
            y = torch.empty((case["M"], case["N"]), dtype=torch.float32, device=DEV)
            blob, table = _coded(q, sc)[:2] if case["nvfp4"] else (L.retile_fp8(q), None)
            targets.append((blob, table, g if case["nvfp4"] else sc, y, case["N"]))
        s.update(x=d["x"], norm=d["norm"], targets=targets)
    elif kind == "gather":
        s.update(x=d["x"], w=L.retile_nvfp4(d["w"], d["sc"]), g=d["g"], rows=d["rows"],
                 count=torch.tensor([d["count"]], dtype=torch.int32, device=DEV))
    elif kind in ("prefill_block", "prefill_tensor"):
        s.update(x=d["x"], w=L.retile_fp8(d["w"]), s=d["s"], in_scale=d.get("in_scale"))
    elif kind == "prefill_nvfp4":
        s.update(x=d["x"], resid=d["resid"], w=L.retile_nvfp4(d["w"], d["sc"]), g=d["g"], in_scale=d["in_scale"])
    else:
        s.update(x=d["x"], norm=d["norm"], gate=L.retile_nvfp4(*d["gate"][:2]), up=L.retile_nvfp4(*d["up"][:2]),
                 g_gate=d["gate"][2], g_up=d["up"][2], in_scale=d["in_scale"], out_scale=d["out_scale"])
    return s


def run(s):
    kind = s["kind"]
    if kind == "rows_linear":
        if s["resid"] is not None:
            return L.stream_fp8_pc_residual(s["x"], s["w"], s["s"], s["resid"], s["N"])
        return L.stream_fp8_pc(s["x"], s["w"], s["s"], s["N"])
    if kind == "rows_mlp":
        h = L.stream_fp8_pc_silu_mul(s["x"], s["gate"], s["s_gate"], s["up"], s["s_up"], s["F"])
        return h, L.stream_fp8_pc_residual(h, s["down"], s["s_down"], s["resid"], s["H"])
    if kind == "rows_nvfp4":
        return L.stream_nvfp4_bf16(s["x"], s["w"], s["table"], s["g"], s["N"])
    if kind == "rows_multi":
        out, xh, xinv = L.rmsnorm_half(s["x"], s["norm"], EPS)
        L.stream_gemm_multi(s["nvfp4"], xh, xinv, s["targets"], s["K"])
        return [out] + [t[3] for t in s["targets"]]
    if kind == "gather":
        xh, xinv = L.bf16_to_half_rows(s["x"])
        return L.stream_gemm_gather_nvfp4(xh, xinv, s["w"], None, s["g"], s["rows"], s["count"], s["cap"], s["N"], s["K"])
    if kind == "prefill_block":
        q, xs = L.quant_act_fp8_g128(s["x"])
        return L.prefill_fp8_block(q, xs, s["w"], s["s"], s["N"])
    if kind == "prefill_tensor":
        q = L.quant_act_fp8_bf16in(s["x"], s["in_scale"])
        return L.prefill_gemm_fp8(q, s["w"], s["in_scale"] * s["s"], s["N"])
    if kind == "prefill_nvfp4":
        q, sf = L.quant_act_nvfp4(s["x"], s["in_scale"])
        y = s["resid"].clone()  # the layer's input stays; the sum is its output
        return L.prefill_gemm_nvfp4(q, sf, s["w"], s["in_scale"] * s["g"], s["N"], y=y, accumulate=True)
    _, q, sf = L.rmsnorm_quant(s["x"], s["norm"], EPS, True, s["in_scale"], with_out=False)
    return L.prefill_swiglu_nvfp4(q, sf, s["gate"], s["in_scale"] * s["g_gate"], s["up"], s["in_scale"] * s["g_up"], s["N"],
                                  s["out_scale"])


# ---------------- the work, the tolerance, the exact results ----------------
def work(case):
    kind, M = case["kind"], case["M"]
    if kind == "rows_mlp":
        H, F = case["H"], case["F"]
        # weights and scales, the input and the residual, h written and the sum written (h stays on the chip's side)
        return {"bytes": 3 * H * F + 4 * (2 * F + H) + 2 * M * H * 3 + 2 * M * F, "flops": 6.0 * M * H * F}
    N, K = case["N"], case["K"]
    flops = 2.0 * M * N * K
    fp4 = N * K // 2 + N * K // 16
    if kind == "rows_linear":
        return {"bytes": N * K + 4 * N + 2 * M * K + 2 * M * N * (2 if case["residual"] else 1), "flops": flops}
    if kind == "rows_nvfp4":
        return {"bytes": fp4 + 2 * M * K + 2 * M * N, "flops": flops}
    if kind == "rows_multi":
        return {"bytes": 2 * (fp4 if case["nvfp4"] else N * K) + 2 * 4 * M * K + 2 * K + 2 * 4 * M * N, "flops": 2 * flops}
    if kind == "gather":
        cap = case["cap"]
        return {"bytes": cap * (K // 2 + K // 16) + 2 * M * K + 4 * M * cap + 4 * cap, "flops": 2.0 * M * cap * K}
    if kind == "prefill_block":
        return {"bytes": N * K + N * K // 4096 + 2 * M * K + 2 * M * N, "flops": flops}
    if kind == "prefill_tensor":
        return {"bytes": N * K + 2 * M * K + 4 * M * N, "flops": flops}
    if kind == "prefill_nvfp4":
        return {"bytes": fp4 + 4 * M * K + 2 * 4 * M * N, "flops": flops}
    return {"bytes": 2 * fp4 + 4 * M * K + 2 * K + M * N // 2 + M * N // 16, "flops": 2 * flops}


def tolerance(case):
    kind = case["kind"]
    if kind in ("rows_linear", "rows_mlp", "rows_nvfp4", "prefill_block"):
        return {"rel": 7e-3}  # BF16 outputs: 1.7e-3 from the result in 64 bits, the rounding of the output alone
    if kind == "prefill_tensor":
        return {"rel": 2e-4}  # the FP8 matrix instruction adds the products of a block at reduced precision
    if kind in ("rows_multi", "gather"):
        return {"rel": 1e-3}  # the FP16 copy of the activations
    if kind == "prefill_nvfp4":
        return {"rel": 1e-5}  # exact products, 32-bit sums
    return {"rel": 0.0, "differ": 2e-3}  # codes: a sum in another order moves the values that lie on a boundary


def exact(case, seed):
    kind, d = case["kind"], _inputs(case, seed)
    if kind == "rows_linear":
        y = d["x"].double() @ (_e4m3(d["w"]) * d["s"].double()[:, None]).t()
        return y if d["resid"] is None else y + d["resid"].double()
    if kind == "rows_mlp":
        x = d["x"].double()
        gate = x @ (_e4m3(d["gate"]) * d["s_gate"].double()[:, None]).t()
        up = x @ (_e4m3(d["up"]) * d["s_up"].double()[:, None]).t()
        h = torch.nn.functional.silu(gate) * up
        return h, h @ (_e4m3(d["down"]) * d["s_down"].double()[:, None]).t() + d["resid"].double()
    if kind == "rows_nvfp4":
        return (d["x"].double() @ _nvfp4_values(d["w"], d["sc"]).t()) * d["g"]
    if kind == "rows_multi":
        x = d["x"].double()
        x = x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * (1.0 + d["norm"].double())
        if case["nvfp4"]:
            return [x] + [(x @ _nvfp4_values(q, sc).t()) * g for q, sc, g in d["mats"]]
        return [x] + [(x @ _e4m3(q).t()) * s for q, s, _ in d["mats"]]
    if kind == "gather":
        rows = d["rows"].long()
        y = (d["x"].double() @ _nvfp4_values(d["w"][rows], d["sc"][rows]).t()) * d["g"]
        y[:, d["count"]:] = -math.inf
        return y
    if kind == "prefill_block":
        # the quantizer's own codes and scales are part of the definition: 32-bit, as the format states them
        x = d["x"].float().view(case["M"], -1, 128)
        s = x.abs().amax(2, keepdim=True) / torch.tensor(448.0, device=DEV)
        q = (x * (1.0 / s)).clamp(-448.0, 448.0).to(torch.float8_e4m3fn).double() * s.double()
        N, K = case["N"], case["K"]
        w = _e4m3(d["w"]).view(N // 128, 128, K // 128, 128) * d["s"].double()[:, None, :, None]
        return q.view(case["M"], K) @ w.view(N, K).t()
    if kind == "prefill_tensor":
        inv = torch.tensor(1.0, device=DEV) / torch.tensor(d["in_scale"], dtype=torch.float32, device=DEV)
        q = (d["x"].float() * inv).clamp(-448.0, 448.0).to(torch.float8_e4m3fn).double()
        return (q @ _e4m3(d["w"]).t()) * (d["in_scale"] * d["s"])
    if kind == "prefill_nvfp4":
        g = torch.tensor(1.0, device=DEV) / torch.tensor(d["in_scale"], dtype=torch.float32, device=DEV)
        v = d["x"].to(torch.bfloat16).float().view(case["M"], -1, 16)
        sc = (g * (v.abs().amax(2) * torch.tensor(1.0 / 6.0, device=DEV))).clamp(max=448.0).to(torch.float8_e4m3fn)
        step = torch.where(sc.float() != 0, 1.0 / (sc.float() * (1.0 / g)), torch.zeros_like(g))
        v = v * step[:, :, None]
        a = v.abs()
        # E2M1, to the nearest, ties to the even code
        mag = torch.zeros_like(a)
        for at, up, value in ((0.25, False, 0.5), (0.75, True, 1.0), (1.25, False, 1.5), (1.75, True, 2.0), (2.5, False, 3.0),
                              (3.5, True, 4.0), (5.0, False, 6.0)):
            mag = torch.where(a >= at if up else a > at, torch.full_like(a, value), mag)
        x = (torch.copysign(mag, v).double() * sc.double()[:, :, None]).view(case["M"], -1)
        return d["resid"].double() + (x @ _nvfp4_values(d["w"], d["sc"]).t()) * (d["in_scale"] * d["g"])
    return None  # codes only
