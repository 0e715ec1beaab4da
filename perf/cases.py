"""What users have this library compute, as timed cases: the RMSNorm, the FFNs, the reference-shaped FFN block and
the Q/K/V projection + attention block, at Llama-3-8B and Falcon-7B widths, from one new token to whole prompts.

`listed()` holds representative calls, `draw(rng)` more of the same ranges: 1 to 4096 rows of RMSNorm, 1 to 2048
tokens through an FFN, 1 to 512 through the FFN block, 1 to 4096 new tokens of attention over up to 32768 cached keys,
fp16 and bf16, row-major weights and the views of torch.nn.Linear weights, 16-bit and fp8 KV caches.
"""
import math
import types

import torch

from trinity_amd import blocks, ext
from trinity_amd.codegen.convert_module import convert_ir_to_triton
from trinity_amd.evaluation import cases as ir_cases
from trinity_amd.evaluation import harness

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}
# model width, FFN width, activation
FFN = {"llama": (4096, 14336, "swiglu"), "falcon": (4544, 18176, "gelu")}
# FFN block of the reference: model width, FFN width, residual + RMSNorm at the end
BLOCK = {"llama": (4096, 14336, False), "falcon": (4544, 4544, True)}
# model width, query heads, KV heads, head dimension; "llama_mha": the reference's own shape, a KV head per query head
HEADS = {"llama": (4096, 32, 8, 128), "llama_mha": (4096, 32, 32, 128), "falcon": (4544, 71, 1, 64)}
# the generated modules of the reference: model width, heads, head dimension
MODULE = {"llama": (4096, 32, 128), "falcon": (4544, 71, 64)}
VARIANTS = ("vanilla", "prenorm", "qknorm", "keyformer", "roco")


def listed():
    return [
        # the norm of a decode step over a small batch: nothing but latency
        {"name": "rmsnorm_16", "kind": "rmsnorm", "rows": 16, "n": 4096, "dtype": "f16"},
        # the norm of a long prompt: bandwidth
        {"name": "rmsnorm_4096", "kind": "rmsnorm", "rows": 4096, "n": 4096, "dtype": "f16"},
        # the FFN half of a layer at the reference's evaluation shape (16 tokens), through its plan
        {"name": "block_llama_16", "kind": "block", "model": "llama", "tokens": 16},
        # one decode step of one sequence, weights as torch.nn.Linear holds them
        {"name": "ffn_llama_1_linear", "kind": "ffn", "model": "llama", "tokens": 1, "dtype": "bf16", "layout": "linear"},
        # a chunk of a prompt or a large decode batch, ragged
        {"name": "ffn_falcon_333", "kind": "ffn", "model": "falcon", "tokens": 333, "dtype": "f16", "layout": "row"},
        # the benchmark's FFN: a whole prompt
        {"name": "ffn_llama_2048", "kind": "ffn", "model": "llama", "tokens": 2048, "dtype": "f16", "layout": "row"},
        # decode of one token over a cached conversation
        {"name": "decode_llama_1_4095", "kind": "attention", "heads": "llama", "variant": "vanilla", "new": 1,
         "cached": 4095, "dtype": "bf16", "fp8": False},
        # a generated module at the reference's evaluation shape, with per-key statistics
        {"name": "module_roco_llama_16_1024", "kind": "module", "model": "llama", "variant": "roco", "new": 16,
         "cached": 1024},
        # a few tokens (speculative decoding) over a long context held in fp8
        {"name": "decode_llama_16_32752_fp8", "kind": "attention", "heads": "llama", "variant": "vanilla", "new": 16,
         "cached": 32752, "dtype": "f16", "fp8": True},
        # a prompt of a thousand tokens, ragged, multi-query attention
        {"name": "prefill_prenorm_falcon_1000", "kind": "attention", "heads": "falcon", "variant": "prenorm",
         "new": 1000, "cached": 0, "dtype": "bf16", "fp8": False},
        # a long prompt
        {"name": "prefill_llama_4096", "kind": "attention", "heads": "llama", "variant": "vanilla", "new": 4096,
         "cached": 0, "dtype": "f16", "fp8": False},
        # a prompt whose per-key scores are kept for cache eviction
        {"name": "prefill_keyformer_llama_2048", "kind": "attention", "heads": "llama", "variant": "keyformer",
         "new": 2048, "cached": 0, "dtype": "f16", "fp8": False},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("rmsnorm", "ffn", "ffn", "block", "module", "decode", "decode", "chunk", "prefill"))
    dtype = rng.choice(("f16", "bf16"))
    if kind == "rmsnorm":
        return {"kind": kind, "rows": _log_int(rng, 1, 4096), "n": rng.choice((4096, 4544)), "dtype": dtype}
    if kind == "ffn":
        return {"kind": kind, "model": rng.choice(("llama", "falcon")), "tokens": _log_int(rng, 1, 2048),
                "dtype": dtype, "layout": rng.choice(("row", "linear"))}
    if kind == "block":
        return {"kind": kind, "model": rng.choice(("llama", "falcon")), "tokens": _log_int(rng, 1, 512)}
    if kind == "module":
        return {"kind": kind, "model": rng.choice(("llama", "falcon")), "variant": rng.choice(VARIANTS),
                "new": _log_int(rng, 1, 32), "cached": _log_int(rng, 64, 2048)}
    heads, variant = rng.choice(("llama", "falcon")), rng.choice(VARIANTS)
    if kind == "decode":
        heads = rng.choice(tuple(HEADS))
        new, cached = _log_int(rng, 1, 32), _log_int(rng, 128, 32736)
    elif kind == "chunk":
        new, cached = _log_int(rng, 33, 512), _log_int(rng, 128, 16384)
    else:
        new, cached = _log_int(rng, 128, 4096), 0
        if heads == "falcon":
            variant = rng.choice(("vanilla", "prenorm", "qknorm"))
    return {"kind": "attention", "heads": heads, "variant": variant, "new": new, "cached": cached, "dtype": dtype,
            "fp8": cached > 0 and rng.random() < 0.3}


class _Random:
    """Normal values on the GPU from a seed of their own."""

    def __init__(self, seed):
        self.dev = torch.device("cuda:0")
        self.gen = torch.Generator(device=self.dev)
        self.gen.manual_seed(seed)

    def __call__(self, *shape, std=1.0, mean=0.0, dtype=torch.float16):
        t = torch.empty(*shape, dtype=dtype, device=self.dev)
        return t.normal_(mean, std, generator=self.gen)


def _prepare_rmsnorm(case, rn):
    dt = DTYPES[case["dtype"]]
    x = rn(case["rows"], case["n"], dtype=dt)
    w = rn(case["n"], std=0.1, mean=1.0, dtype=dt)
    return {"plan": blocks.RmsNormPlan(eps=1e-5), "x": x, "w": w, "y": torch.empty_like(x)}


def _prepare_ffn(case, rn):
    n, f, act = FFN[case["model"]]
    dt, t = DTYPES[case["dtype"]], case["tokens"]

    def weight(k, cols):
        if case["layout"] == "linear":
            return rn(cols, k, std=0.02, dtype=dt).t()
        return rn(k, cols, std=0.02, dtype=dt)

    s = {"act": act, "x": rn(t, n, dtype=dt), "w1": weight(n, f), "w2": weight(f, n)}
    s["w_up"] = weight(n, f) if act == "swiglu" else None
    s["out"] = torch.empty(t, n, dtype=dt, device=rn.dev)
    if dt == torch.float16:  # the plan keeps the hidden activation (fp16) and the workspace
        s["plan"] = blocks.FfnPlan(act)
    else:
        s["hidden"] = torch.empty(t, f, dtype=dt, device=rn.dev)
        ws = ext.ffn_workspace_bytes(t, n, f)
        s["ws"] = torch.empty(ws, dtype=torch.uint8, device=rn.dev) if ws else None
    return s


def _prepare_block(case, rn):
    n, f, tail = BLOCK[case["model"]]
    m = case["tokens"]
    s = {"plan": blocks.FfnBlockPlan(falcon_tail=tail), "O2": rn(m, n), "X": rn(m, n)}
    s["WO"], s["WFF1a"], s["WFF1b"], s["WFF2"] = (rn(n, n, std=0.02), rn(n, f, std=0.02), rn(n, f, std=0.02),
                                                 rn(f, n, std=0.02))
    s["attn_O2"], s["FF2"] = torch.empty_like(s["X"]), torch.empty_like(s["X"])
    s["O_FF_norm"] = torch.empty_like(s["X"]) if tail else None
    return s


def _prepare_module(case, seed):
    n, h, d = MODULE[case["model"]]
    m, p, variant = case["new"], case["cached"], case["variant"]
    base = variant if variant in ("keyformer", "roco") else "vanilla"
    ir = ir_cases.attention_ir(base, m, n, d, p, prenorm=variant == "prenorm", qknorm=variant == "qknorm")
    module = types.ModuleType("generated")
    exec(convert_ir_to_triton(ir, None, {"M": m, "D": d, "N": n, "P": p, "H": h}), module.__dict__)
    tensors = harness.attention_tensors(m, n, d, p, h, torch.device("cuda:0"), seed=seed)
    if base != "vanilla":  # scores as fp32, as the kernels accumulate them
        for name in ("C_out", "C_out1", "C_out2"):
            tensors[name] = tensors[name].float()
    args = harness.positional_args(module, tensors, {"block_k": 32, "block_p": 16, "block_n": 64})
    outputs = ["O2", "K_cache", "V_cache"] + {"keyformer": ["C_out"], "roco": ["C_out1", "C_out2"]}.get(base, [])
    return {"forward": module.forward, "args": args, "outputs": [tensors[name] for name in outputs]}


def _prepare_attention(case, rn, seed):
    n, hq, hkv, d = HEADS[case["heads"]]
    s, p, variant, dt = case["new"], case["cached"], case["variant"], DTYPES[case["dtype"]]
    base = variant if variant in ("keyformer", "roco") else "vanilla"
    total = p + s
    st = {"variant": base, "x": rn(s, n, dtype=dt)}
    st["wq"], st["wk"], st["wv"] = (rn(n, hq * d, std=0.02, dtype=dt), rn(n, hkv * d, std=0.02, dtype=dt),
                                    rn(n, hkv * d, std=0.02, dtype=dt))
    st["norm_w"] = rn(n, std=0.1, mean=1.0, dtype=dt) if variant == "prenorm" else None
    # keys and values as this projection yields them: N(0, 0.02^2 * n)
    std = 0.02 * math.sqrt(n) if variant != "qknorm" else 1.0
    st["k"], st["v"] = rn(hkv, total, d, std=std, dtype=dt), rn(hkv, total, d, std=0.02 * math.sqrt(n), dtype=dt)
    st["o"] = torch.empty(s, hq * d, dtype=dt, device=rn.dev)
    names = {"keyformer": 1, "roco": 2}.get(base, 0)
    st["scores"] = [torch.empty(hq, total, dtype=torch.float32, device=rn.dev) for _ in range(names)]
    args = dict(scale=1.0 / math.sqrt(d), causal=True, tau=1.0, noise_seed=seed, prenorm=variant == "prenorm",
                qknorm=variant == "qknorm")
    if case["fp8"]:
        st["k"], st["v"] = st["k"].to(torch.float8_e4m3fn), st["v"].to(torch.float8_e4m3fn)
        st["p"] = ext.attn_params(hq, hkv, d, s, kv_prefix=p, rms_eps=1e-5, kv_fp8=True, k_scale=1.0, v_scale=1.0, **args)
        st["scratch"] = torch.empty(ext.qkv_scratch_bytes(st["p"], n), dtype=torch.uint8, device=rn.dev)
    else:
        st["plan"] = blocks.AttentionPlan(variant=base, N=n, D=d, H=hq, P=p, n_kv_heads=hkv, eps=1e-5, **args)
    return st


def prepare(case, seed):
    rn, kind = _Random(seed), case["kind"]
    if kind == "rmsnorm":
        state = _prepare_rmsnorm(case, rn)
    elif kind == "ffn":
        state = _prepare_ffn(case, rn)
    elif kind == "block":
        state = _prepare_block(case, rn)
    elif kind == "module":
        state = _prepare_module(case, seed)
    else:
        state = _prepare_attention(case, rn, seed)
    state["kind"] = kind
    return state


def run(s):
    kind = s["kind"]
    if kind == "rmsnorm":
        s["plan"].run(s["x"], s["y"], weight=s["w"])
        return s["y"]
    if kind == "ffn":
        if "plan" in s:
            s["plan"].run(s["x"], s["w1"], s["w2"], s["out"], W_up=s["w_up"])
        elif s["act"] == "swiglu":
            ext.ffn_swiglu(s["x"], s["w1"], s["w_up"], s["w2"], s["hidden"], s["out"], workspace=s["ws"])
        else:
            ext.ffn_gelu(s["x"], s["w1"], s["w2"], s["hidden"], s["out"], workspace=s["ws"])
        return s["out"]
    if kind == "block":
        s["plan"].run(s["O2"], s["WO"], s["X"], s["WFF1a"], s["WFF1b"], s["WFF2"], attn_O2=s["attn_O2"], FF2=s["FF2"],
                      O_FF_norm=s["O_FF_norm"])
        return [s["attn_O2"], s["FF2"], s["O_FF_norm"]]
    if kind == "module":
        s["forward"](*s["args"])
        return s["outputs"]
    sc = s["scores"]
    if "plan" in s:
        names = {"keyformer": ("C_out",), "roco": ("C_out1", "C_out2")}.get(s["variant"], ())
        s["plan"].run(s["x"], s["wq"], s["wk"], s["wv"], s["o"], K_cache=s["k"], V_cache=s["v"], norm_w=s["norm_w"],
                      **dict(zip(names, sc)))
    elif s["variant"] == "keyformer":
        ext.keyformer(s["x"], s["norm_w"], s["wq"], s["wk"], s["wv"], s["k"], s["v"], s["scratch"], None, s["o"], sc[0],
                      s["p"])
    elif s["variant"] == "roco":
        ext.roco(s["x"], s["norm_w"], s["wq"], s["wk"], s["wv"], s["k"], s["v"], s["scratch"], s["o"], sc[0], sc[1],
                 s["p"])
    else:
        ext.qkv_attention(s["x"], s["norm_w"], s["wq"], s["wk"], s["wv"], s["k"], s["v"], s["scratch"], None, s["o"],
                          s["p"])
    return [s["o"], s["k"], s["v"]] + sc


def work(case):
    kind = case["kind"]
    if kind == "rmsnorm":
        return {"bytes": 4 * case["rows"] * case["n"] + 2 * case["n"], "flops": 4 * case["rows"] * case["n"]}
    if kind == "ffn":
        n, f, act = FFN[case["model"]]
        t, mats = case["tokens"], 3 if act == "swiglu" else 2
        return {"bytes": 2 * (mats * n * f + 2 * t * n), "flops": 2 * t * n * f * mats}
    if kind == "block":
        n, f, tail = BLOCK[case["model"]]
        m = case["tokens"]
        return {"bytes": 2 * (n * n + 3 * n * f + (5 if tail else 4) * m * n), "flops": 2 * m * n * (n + 3 * f)}
    s, p, variant = case["new"], case["cached"], case["variant"]
    if kind == "module":
        n, hq, d = MODULE[case["model"]]
        hkv, pairs, cache = hq, s * (p + s), 2  # no mask
    else:
        n, hq, hkv, d = HEADS[case["heads"]]
        pairs, cache = s * p + s * (s + 1) // 2, 1 if case["fp8"] else 2
    total, cols = p + s, (hq + 2 * hkv) * d
    nbytes = 2 * (n * cols + s * n + s * hq * d) + cache * 2 * hkv * d * (p + s)  # old rows read, new rows written
    nbytes += 4 * hq * total * {"keyformer": 1, "roco": 2}.get(variant, 0)
    if kind == "module" and variant == "keyformer":
        nbytes += 2 * hq * s * total  # the noise tensor
    return {"bytes": nbytes, "flops": 2 * s * n * cols + 4 * d * hq * pairs}


def tolerance(case):
    # Four times what the outputs are off a computation in 64 bits with the same roundings of intermediates (normalised
    # rows, q / k / v, hidden activations): 4.7e-4 in fp16 and 2.4e-3 in bf16, for attention, whose probabilities are
    # 16 bits wide; largest single values 4e-3 and 1.5e-2.  A value on the edge between two fp8 codes may come out as
    # either: an eighth of the value.
    if case.get("dtype", "f16") == "f16":
        rel, most = 2e-3, 0.016
    else:
        rel, most = 1e-2, 0.06
    return {"rel": rel, "max": 0.15 if case.get("fp8") else most}
