"""The work that a user of ``nova_amd`` has it do, as cases that can be timed and compared.

Each case is one call, or one captured step, of the package's public entry points: the decode step
of one layer and of a whole stack (one launch per layer, or chained), one-call decode attention, a
ragged paged batch, chunked prefill attention, a whole prompt through the streaming cache, the bulk
quantizers, decoder layers on the kernels and a whole ``GraphDecoder`` step. Head counts, widths and
contexts are those of the repository's configurations, benchmark and tests.

A captured step leaves the write position where it is, so a pass can be repeated: it stores the
same token into the same slot and attends the same tokens.
"""

from __future__ import annotations

import math
import random

import torch

D = 128
GROUP = 64
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
EPS = 1e-6
THETA = 1_000_000.0


# ---------------------------------------------------------------- the cases


def listed() -> list[dict]:
    return [
        # the smallest call: one layer's append + attention early in a conversation, called eagerly
        {"name": "step_one_layer_200", "kind": "step", "fmt": "t64", "mode": "eager", "layers": 1, "ctx": 203,
         "hq": 32, "hkv": 8},
        # a model's layer loop at a middle context, captured: one launch per layer, per-token format;
        # the projections between the layers are left out
        {"name": "step_tok_36_layers_8k", "kind": "step", "fmt": "tok", "mode": "layers", "layers": 36, "ctx": 8191,
         "hq": 32, "hkv": 8},
        # the benchmark's decode step: 36 layers at 32k in one launch, each reading the one before
        {"name": "step_chain_36_layers_32k", "kind": "step", "fmt": "t64", "mode": "chain", "layers": 36,
         "ctx": 32765, "hq": 32, "hkv": 8},
        # decode attention over a packed cache, as the reference's own benchmark calls it
        {"name": "attn_decode_16k", "kind": "attn", "fmt": "t64", "used": 16384, "hq": 32, "hkv": 8},
        # serving: eight long ragged sequences in pages
        {"name": "paged_8_long", "kind": "paged", "fmt": "t64", "seqs": 8, "lo": 4096, "hi": 16384, "lens": 3,
         "layers": 8, "hq": 32, "hkv": 8},
        # serving: many short sequences in pages, per-token format
        {"name": "paged_tok_48_short", "kind": "paged", "fmt": "tok", "seqs": 48, "lo": 64, "hi": 2048, "lens": 5,
         "layers": 16, "hq": 32, "hkv": 8},
        # a prompt's chunk over a long int8 history (the benchmark's prefill)
        {"name": "prefill_512_over_16k", "kind": "prefill", "n": 512, "used": 16384, "hist": 0, "hq": 32, "hkv": 8},
        # a whole prompt through the streaming cache, in the chunks that the benchmark uses; ragged end
        {"name": "prompt_12k_in_2048", "kind": "prompt", "total": 12001, "chunk": 2048, "layers": 2, "hq": 32,
         "hkv": 8},
        # packing a long prompt's K and V
        {"name": "pack_32k", "kind": "quant", "op": "pack", "axis": "token", "group": 64, "dtype": "fp16", "n": 32768,
         "heads": 8},
        # quantize and dequantize with per-channel-group rulers, bf16, ragged
        {"name": "roundtrip_channel_3001", "kind": "quant", "op": "roundtrip", "axis": "channel", "group": 32,
         "dtype": "bf16", "n": 3001, "heads": 8},
        # eight decoder layers of one token on the kernels (attention block, gate/up, down)
        {"name": "layers_8_4k", "kind": "layers", "layers": 8, "ctx": 4133, "hidden": 2560, "inter": 9728, "hq": 32,
         "hkv": 8},
        # the whole decoder at long context: one token, logits of the full vocabulary
        {"name": "decoder_step_32k", "kind": "model", "layers": 36, "ctx": 32700, "vocab": 151936},
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(("step", "step", "step", "attn", "paged", "paged", "prefill", "prompt", "quant", "quant",
                       "layers", "model"))
    hq, hkv = rng.choice(((32, 8), (32, 8), (32, 8), (16, 8), (8, 8), (16, 2), (32, 2)))
    fmt = rng.choice(("t64", "t64", "tok"))
    if kind == "step":
        mode = rng.choice(("eager", "layers", "chain"))
        if mode == "chain":
            hq, hkv = 32, 8
        return {"kind": kind, "fmt": fmt, "mode": mode, "layers": 1 if mode == "eager" else rng.randint(4, 36),
                "ctx": _log_int(rng, 1, 32768), "hq": hq, "hkv": hkv}
    if kind == "attn":
        return {"kind": kind, "fmt": fmt, "used": _log_int(rng, 7, 65536), "hq": hq, "hkv": hkv}
    if kind == "paged":
        seqs = _log_int(rng, 1, 64)
        hi = _log_int(rng, 128, min(16384, 200000 // seqs))
        return {"kind": kind, "fmt": fmt, "seqs": seqs, "lo": max(1, hi // rng.randint(2, 16)), "hi": hi,
                "lens": rng.randint(0, 1 << 20), "layers": rng.randint(2, 12), "hq": hq, "hkv": hkv}
    if kind == "prefill":
        return {"kind": kind, "n": _log_int(rng, 2, 2048), "used": GROUP * _log_int(rng, 1, 512) - GROUP,
                "hist": rng.choice((0, 0, rng.randint(1, 512))), "hq": hq, "hkv": hkv}
    if kind == "prompt":
        total = _log_int(rng, 5, 12001)
        chunk = rng.choice((0, 1024, 2048)) if total > 4096 else rng.choice((0, 256, 512, 1024))
        return {"kind": kind, "total": total, "chunk": chunk, "layers": rng.randint(1, 2), "hq": hq, "hkv": hkv}
    if kind == "quant":
        op = rng.choice(("pack", "roundtrip", "roundtrip", "tok"))
        axis = "token" if op != "roundtrip" else rng.choice(("token", "channel"))
        group = 64 if op != "roundtrip" else rng.choice((32, 64) if axis == "channel" else (64, 64, 32, 0))
        return {"kind": kind, "op": op, "axis": axis, "group": group, "dtype": rng.choice(("fp16", "fp16", "bf16", "fp32")),
                "n": _log_int(rng, 1, 2048 if group == 0 else 65536), "heads": rng.choice((1, 2, 8, 8))}
    if kind == "layers":
        hidden, inter = rng.choice(((2560, 9728), (1024, 3072)))
        return {"kind": kind, "layers": rng.randint(1, 8), "ctx": _log_int(rng, 1, 32768), "hidden": hidden,
                "inter": inter, "hq": rng.choice((16, 32)), "hkv": 8}
    return {"kind": "model", "layers": rng.randint(2, 16), "ctx": _log_int(rng, 64, 32700),
            "vocab": rng.choice((2048, 32000, 151936))}


# ---------------------------------------------------------------- inputs


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(gen: torch.Generator, *shape: int, scale: float = 1.0, dtype: torch.dtype = torch.float16) -> torch.Tensor:
    x = torch.randn(shape, generator=gen, device="cuda", dtype=dtype)
    return x if scale == 1.0 else x.mul_(scale)


def _kv(gen: torch.Generator, hkv: int, n: int, dtype: torch.dtype = torch.float16) -> tuple[torch.Tensor, torch.Tensor]:
    """K ~ N(0, 1) with four channels per head eight times as large (the outlier channels that K
    has), V ~ N(0, 1); ``[1, hkv, n, D]``."""
    gain = torch.ones(hkv, D, device="cuda", dtype=dtype)
    gain.scatter_(1, torch.rand(hkv, D, generator=gen, device="cuda").argsort(1)[:, :4], 8.0)
    k = _normal(gen, 1, hkv, n, D, dtype=dtype).mul_(gain[None, :, None])
    return k, _normal(gen, 1, hkv, n, D, dtype=dtype)


def _query(gen: torch.Generator, *shape: int) -> torch.Tensor:
    return _normal(gen, *shape, scale=0.7)


def _token(gen: torch.Generator, case: dict) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """One layer's new k, v ``[1, hkv, 1, D]`` and q ``[1, hq, 1, D]``."""
    k, v = _kv(gen, case["hkv"], 1)
    return k, v, _query(gen, 1, case["hq"], 1, D)


def _layer_weights(gen: torch.Generator, hidden: int, inter: int, hq: int, hkv: int) -> dict:
    def w(out: int, fan_in: int) -> torch.Tensor:
        return _normal(gen, out, fan_in, scale=fan_in ** -0.5)

    def gamma(n: int) -> torch.Tensor:
        return _normal(gen, n, scale=0.1).add_(1.0)

    return {"qkv": w((hq + 2 * hkv) * D, hidden), "o": w(hidden, hq * D), "gate_up": w(2 * inter, hidden),
            "down": w(hidden, inter), "norm": gamma(hidden), "post": gamma(hidden), "q_norm": gamma(D),
            "k_norm": gamma(D)}


def _inv_freq() -> torch.Tensor:
    return (1.0 / (THETA ** (torch.arange(0, D, 2, dtype=torch.float32) / D))).to("cuda")


def _lengths(case: dict) -> list[int]:
    rng = random.Random(case["lens"])
    return [_log_int(rng, case["lo"], case["hi"]) for _ in range(case["seqs"])]


def _chunks(case: dict) -> list[tuple[int, int]]:
    total, size = case["total"], case["chunk"] or case["total"]
    return [(c, min(total, c + size)) for c in range(0, total, size)]


# ---------------------------------------------------------------- prepare and run


def _capture(fn) -> torch.cuda.CUDAGraph:
    """``fn`` captured after a warmup on a side stream."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        fn()
    return graph


def _fill(cache, gen: torch.Generator, case: dict) -> None:
    """``ctx`` prompt tokens per layer, through the cache's own prefill."""
    cache.begin_prefill(case["ctx"])
    cache.set_prefill_pos(0)
    for layer in range(case["layers"]):
        cache.update(*_kv(gen, case["hkv"], case["ctx"]), layer)
    cache.finish_prefill(case["ctx"])


def _room(ctx: int) -> int:
    return (ctx + 1 + GROUP) // GROUP * GROUP


def _prepare_step(case: dict, gen: torch.Generator) -> dict:
    from nova_amd.chain import ChainedStep
    from nova_amd.kvattn import KVInt8Cache
    from nova_amd.kvtok import KVInt8TokCache

    n, hq, hkv = case["layers"], case["hq"], case["hkv"]
    cls = KVInt8TokCache if case["fmt"] == "tok" else KVInt8Cache
    cache = cls(num_slots=n, num_kv_heads=hkv, head_dim=D, max_len=_room(case["ctx"]), num_q_heads=hq)
    _fill(cache, gen, case)
    s = {"case": case, "cache": cache}
    if case["mode"] == "chain":
        s["x"], s["outs"] = _query(gen, 1, hq, 1, D), torch.zeros(n, 1, hq, 1, D, dtype=torch.float16, device="cuda")
        src = [s["x"], *s["outs"][:-1]]
        gq = hq // hkv
        s["chain"] = ChainedStep(cache, [x[:, 0::gq] for x in src], [x[:, 1::gq] for x in src], src, list(s["outs"]))
        s["graph"] = _capture(s["chain"])
    else:
        s["tokens"] = [_token(gen, case) for _ in range(n)]
        if case["mode"] == "layers":
            s["outs"] = torch.zeros(n, 1, hq, 1, D, dtype=torch.float16, device="cuda")

            def step() -> None:
                for layer, (k, v, q) in enumerate(s["tokens"]):
                    cache.update_attend(k, v, q, layer, out=s["outs"][layer])

            s["graph"] = _capture(step)
    return s


def _run_step(s: dict):
    cache = s["cache"]
    if s["case"]["mode"] == "eager":
        k, v, q = s["tokens"][0]
        out = cache.update_attend(k, v, q, 0)
    else:
        s["graph"].replay()
        out = s["outs"]
    state = (cache.kq[0], cache.vq[0], *((cache.ksc[0], cache.vsc[0]) if s["case"]["fmt"] == "tok" else
                                        (cache.kmn[0], cache.kst[0], cache.tail_k[0], cache.tail_v[0])))
    return {"out": out, "state": state}


def _prepare_attn(case: dict, gen: torch.Generator) -> dict:
    from nova_amd.kvattn import pack_int8_kv
    from nova_amd.kvtok import quantize_tok

    k, v = _kv(gen, case["hkv"], _room(case["used"]))
    packed = (*quantize_tok(k), *quantize_tok(v)) if case["fmt"] == "tok" else pack_int8_kv(k, v)
    return {"case": case, "packed": packed, "q": _query(gen, 1, case["hq"], 1, D),
            "lse": torch.zeros(1, case["hq"], device="cuda")}


def _run_attn(s: dict):
    from nova_amd.kvattn import int8_attn_decode
    from nova_amd.kvtok import int8_tok_attn_decode

    fn = int8_tok_attn_decode if s["case"]["fmt"] == "tok" else int8_attn_decode
    return {"out": fn(s["q"], *s["packed"], used=s["case"]["used"], lse_out=s["lse"]), "lse": s["lse"]}


def _prepare_paged(case: dict, gen: torch.Generator) -> dict:
    from nova_amd.paged import PagedKVInt8Cache, PagedKVInt8TokCache

    lens = _lengths(case)
    pages = [-(-(n + 1) // GROUP) for n in lens]
    cls = PagedKVInt8TokCache if case["fmt"] == "tok" else PagedKVInt8Cache
    cache = cls(case["layers"], case["hkv"], D, case["hq"], max_seqs=len(lens), num_pages=sum(pages),
                max_pages_per_seq=max(pages))
    for b, n in enumerate(lens):
        for layer in range(case["layers"]):
            cache.prefill(b, layer, *_kv(gen, case["hkv"], n))
    cache.plan()
    tokens = []
    for _ in range(case["layers"]):
        k, v = _kv(gen, case["hkv"], len(lens))
        tokens.append((k.transpose(0, 2).contiguous(), v.transpose(0, 2).contiguous(),
                       _query(gen, len(lens), case["hq"], 1, D)))

    def step() -> None:
        for layer, (k, v, q) in enumerate(tokens):
            cache.decode_step(k, v, q, layer)

    return {"case": case, "cache": cache, "tokens": tokens, "graph": _capture(step)}


def _run_paged(s: dict):
    s["graph"].replay()
    cache = s["cache"]
    return {"out": cache.merged, "lse": cache.lse, "pages": cache.pages[-1],
            "rings": cache.rings[-1] if cache.rings is not None else None}


def _prepare_prefill(case: dict, gen: torch.Generator) -> dict:
    from nova_amd.kvattn import pack_int8_kv

    n, hq, hkv = case["n"], case["hq"], case["hkv"]
    s = {"case": case, "packed": pack_int8_kv(*_kv(gen, hkv, case["used"] + GROUP))}
    s["k"], s["v"] = _kv(gen, hkv, case["hist"] + n)
    s["q"] = _query(gen, 1, hq, n, D)
    return s


def _run_prefill(s: dict):
    from nova_amd.kvattn import int8_prefill_attend

    return int8_prefill_attend(s["q"], s["k"], s["v"], *s["packed"], s["case"]["used"])


def _prompt_inputs(case: dict, gen: torch.Generator) -> list[tuple[torch.Tensor, ...]]:
    """Per layer k, v, q of the whole prompt as a model's projections leave them: token-major
    ``[1, total, heads, D]``."""
    got = []
    for _ in range(case["layers"]):
        k, v = _kv(gen, case["hkv"], case["total"])
        q = _query(gen, 1, case["total"], case["hq"], D)
        got.append((k.transpose(1, 2).contiguous(), v.transpose(1, 2).contiguous(), q))
    return got


def _prepare_prompt(case: dict, gen: torch.Generator) -> dict:
    from nova_amd.kvattn import KVInt8Cache

    cache = KVInt8Cache(num_slots=case["layers"], num_kv_heads=case["hkv"], head_dim=D, max_len=_room(case["total"]),
                        num_q_heads=case["hq"])
    return {"case": case, "cache": cache, "inputs": _prompt_inputs(case, gen)}


def _run_prompt(s: dict):
    case, cache = s["case"], s["cache"]
    cache.reset()
    cache.begin_prefill(case["total"], stream_chunk=case["chunk"])
    outs = []
    for c0, c1 in _chunks(case):
        cache.set_prefill_pos(c0)
        for layer, (k, v, q) in enumerate(s["inputs"]):
            cache.update(k[:, c0:c1].transpose(1, 2), v[:, c0:c1].transpose(1, 2), layer)
            outs.append(cache.attend_prefill(q[:, c0:c1].transpose(1, 2), layer))
    cache.finish_prefill(case["total"])
    n = case["total"] // GROUP * GROUP
    state = [x[:, :, :n] for x in (cache.kq[-1], cache.vq[-1])]
    state += [x[:, :, :n // GROUP] for x in (cache.kmn[-1], cache.kst[-1], cache.vmn[-1], cache.vst[-1])]
    return {"out": outs, "state": state}


def _prepare_quant(case: dict, gen: torch.Generator) -> dict:
    return {"case": case, "kv": _kv(gen, case["heads"], case["n"], DTYPES[case["dtype"]])}


def _run_quant(s: dict):
    from nova_amd import kvattn, kvquant, kvtok

    case, (k, v) = s["case"], s["kv"]
    if case["op"] == "pack":
        return kvattn.pack_int8_kv(k, v, case["group"])
    if case["op"] == "tok":
        q, scale = kvtok.quantize_tok(k)
        return q, scale, kvtok.dequantize_tok(q, scale, k.dtype)
    q, mins, steps = kvquant.quantize_int8(k, case["group"], case["axis"])
    return q, mins, steps, kvquant.dequantize_int8(q, mins, steps, case["group"], case["axis"], k.dtype)


def _prepare_layers(case: dict, gen: torch.Generator) -> dict:
    from nova_amd.gemv import rms_gemv, swiglu_gemv
    from nova_amd.kvattn import KVInt8Cache

    cache = KVInt8Cache(num_slots=case["layers"], num_kv_heads=case["hkv"], head_dim=D, max_len=_room(case["ctx"]),
                        num_q_heads=case["hq"])
    _fill(cache, gen, case)
    x = _normal(gen, case["hidden"])
    weights = [_layer_weights(gen, case["hidden"], case["inter"], case["hq"], case["hkv"])
               for _ in range(case["layers"])]
    inv = _inv_freq()
    s = {"case": case, "cache": cache, "x": x, "weights": weights, "inv": inv}

    def step() -> None:
        h, s["h"] = x, []
        for layer, w in enumerate(weights):
            h1 = cache.update_attend_block(h, w["qkv"], w["norm"], EPS, w["q_norm"], w["k_norm"], EPS, inv, w["o"], layer)
            act = swiglu_gemv(h1, w["gate_up"], w["post"], EPS)
            h = rms_gemv(act, w["down"], residual=h1, out=h1)
            s["h"].append(h)

    s["graph"] = _capture(step)
    return s


def _run_layers(s: dict):
    s["graph"].replay()
    return {"h": s["h"], "ring": (s["cache"].tail_k[0], s["cache"].tail_v[0])}


def _prepare_model(case: dict, gen: torch.Generator) -> dict:
    from nova_amd.decode import GraphDecoder
    from nova_amd.skeleton import SkeletonConfig, SkeletonForCausalLM

    cfg = SkeletonConfig(num_hidden_layers=case["layers"], vocab_size=case["vocab"])
    hq, hkv = cfg.num_attention_heads, cfg.num_key_value_heads
    model = SkeletonForCausalLM(cfg, device="cuda", dtype=torch.float16).eval()
    with torch.no_grad():
        model.model.embed_tokens.weight.copy_(_normal(gen, cfg.vocab_size, cfg.hidden_size))
        model.lm_head.weight.copy_(_normal(gen, cfg.vocab_size, cfg.hidden_size, scale=cfg.hidden_size ** -0.5))
        for layer in model.model.layers:
            w = _layer_weights(gen, cfg.hidden_size, cfg.intermediate_size, hq, hkv)
            a, m = layer.attn, layer.mlp
            for p, x in zip((a.q_proj.weight, a.k_proj.weight, a.v_proj.weight), w["qkv"].split((hq * D, hkv * D, hkv * D))):
                p.copy_(x)
            for p, x in zip((m.gate_proj.weight, m.up_proj.weight), w["gate_up"].chunk(2)):
                p.copy_(x)
            for p, x in ((a.o_proj.weight, w["o"]), (m.down_proj.weight, w["down"]), (layer.norm, w["norm"]),
                         (layer.post_norm, w["post"]), (a.q_norm, w["q_norm"]), (a.k_norm, w["k_norm"])):
                p.copy_(x)
    model.use_decode_kernels()
    dec = GraphDecoder(model, max_len=_room(case["ctx"] + 8), quant="int8")
    _fill(dec.cache, gen, {**case, "hkv": hkv})
    ids = torch.randint(0, case["vocab"], (1, 1), generator=gen, device="cuda")
    dec.input_ids.copy_(ids)
    dec.capture()
    return {"case": case, "dec": dec, "ids": ids, "pos": torch.full((1,), case["ctx"], dtype=torch.long, device="cuda")}


def _run_model(s: dict):
    # back to the token after the prompt, then one captured step
    dec = s["dec"]
    dec.cache.pos.copy_(s["pos"])
    dec.input_ids.copy_(s["ids"])
    return {"logits": dec.step(), "ring": (dec.cache.tail_k[0], dec.cache.tail_v[0])}


_KINDS = {"step": (_prepare_step, _run_step), "attn": (_prepare_attn, _run_attn), "paged": (_prepare_paged, _run_paged),
          "prefill": (_prepare_prefill, _run_prefill), "prompt": (_prepare_prompt, _run_prompt),
          "quant": (_prepare_quant, _run_quant), "layers": (_prepare_layers, _run_layers),
          "model": (_prepare_model, _run_model)}


def prepare(case: dict, seed: int) -> dict:
    return _KINDS[case["kind"]][0](case, _gen(seed))


def run(state: dict):
    return _KINDS[state["case"]["kind"]][1](state)


# ---------------------------------------------------------------- work


def _step_bytes(fmt: str, tokens: int, hq: int, hkv: int) -> int:
    """One decode step over ``tokens`` tokens (the new one included): codes and rulers of what is
    attended as int8, the fp16 tokens attended from the ring, the append, q and out."""
    if fmt == "tok":
        return hkv * (260 * tokens + 512) + 512 * hq
    whole = tokens // GROUP * GROUP
    # the append reads the ring's live tokens and writes the new one, its group's codes and rulers
    return hkv * (272 * whole + 512 * (tokens - whole) + 512 + 256 * max(1, tokens % GROUP) + 1024) + 512 * hq


def _layer_bytes(hidden: int, inter: int, hq: int, hkv: int) -> int:
    return 2 * ((hq + 2 * hkv) * D * hidden + hidden * hq * D + 3 * inter * hidden + 4 * hidden)


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "step":
        n, t = case["layers"], case["ctx"] + 1
        return {"bytes": n * _step_bytes(case["fmt"], t, case["hq"], case["hkv"]), "flops": n * 4 * case["hq"] * D * t}
    if kind == "attn":
        t = case["used"]
        per = 260 * t if case["fmt"] == "tok" else 256 * t + 1024 * -(-t // GROUP)
        return {"bytes": case["hkv"] * per + case["hq"] * 516, "flops": 4 * case["hq"] * D * t}
    if kind == "paged":
        lens = [n + 1 for n in _lengths(case)]
        return {"bytes": case["layers"] * sum(_step_bytes(case["fmt"], t, case["hq"], case["hkv"]) for t in lens),
                "flops": case["layers"] * 4 * case["hq"] * D * sum(lens)}
    if kind == "prefill":
        n, hq, hkv = case["n"], case["hq"], case["hkv"]
        pairs = n * (case["used"] + case["hist"]) + n * (n + 1) // 2
        return {"bytes": hkv * (272 * case["used"] + 512 * (case["hist"] + n)) + 512 * hq * n, "flops": 4 * D * hq * pairs}
    if kind == "prompt":
        t, hq, hkv = case["total"], case["hq"], case["hkv"]
        return {"bytes": case["layers"] * t * (hkv * (512 + 272) + 512 * hq),
                "flops": case["layers"] * 4 * D * hq * (t * (t + 1) // 2)}
    if kind == "quant":
        size = torch.empty(0, dtype=DTYPES[case["dtype"]]).element_size()
        n, h = case["n"], case["heads"]
        group = case["group"] or n
        rulers = 2 * n * h if case["op"] == "tok" else 4 * h * (n * (D // group) if case["axis"] == "channel"
                                                               else -(-n // group) * D)
        one = n * h * D * (size + 1) + rulers
        return {"bytes": 2 * one, "flops": 6 * n * h * D}
    hidden, inter, hq, hkv = case.get("hidden", 2560), case.get("inter", 9728), case.get("hq", 32), case.get("hkv", 8)
    t = case["ctx"] + 1
    weights = _layer_bytes(hidden, inter, hq, hkv)
    total = case["layers"] * (weights + _step_bytes("t64", t, hq, hkv)) + 2 * hidden * (2 + 2 * case.get("vocab", 0) // 2)
    flops = case["layers"] * (weights + 4 * hq * D * t) + 2 * hidden * case.get("vocab", 0)
    return {"bytes": total, "flops": flops}


# ---------------------------------------------------------------- tolerance and exact


def tolerance(case: dict):
    kind = case["kind"]
    if kind == "quant":
        return "exact"  # codes, rulers and dequantized values are fixed to the last bit by the formats
    # about four times the distance from 64 bits: fp16 outputs of values dequantized to fp16 (7e-4); an
    # fp16 residual stream after eight layers (1.6e-3); logits after 36 layers (4e-3). Stored codes
    # and rulers follow from the inputs alone and are the same.
    return {"rel": {"layers": 6.4e-3, "model": 1.6e-2}.get(kind, 3e-3), "differ": 0.0}


def _rulers(x: torch.Tensor, group: int) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """Token-axis codes, mins and steps of ``x`` ``[..., n, D]``: the ruler of a group from its
    tokens in 32 bits, the codes from that ruler; mins and steps as stored (fp16)."""
    n = x.shape[-2]
    codes, mins, steps = [], [], []
    for c in range(0, n, group):
        xf = x[..., c:c + group, :].float()
        lo, hi = xf.amin(-2, keepdim=True), xf.amax(-2, keepdim=True)
        st = ((hi - lo) / 255).clamp_min(1e-8)
        codes.append(((xf - lo) / st).round_().clamp_(0, 255))
        mins.append(lo.half())
        steps.append(st.half())
    return torch.cat(codes, -2), torch.cat(mins, -2), torch.cat(steps, -2)


def _int8(x: torch.Tensor, fmt: str) -> torch.Tensor:
    """What the cache holds of ``x`` ``[..., n, D]``, in 64 bits: whole 64-token groups for t64."""
    if x.shape[-2] == 0:
        return x.double()
    if fmt == "tok":
        xf = x.float()
        sc = (xf.abs().amax(-1, keepdim=True) / 127).clamp_min(1e-8)
        return (xf / sc).round_().clamp_(-127, 127).double() * sc.half().double()
    *lead, n, d = x.shape
    xf = x.float().view(*lead, n // GROUP, GROUP, d)
    lo, hi = xf.amin(-2, keepdim=True), xf.amax(-2, keepdim=True)
    st = ((hi - lo) / 255).clamp_min(1e-8)
    q = ((xf - lo) / st).round_().clamp_(0, 255)
    return (q.double() * st.half().double() + lo.half().double()).view(*lead, n, d)


def _cached(x: torch.Tensor, fmt: str) -> torch.Tensor:
    """``x`` ``[..., n, D]`` as a decode step attends it: whole groups int8, the rest fp16 (t64)."""
    if fmt == "tok":
        return _int8(x, fmt)
    whole = x.shape[-2] // GROUP * GROUP
    return torch.cat((_int8(x[..., :whole, :], fmt), x[..., whole:, :].double()), -2)


def _attend(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    """64-bit attention of ``q`` ``[hq, D]`` over ``k`` / ``v`` ``[hkv, n, D]``: out and log-sum-exp."""
    hkv, hq = k.shape[0], q.shape[0]
    s = torch.matmul(q.double().view(hkv, hq // hkv, D), k.transpose(1, 2).contiguous()) * D ** -0.5
    return torch.matmul(s.softmax(-1), v).view(hq, D), s.logsumexp(-1).view(hq)


def _attend_causal(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> torch.Tensor:
    """64-bit causal attention of the last ``n`` of ``m`` tokens: ``q`` ``[hq, n, D]``, ``k`` / ``v``
    ``[hkv, m, D]``."""
    hq, n, _ = q.shape
    hkv, m, _ = k.shape
    out = torch.empty(hq, n, D, dtype=torch.float64, device="cuda")
    hidden = torch.arange(m, device="cuda")[None] > torch.arange(m - n, m, device="cuda")[:, None]
    for h in range(hq):
        kv = h // (hq // hkv)
        s = (q[h].double() @ k[kv].t().contiguous() * D ** -0.5).masked_fill_(hidden, -math.inf)
        out[h] = s.softmax(-1) @ v[kv]
    return out


def _rms64(x: torch.Tensor, gamma: torch.Tensor) -> torch.Tensor:
    return x * (x.square().mean(-1, keepdim=True) + EPS).rsqrt() * gamma.double()


def _rope64(x: torch.Tensor, pos: int) -> torch.Tensor:
    angle = pos * _inv_freq().double()
    cos, sin = angle.cos().repeat(2), angle.sin().repeat(2)
    return x * cos + torch.cat((-x[..., D // 2:], x[..., :D // 2]), -1) * sin


def _layer64(h: torch.Tensor, w: dict, past: tuple[torch.Tensor, torch.Tensor], hq: int, hkv: int) -> torch.Tensor:
    """One decoder layer of one token in 64 bits; ``past``: its fp16 K and V ``[hkv, ctx, D]``."""
    ctx = past[0].shape[1]
    q, k, v = (w["qkv"].double() @ _rms64(h, w["norm"])).split((hq * D, hkv * D, hkv * D))
    q = _rope64(_rms64(q.view(hq, D), w["q_norm"]), ctx)
    k = _rope64(_rms64(k.view(hkv, D), w["k_norm"]), ctx)
    keys, values = (_cached(torch.cat((p.double(), x.view(hkv, 1, D)), 1), "t64") for p, x in zip(past, (k, v)))
    h = h + w["o"].double() @ _attend(q, keys, values)[0].reshape(-1)
    gate, up = (w["gate_up"].double() @ _rms64(h, w["post"])).chunk(2)
    return h + w["down"].double() @ (torch.nn.functional.silu(gate) * up)


def _exact_step(case: dict, gen: torch.Generator):
    n, hq, hkv, fmt = case["layers"], case["hq"], case["hkv"], case["fmt"]
    past = [_kv(gen, hkv, case["ctx"]) for _ in range(n)]
    state = (None,) * (4 if fmt == "tok" else 6)
    outs = []
    if case["mode"] == "chain":
        x, gq = _query(gen, 1, hq, 1, D)[0, :, 0].double(), hq // hkv
    for layer in range(n):
        if case["mode"] == "chain":
            k, v, q = x[0::gq, None], x[1::gq, None], x
        else:
            k, v, q = _token(gen, case)
            k, v, q = k[0].double(), v[0].double(), q[0, :, 0]
        x, _ = _attend(q, *(_cached(torch.cat((p[0].double(), y), 1), fmt) for p, y in zip(past[layer], (k, v))))
        outs.append(x)
        past[layer] = None
    out = torch.stack(outs).view(n, 1, hq, 1, D)
    return {"out": out[0] if case["mode"] == "eager" else out, "state": state}


def _exact_attn(case: dict, gen: torch.Generator):
    k, v = _kv(gen, case["hkv"], _room(case["used"]))
    q = _query(gen, 1, case["hq"], 1, D)
    # every token is int8 here, the last partial group too
    out, lse = _attend(q[0, :, 0], *(_int8(x[0], case["fmt"])[:, :case["used"]] for x in (k, v)))
    return {"out": out.view(1, -1, 1, D), "lse": lse.view(1, -1)}


def _exact_paged(case: dict, gen: torch.Generator):
    lens, n = _lengths(case), case["layers"]
    past = []
    for length in lens:
        for layer in range(n):
            kv = _kv(gen, case["hkv"], length)
            if layer == n - 1:
                past.append(kv)
    for _ in range(n):
        k, v = _kv(gen, case["hkv"], len(lens))
        q = _query(gen, len(lens), case["hq"], 1, D)
    out, lse = [], []
    for b, (pk, pv) in enumerate(past):
        o, e = _attend(q[b, :, 0], *(_cached(torch.cat((p[0], x[0, :, b:b + 1]), 1), case["fmt"])
                                     for p, x in ((pk, k), (pv, v))))
        out.append(o)
        lse.append(e)
    return {"out": torch.stack(out)[:, :, None], "lse": torch.stack(lse), "pages": None, "rings": None}


def _exact_prefill(case: dict, gen: torch.Generator):
    pk, pv = _kv(gen, case["hkv"], case["used"] + GROUP)
    k, v = _kv(gen, case["hkv"], case["hist"] + case["n"])
    q = _query(gen, 1, case["hq"], case["n"], D)
    keys, values = (torch.cat((_int8(p[0, :, :case["used"]], "t64"), x[0].double()), 1) for p, x in ((pk, k), (pv, v)))
    return _attend_causal(q[0], keys, values)[None]


def _exact_prompt(case: dict, gen: torch.Generator):
    outs = []
    inputs = [[x[0].transpose(0, 1) for x in layer] for layer in _prompt_inputs(case, gen)]
    for c0, c1 in _chunks(case):
        for k, v, q in inputs:
            # a streamed chunk reads its history from the int8 cache, a staged one in fp16
            past = [_int8(x[:, :c0].contiguous(), "t64") if case["chunk"] else x[:, :c0].double() for x in (k, v)]
            keys, values = (torch.cat((p, x[:, c0:c1].double()), 1) for p, x in zip(past, (k, v)))
            outs.append(_attend_causal(q[:, c0:c1], keys, values)[None])
    return {"out": outs, "state": [None] * 6}


def _exact_quant(case: dict, gen: torch.Generator):
    k, v = _kv(gen, case["heads"], case["n"], DTYPES[case["dtype"]])
    if case["op"] == "tok":
        sc = (k.float().abs().amax(-1) / 127).clamp_min(1e-8)
        return None, sc.double(), _int8(k, "tok")
    if case["axis"] == "channel":
        shape = (*k.shape[:-1], D // case["group"], case["group"])
        x = k.float().view(shape)
        lo, hi = x.amin(-1, keepdim=True), x.amax(-1, keepdim=True)
        st = ((hi - lo) / 255).clamp_min(1e-8)
        deq = ((x - lo) / st).round_().clamp_(0, 255).double() * st.half().double() + lo.half().double()
        return None, lo[..., 0].double(), st[..., 0].double(), deq.view(k.shape)
    group = case["group"] or case["n"]
    got = []
    for x in (k, v) if case["op"] == "pack" else (k,):
        codes, mins, steps = _rulers(x, group)
        got += [None, mins.double(), steps.double()]
    if case["op"] == "pack":
        return tuple(got)
    spread = [r.repeat_interleave(group, -2)[..., :case["n"], :].double() for r in (mins, steps)]
    return (*got, codes.double() * spread[1] + spread[0])


def _exact_layers(case: dict, gen: torch.Generator):
    past = [_kv(gen, case["hkv"], case["ctx"]) for _ in range(case["layers"])]
    h, got = _normal(gen, case["hidden"]).double(), []
    for layer in range(case["layers"]):
        w = _layer_weights(gen, case["hidden"], case["inter"], case["hq"], case["hkv"])
        h = _layer64(h, w, tuple(x[0] for x in past[layer]), case["hq"], case["hkv"])
        got.append(h)
    return {"h": got, "ring": (None, None)}


def _exact_model(case: dict, gen: torch.Generator):
    hidden, hq, hkv = 2560, 32, 8
    embed = _normal(gen, case["vocab"], hidden)
    head = _normal(gen, case["vocab"], hidden, scale=hidden ** -0.5)
    weights = [_layer_weights(gen, hidden, 9728, hq, hkv) for _ in range(case["layers"])]
    past = [_kv(gen, hkv, case["ctx"]) for _ in range(case["layers"])]
    ids = torch.randint(0, case["vocab"], (1, 1), generator=gen, device="cuda")
    h = embed[ids[0, 0]].double()
    for layer in range(case["layers"]):
        h = _layer64(h, weights[layer], tuple(x[0] for x in past[layer]), hq, hkv)
    h = _rms64(h, torch.ones(hidden, device="cuda"))
    logits = torch.cat([part.double() @ h for part in head.split(16384)])
    return {"logits": logits.view(1, 1, -1), "ring": (None, None)}


def exact(case: dict, seed: int):
    """The outputs in 64 bits, from the same inputs, in plain torch; None in the place of state."""
    return {"step": _exact_step, "attn": _exact_attn, "paged": _exact_paged, "prefill": _exact_prefill,
            "prompt": _exact_prompt, "quant": _exact_quant, "layers": _exact_layers,
            "model": _exact_model}[case["kind"]](case, _gen(seed))
