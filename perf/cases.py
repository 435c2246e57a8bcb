"""What the speed of this framework is measured on: training steps, context encoding and token generation of its model
families at the layer sizes of real models, through its public entry points, with random weights and tokens.

Kinds of cases
  decode  one token for each of `batch` sequences over caches that hold `context` tokens (and fewer: sequences of a batch are
          of different lengths), captured in a hipGraph as the generation loop captures it
  prefill a batch of prompts through the application (padded to its bucket, last token's logits)
  train   one training step: forward, backward, clipping, AdamW over 32-bit master weights
  moe     forward and backward of one dropless mixture-of-experts layer into 32-bit main gradients
`exact` computes the same in plain torch in 64 bits."""

import math

import torch
import torch.nn.functional as F

VOCAB = 128256


def listed():
    return [
        # one user's chat at the context length of the inference notebook: nothing but weights, launches and latency
        dict(name="decode_1b_1", kind="decode", model="llama3.2-1b", layers=16, batch=1, context=2048, int8=False),
        # a few users
        dict(name="decode_1b_4", kind="decode", model="llama3.2-1b", layers=16, batch=4, context=700, int8=False),
        # a server's batch, long and ragged contexts
        dict(name="decode_1b_32", kind="decode", model="llama3.2-1b", layers=16, batch=32, context=2048, int8=False),
        # the width of the 8B model, a batch that is no power of two
        dict(name="decode_8b_13", kind="decode", model="llama3-8b", layers=8, batch=13, context=1500, int8=False),
        # int8 weight-only serving of a few users
        dict(name="decode_int8_6", kind="decode", model="llama3.2-1b", layers=16, batch=6, context=1024, int8=True),
        # the hybrid decoder: recurrent states, windowed two-map attention
        dict(name="decode_golitar_16", kind="decode", model="golitar-2k", layers=16, batch=16, context=2048, int8=False),
        # short prompts of different lengths, padded to a bucket
        dict(name="prefill_1b_3x700", kind="prefill", model="llama3.2-1b", layers=16, batch=3, tokens=700),
        # a long prompt of the hybrid decoder
        dict(name="prefill_golitar_4096", kind="prefill", model="golitar-2k", layers=16, batch=1, tokens=4096),
        # pre-training at the sequence length of the headline configuration, two of the layers (multi-head attention)
        dict(name="train_7b_8192", kind="train", model="llama2-7b", layers=2, batch=1, tokens=8192),
        # fine-tuning of a small model on sequences of an odd length (grouped-query attention, 64 wide heads)
        dict(name="train_1b_3x1000", kind="train", model="llama3.2-1b", layers=4, batch=3, tokens=1000),
        # one expert layer of Mixtral's size
        dict(name="moe_4096", kind="moe", model="mixtral", layers=1, batch=1, tokens=4096),
    ]


def _spread(rng, lo, hi):
    """A whole number of [lo, hi], even over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "train", "moe"])
    if kind == "decode":
        model, layers = rng.choice([("llama3.2-1b", 16), ("llama3.2-1b", 16), ("llama3-8b", 8), ("golitar-2k", 16)])
        int8 = model == "llama3.2-1b" and rng.random() < 0.3
        return dict(kind=kind, model=model, layers=layers, batch=_spread(rng, 1, 32), context=_spread(rng, 64, 2048), int8=int8)
    if kind == "prefill":
        model = rng.choice(["llama3.2-1b", "golitar-2k"])
        tokens = _spread(rng, 128, 4096)
        return dict(kind=kind, model=model, layers=16, batch=rng.randint(1, max(1, min(4, 4096 // tokens))), tokens=tokens)
    if kind == "train":
        model, layers = rng.choice([("llama2-7b", 2), ("llama3.2-1b", 4)])
        tokens = _spread(rng, 256, 4096)
        return dict(kind=kind, model=model, layers=layers, batch=rng.randint(1, max(1, min(4, 4096 // tokens))), tokens=tokens)
    return dict(kind=kind, model="mixtral", layers=1, batch=1, tokens=_spread(rng, 512, 4096))


# ------------------------------------------------------------------------------------------------ sizes
def _raw(case):
    """Sizes of the case's model: a Llama preset's, the benchmark Golitar's config.json, one Mixtral layer's."""
    m = case["model"]
    if m == "mixtral":
        return dict(experts=8, top=2, width=4096, ff=14336)
    if m == "golitar-2k":
        from neuronx_distributed_llama3_2_amd.inference.serve_bench import golitar_config

        g = golitar_config("2k")
        return dict(g, layers=g["layers"][:case["layers"]])
    return _llama_config(case)


def _llama_config(case):
    from neuronx_distributed_llama3_2_amd.models.llama.modeling_llama import llama_config

    more = {}
    if case["kind"] == "train" and case["model"] == "llama2-7b":
        more["max_position_embeddings"] = 8192   # (the long-sequence configuration)
    return llama_config(case["model"], num_hidden_layers=case["layers"], **more)


def _dims(cfg):
    nq, nkv = cfg.num_attention_heads, cfg.num_key_value_heads
    return nq, nkv, cfg.hidden_size // nq, cfg.hidden_size, cfg.intermediate_size


def _lengths(case, seed):
    """Tokens of each sequence: the first has all of them, the others from half of them on."""
    g = torch.Generator().manual_seed(seed * 7 + 3)
    T = case["context"] if case["kind"] == "decode" else case["tokens"]
    n = torch.randint(max(1, T // 2), T + 1, (case["batch"],), generator=g)
    n[0] = T
    return n


def _draws(seed):
    return torch.Generator(device="cuda").manual_seed(seed * 1009 + 17)


def _normal(g, shape, std, dtype=torch.bfloat16, mean=0.0):
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(mean, std, generator=g)


def _uniform(g, shape, lo, hi):
    return torch.empty(shape, dtype=torch.float32, device="cuda").uniform_(lo, hi, generator=g)


def _ids(case, seed, vocab, T):
    return torch.randint(0, vocab, (case["batch"], T), generator=_draws(seed + 500009), device="cuda")


# ------------------------------------------------------------------------------------------------ weights, by parameter name
def _llama_weights(cfg, seed):
    """As in a trained model the residual is of order one and every sublayer adds a small part to it (output projections
    scaled down by the square root of the sublayers); logits are of order one."""
    nq, nkv, D, H, I = _dims(cfg)
    g, std, out, w = _draws(seed), 0.02, 0.02 * 32 ** -0.5, {}
    w["model.embed_tokens.weight"] = _normal(g, (cfg.vocab_size, H), 1.0)
    for i in range(cfg.num_hidden_layers):
        p = f"model.layers.{i}."
        w[p + "self_attn.qkv_proj.weight_qkv"] = _normal(g, ((nq + 2 * nkv) * D, H), std)
        w[p + "self_attn.o_proj.weight"] = _normal(g, (H, nq * D), out)
        w[p + "mlp.gate_up_proj.weight"] = _normal(g, (2 * I, H), std)
        w[p + "mlp.down_proj.weight"] = _normal(g, (H, I), out)
        w[p + "input_layernorm.weight"] = _normal(g, (H,), 0.1, mean=1.0)
        w[p + "post_attention_layernorm.weight"] = _normal(g, (H,), 0.1, mean=1.0)
    last = std if cfg.tie_word_embeddings else 1.0
    w["model.norm.weight"] = _normal(g, (H,), 0.1 * last, mean=last)
    w["lm_head.weight"] = w["model.embed_tokens.weight"] if cfg.tie_word_embeddings else _normal(g, (cfg.vocab_size, H), std)
    return w


def _golitar_weights(raw, seed):
    g, W, S, w = _draws(seed), raw["width"], raw["streams"], {}
    lin = lambda rows, cols, pad=0: torch.cat([_normal(g, (rows, cols), cols ** -0.5),  # noqa: E731
                                               torch.zeros((pad, cols), dtype=torch.bfloat16, device="cuda")])
    pad16 = lambda n: -n % 16  # noqa: E731
    w["model.embed_tokens.weight"] = _normal(g, (raw["vocab"], W), 1.0)
    for i, layer in enumerate(raw["layers"]):
        p, m = f"model.layers.{i}.", layer["mixer"]
        H, G, D, V = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        if layer["type"] == "delta":
            C = 2 * G * D + H * V
            n = C + H * V + 2 * H
            w[p + "mixer.in_proj.weight"] = lin(n, W, pad16(n))
            w[p + "mixer.conv"] = _uniform(g, (m["conv"], C), -0.5, 0.5)
            w[p + "mixer.a_log"] = _uniform(g, (H,), -2.0, 1.0)
            w[p + "mixer.dt_bias"] = _uniform(g, (H,), -3.0, 0.0)
            w[p + "mixer.out_norm"] = _uniform(g, (V,), 0.8, 1.2)
        else:
            n = 2 * (H + G) * D + G * V
            w[p + "mixer.qkv_proj.weight"] = lin(n, W, pad16(n))
            w[p + "mixer.qkv_bias"] = _uniform(g, (n,), -0.1, 0.1)
            w[p + "mixer.q_norm"] = _uniform(g, (D,), 0.8, 1.2)
            w[p + "mixer.k_norm"] = _uniform(g, (D,), 0.8, 1.2)
            for k in ("lq1", "lk1", "lq2", "lk2"):
                w[p + "mixer." + k] = _normal(g, (D,), 0.1, torch.float32)
            w[p + "mixer.o_bias"] = _uniform(g, (W,), -0.1, 0.1)
        w[p + "mixer.o_proj.weight"] = lin(W, H * V)
        w[p + "mlp.up_proj.weight"] = lin(layer["mlp"]["ff"], W)
        w[p + "mlp.down_proj.weight"] = lin(W, layer["mlp"]["ff"])
        for s in range(2):
            w[p + f"norms.{s}"] = _uniform(g, (W,), -0.1, 0.1)
            w[p + f"hyper.{s}.read"] = _uniform(g, (S,), 0.5 / S, 1.5 / S)
            w[p + f"hyper.{s}.mix"] = torch.eye(S, device="cuda") + _uniform(g, (S, S), -0.05, 0.05)
            w[p + f"hyper.{s}.write"] = _uniform(g, (S,), 0.5, 1.5)
    w["model.norm.weight"] = _uniform(g, (W,), -0.1, 0.1)
    w["lm_head.weight"] = lin(raw["vocab"], W)
    return w


def _load(model, weights):
    params = dict(model.named_parameters())
    with torch.no_grad():
        for n, p in params.items():
            p.copy_(weights[n])


# ------------------------------------------------------------------------------------------------ caches of decode cases
def _llama_cache(cfg, case, seed, rows):
    """Keys and values [layers, 2, batch, kv heads, rows, D] of random weights' projections."""
    nq, nkv, D, H, _ = _dims(cfg)
    return _normal(_draws(seed + 900001), (cfg.num_hidden_layers, 2, case["batch"], nkv, rows, D), 0.02 * math.sqrt(H))


def _golitar_cache(raw, case, seed, shapes):
    """What the layers keep: states and the last inputs of the convolutions, normalised keys and values."""
    g, out = _draws(seed + 900001), []
    for c in shapes:
        if "state" in c:
            out.append(dict(state=_normal(g, c["state"], 0.05, torch.float32), ring=_normal(g, c["ring"], 1.0)))
        else:
            out.append(dict(k=_normal(g, c["k"], 1.0), v=_normal(g, c["v"], 1.0)))
    return out


def _golitar_shapes(raw, slots, max_len):
    out = []
    for layer in raw["layers"]:
        m = layer["mixer"]
        H, G, D, V = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        if layer["type"] == "delta":
            out.append(dict(state=(slots, H, V, D), ring=(slots, m["conv"], 2 * G * D + H * V)))
        else:
            cap = min(max_len, (m["mask"]["size"] + 15 + 63) // 64 * 64)
            out.append(dict(k=(slots, 2 * G, cap, D), v=(slots, G, cap, V)))
    return out


def _max_len(case):
    return case["context"] + 256 if case["kind"] == "decode" else max(8192, case["tokens"])


GRAPH_STEPS = 8


# ------------------------------------------------------------------------------------------------ prepare and run
def _app(case, seed):
    from neuronx_distributed_llama3_2_amd.inference.config import InferenceConfig

    raw, n = _raw(case), _max_len(case)
    icfg = InferenceConfig(batch_size=case["batch"], seq_len=n, max_context_length=n, enable_bucketing=True,
                           decode_graph_steps=GRAPH_STEPS)
    if case["model"].startswith("golitar"):
        from neuronx_distributed_llama3_2_amd.inference.golitar import GolitarForCausalLMInference
        from neuronx_distributed_llama3_2_amd.models.golitar import GolitarConfig

        app = GolitarForCausalLMInference(GolitarConfig(raw), icfg)
        _load(app.model, _golitar_weights(raw, seed))
        app.model.post_load()
        app.model.setup_kv_cache(app.max_batch, app.cache_len)
    else:
        from neuronx_distributed_llama3_2_amd.inference.generation import LlamaForCausalLMInference

        app = LlamaForCausalLMInference(raw, icfg)
        _load(app.model, _llama_weights(raw, seed))
        if case.get("int8"):
            from neuronx_distributed_llama3_2_amd.quantization import convert, get_default_per_channel_custom_qconfig_dict

            convert(app.model, get_default_per_channel_custom_qconfig_dict(), inplace=True)
    return app


def _prepare_decode(case, seed):
    from neuronx_distributed_llama3_2_amd.utils.graph_capture import graph_capture

    app = _app(case, seed)
    model, B = app.model, case["batch"]
    n = _lengths(case, seed).cuda()
    tokens = _ids(case, seed, VOCAB, 1)
    args = (tokens, n.view(B, 1), torch.arange(B, dtype=torch.int32, device="cuda"), (n + 1).to(torch.int32))
    state = dict(app=app, args=args, outputs={})
    if case["model"].startswith("golitar"):
        shapes = [{k: tuple(t.shape) for k, t in c.items() if k != "tickets"} for c in model.kv_cache.layers]
        filled = _golitar_cache(_raw(case), case, seed, shapes)
        for c, f in zip(model.kv_cache.layers, filled):
            for k, t in f.items():
                c[k].copy_(t)
        state["outputs"]["states"] = [c["state"] for c in model.kv_cache.layers if "state" in c]
    else:
        model.kv_cache.copy_(_llama_cache(_raw(case), case, seed, app.cache_len))
    saved = model.save_cache() if hasattr(model, "save_cache") else None
    with torch.no_grad():
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            model.forward_tokens(*args)
        torch.cuda.current_stream().wait_stream(side)
        if saved is not None:
            model.load_cache(saved)
        state["graph"] = torch.cuda.CUDAGraph()
        with graph_capture(state["graph"]):
            state["outputs"]["logits"] = model.forward_tokens(*args)
    return state


def _prepare_prefill(case, seed):
    app = _app(case, seed)
    n = _lengths(case, seed).cuda()
    ids = _ids(case, seed, VOCAB, case["tokens"])
    mask = (torch.arange(case["tokens"], device="cuda")[None] < n[:, None]).long()
    outputs = {}
    if case["model"].startswith("golitar"):
        outputs["states"] = [c["state"] for c in app.model.kv_cache.layers if "state" in c]
    else:
        outputs["cache"] = app.model.kv_cache[:, :, :, :, :max(1, case["tokens"] // 2)]   # what every sequence has
    with torch.no_grad():
        app(ids, mask)   # (captures the bucket's graph)
    return dict(app=app, ids=ids, mask=mask, outputs=outputs)


def _parallel():
    import torch.distributed as dist

    from neuronx_distributed_llama3_2_amd.parallel_layers import parallel_state as ps

    if not dist.is_initialized():
        dist.init_process_group("gloo", store=dist.HashStore(), rank=0, world_size=1)
    if not ps.model_parallel_is_initialized():
        ps.initialize_model_parallel(1)


class _Training(dict):
    """A state with an optimizer: its buffers' gradient hooks would keep their memory after the state is gone."""

    def __del__(self):
        for b in self["opt"].buffers:
            for h in b.buf._hooks:
                h.remove()


def _prepare_train(case, seed):
    from neuronx_distributed_llama3_2_amd.models.llama.modeling_llama import LlamaForCausalLM
    from neuronx_distributed_llama3_2_amd.optimizer.flat_optimizer import FlatMixedPrecisionAdamW

    _parallel()
    cfg = _raw(case)
    model = LlamaForCausalLM(cfg, dtype=torch.bfloat16, device=torch.device("cuda", 0))
    _load(model, _llama_weights(cfg, seed))
    opt = FlatMixedPrecisionAdamW(model.parameters(), lr=1e-5, betas=(0.9, 0.95), weight_decay=0.1)
    return _Training(model=model, opt=opt, ids=_ids(case, seed, cfg.vocab_size, case["tokens"]))


def _moe_weights(raw, seed):
    g = _draws(seed)
    E, W, I = raw["experts"], raw["width"], raw["ff"]
    return {"router.linear_router.weight": _normal(g, (E, W), 0.02, torch.float32),
            "expert_mlps.mlp_op.gate_up_proj.weight": _normal(g, (E, W, 2 * I), 0.02),
            "expert_mlps.mlp_op.down_proj.weight": _normal(g, (E, I, W), 0.02)}


def _moe_inputs(case, raw, seed):
    g = _draws(seed + 300007)
    shape = (case["tokens"], case["batch"], raw["width"])
    return _normal(g, shape, 1.0), _normal(g, shape, 1.0)


def _prepare_moe(case, seed):
    from neuronx_distributed_llama3_2_amd.modules.moe import ExpertMLPs, MoE, RouterTopK
    from neuronx_distributed_llama3_2_amd.optimizer.flat_optimizer import FlatMixedPrecisionAdamW

    _parallel()
    raw = _raw(case)
    E, top, W, I = (raw[k] for k in ("experts", "top", "width", "ff"))
    device = torch.device("cuda", 0)
    none = lambda w: w  # noqa: E731
    layer = MoE(RouterTopK(E, top, W, device=device),
                ExpertMLPs(E, top, W, I, "silu", True, None, normalize_top_k_affinities=True, dtype=torch.bfloat16, device=device,
                           init_method=none, output_layer_init_method=none), return_router_logits=False)
    layer.train()
    _load(layer, _moe_weights(raw, seed))
    x, dy = _moe_inputs(case, raw, seed)
    return _Training(layer=layer, opt=FlatMixedPrecisionAdamW(layer.parameters(), lr=1e-5), x=x.requires_grad_(True), dy=dy)


def prepare(case, seed):
    torch.cuda.set_device(0)
    return {"decode": _prepare_decode, "prefill": _prepare_prefill, "train": _prepare_train, "moe": _prepare_moe}[case["kind"]](case, seed)


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["outputs"]
    if "app" in state:
        with torch.no_grad():
            logits = state["app"](state["ids"], state["mask"])
        return dict(state["outputs"], logits=logits)
    if "layer" in state:
        layer, x = state["layer"], state["x"]
        state["opt"].zero_grad()
        x.grad = None
        y = layer(x)
        y.backward(state["dy"])
        return dict(y=y.detach(), dx=x.grad, grads={n: p.main_grad for n, p in layer.named_parameters()})
    model, opt, ids = state["model"], state["opt"], state["ids"]
    opt.zero_grad()
    loss = model(ids, labels=ids).loss
    loss.backward()
    opt.step()
    return dict(loss=loss.detach(), grads={n: p.main_grad for n, p in model.named_parameters()},
                weights={n: p.detach() for n, p in model.named_parameters()})


# ------------------------------------------------------------------------------------------------ work and tolerances
def work(case):
    raw, B = _raw(case), case["batch"]
    if case["kind"] == "moe":
        T, params = case["tokens"], raw["experts"] * 3 * raw["width"] * raw["ff"]
        # weights read once, main gradients written once; activations in and out, forward and backward
        return dict(bytes=params * (2 + 4) + 4 * 2 * T * raw["width"], flops=6 * raw["top"] * T * 3 * raw["width"] * raw["ff"])
    lengths = _lengths(case, 1)
    new = B if case["kind"] == "decode" else int(lengths.sum()) if case["kind"] == "prefill" else B * case["tokens"]
    if case["model"].startswith("golitar"):
        W, linear, small, core, cache = raw["width"], 0, 0, 0, 0
        for layer in raw["layers"]:
            m = layer["mixer"]
            H, G, D, V = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
            linear += W * (H * V + 2 * layer["mlp"]["ff"])
            if layer["type"] == "delta":
                C = 2 * G * D + H * V
                linear += W * (C + H * V + 2 * H)
                core += new * H * 6 * D * V
                cache += B * (2 * 4 * H * D * V + 2 * 2 * m["conv"] * C)
            else:
                window = m["mask"]["size"]
                linear += W * (2 * (H + G) * D + G * V)
                if case["kind"] == "decode":
                    pairs = sum(min(int(n) + 1, window) for n in lengths)
                else:
                    pairs = sum(min(i + 1, window) for n in lengths for i in range(int(n)))
                core += pairs * H * 2 * 2 * (D + V)
                cache += 2 * G * (2 * D + V) * (pairs if case["kind"] == "decode" else sum(min(int(n), window) for n in lengths))
        head, vocab, weights = W * raw["vocab"], raw["vocab"], 2
    else:
        nq, nkv, D, H, I = _dims(raw)
        L, vocab = raw.num_hidden_layers, raw.vocab_size
        linear = L * (H * (nq + 2 * nkv) * D + nq * D * H + 3 * H * I)
        head, weights = H * vocab, 1 if case.get("int8") else 2
        if case["kind"] == "decode":
            core = sum(4 * nq * D * (int(n) + 1) for n in lengths) * L
            cache = sum(4 * nkv * D * (int(n) + 1) for n in lengths) * L
        elif case["kind"] == "prefill":
            core = sum(2 * nq * D * int(n) * (int(n) + 1) for n in lengths) * L
            cache = 4 * nkv * D * new * L
        else:
            T = case["tokens"]
            attn = B * 2 * nq * D * T * (T + 1) * L
            params = linear + head * (1 if raw.tie_word_embeddings else 2)
            # weights and master weights with both moments read and written, gradients written; 8 bytes of ids a token
            return dict(bytes=params * (2 * 2 + 3 * 8 + 4) + 8 * new, flops=6 * new * (linear + head) + 3.5 * attn)
    rows = B   # logits of one token a sequence
    return dict(bytes=weights * (linear + head) + cache + rows * vocab * (4 if case["model"].startswith("golitar") else 2),
                flops=2 * new * linear + 2 * rows * head + core)


def tolerance(case):
    """bf16 weights and activations, 32-bit sums.  Measured between two orders of the same sums (other kernels of this framework):
    0.006 to 0.009 and 0.02 to 0.043; training on the same inputs twice (atomic sums of dQ): 0.001 and 0.027."""
    return {"rel": 0.025, "max": 0.2}


# ------------------------------------------------------------------------------------------------ 64 bits
def _int8(w):
    """Symmetric int8 with a 32-bit scale per row, and back."""
    w = w.float()
    scale = (w.abs().amax(1, keepdim=True) / 127.0).clamp(min=1e-12)
    return torch.round(w / scale).clamp(-127, 127).double() * scale.double()


def _rms(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _inv_freq(cfg, D):
    rope = getattr(cfg, "rope_parameters", None) or {}
    if not rope.get("rope_theta"):
        rope = dict(getattr(cfg, "rope_scaling", None) or {}, rope_theta=cfg.rope_theta)
    f = 1.0 / float(rope["rope_theta"]) ** (torch.arange(0, D, 2, dtype=torch.float64, device="cuda") / D)
    if rope.get("rope_type") != "llama3":
        return f
    return _scaled(f, float(rope["factor"]), float(rope["low_freq_factor"]), float(rope["high_freq_factor"]),
                   float(rope["original_max_position_embeddings"]))


def _scaled(f, factor, low, high, original):
    wave = 2 * math.pi / f
    s = (original / wave - low) / (high - low)
    mid = (1 - s) * f / factor + s * f
    return torch.where(wave > original / low, f / factor, torch.where(wave < original / high, f, mid))


def _rotate(x, angle):
    """x [..., T, D], angle [T, D / 2]: the halves are the pairs."""
    a, b = x.chunk(2, -1)
    c, s = angle.cos(), angle.sin()
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _attend(q, k, v, scale, seen):
    """q [h, t, D], k, v [g, n, D], seen [t, n] or None -> [h, t, D]; one group of heads at a time."""
    rep, out = q.shape[0] // k.shape[0], []
    for g in range(k.shape[0]):
        s = torch.matmul(q[g * rep:(g + 1) * rep], k[g].t()) * scale
        if seen is not None:
            s = s.masked_fill(~seen, float("-inf"))
        out.append(torch.matmul(torch.softmax(s, -1), v[g]))
    return torch.cat(out)


def _llama_block(x, w, p, cfg, attend):
    """x [T, H] of one sequence; attend(q, k, v) [heads, T, D] -> [heads, T, D]."""
    nq, nkv, D, _, _ = _dims(cfg)
    eps, T = cfg.rms_norm_eps, x.shape[0]
    h = _rms(x, w[p + "input_layernorm.weight"], eps)
    qkv = (h @ w[p + "self_attn.qkv_proj.weight_qkv"].t()).view(T, nq + 2 * nkv, D).transpose(0, 1)
    o = attend(qkv[:nq], qkv[nq:nq + nkv], qkv[nq + nkv:])
    x = x + o.transpose(0, 1).reshape(T, nq * D) @ w[p + "self_attn.o_proj.weight"].t()
    h = _rms(x, w[p + "post_attention_layernorm.weight"], eps)
    gate, up = (h @ w[p + "mlp.gate_up_proj.weight"].t()).chunk(2, -1)
    return x + (F.silu(gate) * up) @ w[p + "mlp.down_proj.weight"].t()


class _Double(dict):
    """Weights in 64 bits when they are asked for (kept: as leaves that gather gradients)."""

    def __init__(self, weights, int8=False, grad=False):
        super().__init__(weights)
        self.int8, self.leaves = int8, {}
        if grad:
            self.leaves = {n: t.double().requires_grad_(True) for n, t in weights.items()}

    def __getitem__(self, n):
        if n in self.leaves:
            return self.leaves[n]
        t = dict.__getitem__(self, n)
        return _int8(t) if self.int8 and t.dim() == 2 and "embed" not in n else t.double()


def _exact_decode(case, seed):
    if case["model"].startswith("golitar"):
        return _exact_golitar(case, seed)
    cfg = _raw(case)
    nq, nkv, D, H, _ = _dims(cfg)
    w = _Double(_llama_weights(cfg, seed), int8=case["int8"])
    n = _lengths(case, seed)
    cache = _llama_cache(cfg, case, seed, _max_len(case) + GRAPH_STEPS)
    x = w["model.embed_tokens.weight"][_ids(case, seed, VOCAB, 1)[:, 0]]
    f = _inv_freq(cfg, D)
    for i in range(cfg.num_hidden_layers):
        layer = _Double({k: t for k, t in w.items() if k.startswith(f"model.layers.{i}.")}, int8=case["int8"])
        layer = {k: layer[k] for k in layer}
        rows = []
        for b in range(case["batch"]):
            m = int(n[b])

            def attend(q, k, v):
                angle = f[None] * m
                q, k = _rotate(q, angle), _rotate(k, angle)
                k = torch.cat([cache[i, 0, b, :, :m].double(), k], 1)
                v = torch.cat([cache[i, 1, b, :, :m].double(), v], 1)
                return _attend(q, k, v, D ** -0.5, None)

            rows.append(_llama_block(x[b:b + 1], layer, f"model.layers.{i}.", cfg, attend))
        x = torch.cat(rows)
    logits = _rms(x, w["model.norm.weight"], cfg.rms_norm_eps) @ w["lm_head.weight"].t()
    return dict(logits=logits.unsqueeze(1))


def _causal(T, window=0):
    i = torch.arange(T, device="cuda")
    seen = i[None] <= i[:, None]
    return seen & (i[:, None] - i[None] < window) if window else seen


def _exact_prefill(case, seed):
    if case["model"].startswith("golitar"):
        return _exact_golitar(case, seed)
    cfg = _raw(case)
    nq, nkv, D, H, _ = _dims(cfg)
    w, n, ids = _Double(_llama_weights(cfg, seed)), _lengths(case, seed), _ids(case, seed, VOCAB, case["tokens"])
    f, short = _inv_freq(cfg, D), max(1, case["tokens"] // 2)
    xs = [w["model.embed_tokens.weight"][ids[b, :int(n[b])]] for b in range(case["batch"])]
    kept = torch.empty((cfg.num_hidden_layers, 2, case["batch"], nkv, short, D), dtype=torch.float64, device="cuda")
    for i in range(cfg.num_hidden_layers):
        p = f"model.layers.{i}."
        layer = {k: w[k] for k in w if k.startswith(p)}
        for b, x in enumerate(xs):

            def attend(q, k, v):
                angle = torch.arange(x.shape[0], dtype=torch.float64, device="cuda")[:, None] * f
                q, k = _rotate(q, angle), _rotate(k, angle)
                kept[i, 0, b], kept[i, 1, b] = k[:, :short], v[:, :short]
                return _attend(q, k, v, D ** -0.5, _causal(x.shape[0]))

            xs[b] = _llama_block(x, layer, p, cfg, attend)
    last = torch.stack([x[-1] for x in xs])
    return dict(logits=_rms(last, w["model.norm.weight"], cfg.rms_norm_eps) @ w["lm_head.weight"].t(), cache=kept)


def _exact_train(case, seed):
    from torch.utils.checkpoint import checkpoint

    cfg = _raw(case)
    nq, nkv, D, H, _ = _dims(cfg)
    weights = _llama_weights(cfg, seed)
    tied = cfg.tie_word_embeddings
    if tied:
        del weights["lm_head.weight"]
    w, ids, T = _Double(weights, grad=True), _ids(case, seed, cfg.vocab_size, case["tokens"]), case["tokens"]
    angle = torch.arange(T, dtype=torch.float64, device="cuda")[:, None] * _inv_freq(cfg, D)
    seen = _causal(T)

    def attend(q, k, v):
        q, k = _rotate(q, angle), _rotate(k, angle)
        rep = nq // nkv
        heads = [checkpoint(_attend, q[h:h + 1], k[h // rep:h // rep + 1], v[h // rep:h // rep + 1], D ** -0.5, seen,
                            use_reentrant=False) for h in range(nq)]
        return torch.cat(heads)

    head = w["model.embed_tokens.weight" if tied else "lm_head.weight"]

    def loss_of(h, target):
        return F.cross_entropy(h @ head.t(), target, reduction="sum")

    total, count = 0.0, case["batch"] * (T - 1)
    for b in range(case["batch"]):
        x = w["model.embed_tokens.weight"][ids[b]]
        for i in range(cfg.num_hidden_layers):
            x = checkpoint(_llama_block, x, w, f"model.layers.{i}.", cfg, attend, use_reentrant=False)
        h = _rms(x, w["model.norm.weight"], cfg.rms_norm_eps)[:-1]
        loss = sum(checkpoint(loss_of, h[t:t + 1024], ids[b, 1 + t:1 + t + 1024], use_reentrant=False) for t in range(0, T - 1, 1024))
        (loss / count).backward()
        total += float(loss.detach())
    return dict(loss=torch.tensor(total / count, dtype=torch.float64), grads={n: t.grad for n, t in w.leaves.items()}, weights=None)


def _exact_moe(case, seed):
    raw = _raw(case)
    E, top = raw["experts"], raw["top"]
    w = {n: t.double() for n, t in _moe_weights(raw, seed).items()}
    x, dy = (t.double().reshape(-1, raw["width"]) for t in _moe_inputs(case, raw, seed))
    r, up, down = (w[k] for k in sorted(w, key=lambda k: ("router" not in k, "down" in k)))
    x.requires_grad_(True)
    r.requires_grad_(True)
    logits = x @ r.t()
    index = torch.topk(logits.detach(), top).indices
    chosen = torch.softmax(logits, 1).gather(1, index)
    chosen = chosen / chosen.sum(1, keepdim=True)
    y = torch.zeros_like(x)
    gup, gdown = torch.zeros_like(up), torch.zeros_like(down)
    inputs = x.grad if x.grad is not None else torch.zeros_like(x)
    weight_grad = torch.zeros_like(chosen)
    for e in range(E):   # (one expert at a time: forward, and its part of the backward at once)
        token, choice = (index == e).nonzero(as_tuple=True)
        xe = x.detach()[token].requires_grad_(True)
        ue, de = up[e].clone().requires_grad_(True), down[e].clone().requires_grad_(True)
        gate, u = (xe @ ue).chunk(2, 1)
        out = (F.silu(gate) * u) @ de
        c = chosen.detach()[token, choice]
        y.data.index_add_(0, token, out.detach() * c[:, None])
        out.backward(dy[token] * c[:, None])
        weight_grad[token, choice] = (out.detach() * dy[token]).sum(1)
        inputs.index_add_(0, token, xe.grad)
        gup[e], gdown[e] = ue.grad, de.grad
    chosen.backward(weight_grad)
    shape = (case["tokens"], case["batch"], raw["width"])
    return dict(y=y.detach().view(shape), dx=(x.grad + inputs).view(shape),
                grads={"router.linear_router.weight": r.grad, "expert_mlps.mlp_op.gate_up_proj.weight": gup,
                       "expert_mlps.mlp_op.down_proj.weight": gdown})


def _exact_golitar(case, seed):
    raw = _raw(case)
    eps, S, decode = raw["norm"]["eps"], raw["streams"], case["kind"] == "decode"
    w, n = _Double(_golitar_weights(raw, seed)), _lengths(case, seed)
    B = case["batch"]
    T = 1 if decode else case["tokens"]
    ids = _ids(case, seed, VOCAB, T)
    max_len = _max_len(case) + GRAPH_STEPS
    cache = _golitar_cache(raw, case, seed, _golitar_shapes(raw, B, max_len)) if decode else None
    start = n if decode else torch.zeros(B, dtype=torch.long)
    new = torch.ones(B, dtype=torch.long) if decode else n
    zero_centred = lambda x, g: _rms(x, 1 + g, eps)  # noqa: E731
    streams = w["model.embed_tokens.weight"][ids][:, None].expand(B, S, T, -1).clone()   # [B, S, T, W]
    states = []
    for i, layer in enumerate(raw["layers"]):
        p, m = f"model.layers.{i}.", layer["mixer"]
        lw = {k[len(p):]: w[k] for k in w if k.startswith(p)}
        for s in range(2):
            h = zero_centred(torch.einsum("bstw,s->btw", streams, lw[f"hyper.{s}.read"]), lw[f"norms.{s}"])
            if s == 1:
                y = F.relu(h @ lw["mlp.up_proj.weight"].t()).square() @ lw["mlp.down_proj.weight"].t()
            elif layer["type"] == "delta":
                y, state = _golitar_delta(h, m, lw, eps, cache[i] if decode else None, start, new)
                states.append(state)
            else:
                y = _golitar_attention(h, m, lw, eps, cache[i] if decode else None, start)
            streams = torch.einsum("bstw,sr->brtw", streams, lw[f"hyper.{s}.mix"]) + lw[f"hyper.{s}.write"][:, None, None] * y[:, None]
    last = streams.sum(1)[torch.arange(B, device="cuda"), (new - 1).cuda()]
    logits = zero_centred(last, w["model.norm.weight"]) @ w["lm_head.weight"].t()
    cap = raw.get("logit_softcap")
    logits = cap * torch.tanh(logits / cap) if cap else logits
    return dict(logits=logits.unsqueeze(1) if decode else logits, states=states)


def _golitar_delta(h, m, w, eps, cache, start, new):
    B, T, _ = h.shape
    H, G, D, V, taps = m["heads"], m["kv_heads"], m["dim"], m["vdim"], m["conv"]
    C = 2 * G * D + H * V
    x = h @ w["mixer.in_proj.weight"].t()
    past = torch.zeros((B, taps - 1, C), dtype=torch.float64, device="cuda")
    S = torch.zeros((B, H, V, D), dtype=torch.float64, device="cuda")
    if cache is not None:
        S = cache["state"].double().clone()
        for j in range(taps - 1):
            at = start - (taps - 1) + j
            past[:, j] = torch.where((at >= 0).cuda()[:, None], cache["ring"][torch.arange(B), at % taps].double(), 0.0)
    full = torch.cat([past, x[..., :C]], 1)
    c = F.silu(sum(full[:, j:j + T] * w["mixer.conv"][j] for j in range(taps)))
    unit = lambda t: t / torch.sqrt(t.square().sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    q = (unit(c[..., :G * D].view(B, T, G, D)) * D ** -0.5).repeat_interleave(H // G, 2)
    k = unit(c[..., G * D:2 * G * D].view(B, T, G, D)).repeat_interleave(H // G, 2)
    v = c[..., 2 * G * D:].view(B, T, H, V)
    beta = torch.sigmoid(x[..., C + H * V:C + H * V + H])
    decay = torch.exp(-torch.exp(w["mixer.a_log"]) * F.softplus(x[..., C + H * V + H:C + H * V + 2 * H] + w["mixer.dt_bias"]))
    if T > 1:   # padding tokens leave the state alone
        valid = (torch.arange(T)[None] < new[:, None]).cuda()[..., None]
        beta, decay = torch.where(valid, beta, 0.0), torch.where(valid, decay, 1.0)
    o = torch.empty((B, T, H, V), dtype=torch.float64, device="cuda")
    for t in range(T):
        S.mul_(decay[:, t, :, None, None])
        u = beta[:, t, :, None] * (v[:, t] - torch.matmul(S, k[:, t, :, :, None]).squeeze(-1))
        S.add_(u.unsqueeze(-1) * k[:, t, :, None])
        o[:, t] = torch.matmul(S, q[:, t, :, :, None]).squeeze(-1)
    o = _rms(o, w["mixer.out_norm"], eps) * F.silu(x[..., C:C + H * V]).view(B, T, H, V)
    return o.reshape(B, T, H * V) @ w["mixer.o_proj.weight"].t(), S


def _golitar_attention(h, m, w, eps, cache, start):
    B, T, _ = h.shape
    H, G, D, V, window, diff = m["heads"], m["kv_heads"], m["dim"], m["vdim"], m["mask"]["size"], m["diff"]
    nq, nk = 2 * H * D, 2 * G * D
    x = (h @ w["mixer.qkv_proj.weight"].t())[..., :nq + nk + G * V] + w["mixer.qkv_bias"]
    q = _rms(x[..., :nq].view(B, T, 2 * H, D), w["mixer.q_norm"], eps)
    k = _rms(x[..., nq:nq + nk].view(B, T, 2 * G, D), w["mixer.k_norm"], eps)
    v = x[..., nq + nk:].view(B, T, G, V)
    rot, sc = m["rot"], m["rot"].get("scaling")
    f = float(rot["base"]) ** (-torch.arange(0, rot["dims"], 2, dtype=torch.float64, device="cuda") / rot["dims"])
    if sc:
        f = _scaled(f, sc["factor"], sc["low"], sc["high"], sc["original"])
    angle = (start.cuda()[:, None] + torch.arange(T, device="cuda"))[..., None].double() * f
    lam = torch.exp((w["mixer.lq1"] * w["mixer.lk1"]).sum()) - torch.exp((w["mixer.lq2"] * w["mixer.lk2"]).sum()) + diff

    def turn(t):   # pairs (2i, 2i + 1) of the first `dims` elements
        r, rest = t[..., :rot["dims"]], t[..., rot["dims"]:]
        a, b, c, s = r[..., 0::2], r[..., 1::2], angle.cos()[:, :, None], angle.sin()[:, :, None]
        return torch.cat([torch.stack([a * c - b * s, b * c + a * s], -1).flatten(-2), rest], -1)

    q, k = turn(q), turn(k)
    out = torch.empty((B, T, H, V), dtype=torch.float64, device="cuda")
    for b in range(B):
        kb, vb, seen = k[b].transpose(0, 1), v[b].transpose(0, 1), _causal(T, window)
        if cache is not None:   # one new token at start[b] over a ring of the last keys
            at, cap = int(start[b]), cache["k"].shape[2]
            old = torch.arange(max(0, at - window + 1), at, device="cuda") % cap
            kb = torch.cat([cache["k"][b][:, old].double(), kb], 1)
            vb = torch.cat([cache["v"][b][:, old].double(), vb], 1)
            seen = torch.ones((1, kb.shape[1]), dtype=torch.bool, device="cuda")
        for i in range(H):
            g, a = i // (H // G), []
            for c in range(2):
                z = q[b, :, 2 * i + c] @ kb[2 * g + c].t() * m["scale"]
                z = m["softcap"] * torch.tanh(z / m["softcap"]) if m.get("softcap") else z
                a.append(torch.softmax(z.masked_fill(~seen, float("-inf")), -1) @ vb[g])
            out[b, :, i] = _rms(a[0] - lam * a[1], torch.ones(V, dtype=torch.float64, device="cuda"), eps) * (1 - diff)
    return out.reshape(B, T, H * V) @ w["mixer.o_proj.weight"].t() + w["mixer.o_bias"]


def exact(case, seed):
    torch.cuda.set_device(0)
    if case["kind"] in ("train", "moe"):
        return (_exact_train if case["kind"] == "train" else _exact_moe)(case, seed)
    with torch.no_grad():
        return (_exact_decode if case["kind"] == "decode" else _exact_prefill)(case, seed)
