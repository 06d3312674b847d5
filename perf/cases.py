"""The work this library is used for, as measurable cases.

Two kinds of program call it.  A GPT-2 style training loop runs the QKV
projection and causal multi-head attention, forward and backward, with FP32 or
bf16 activations.  A Qwen style hybrid decoder runs grouped-query attention over
a key/value cache and the gated delta-net: whole prompts, one token for one or
many sequences (with the block-scaled FP8 or bf16 projections around the mixing
step), and whole sequences forward and backward when it is trained.

Every case goes through pluto_amd.capi with buffers and workspaces kept between
calls wherever an entry point lets the caller keep them.
"""
import math

import torch

from pluto_amd import capi

BF16 = torch.bfloat16

# The decoder's shapes: 24 query and 4 key/value heads over a 5120-wide residual
# stream, delta-net layers of 16 key and 48 value heads of 128 x 128.
WIDTH, QUERY_HEADS, KV_HEADS = 5120, 24, 4
KEY_HEADS, VALUE_HEADS, DELTA_DIM, CONV_TAPS = 16, 48, 128, 4
ROTARY = {64: 16, 128: 32, 256: 64}
STORAGE = {"fp8": capi.MATRIX_FP8_E4M3, "bf16": capi.MATRIX_BF16}


def listed():
    return [
        # A training step of one attention layer at the CPU reference's size, in
        # the reference's own storage type.  The smallest training work.
        dict(name="mha train f32 256", kind="mha_train", dtype="f32", batch=4, length=256, heads=12, head_dim=64),
        # The benchmark's headline: a GPT-2-small attention layer at its full context, bf16.
        dict(name="mha train bf16 1024", kind="mha_train", dtype="bf16", batch=16, length=1024, heads=12, head_dim=64),
        # The QKV projection in front of it: forward, input, weight and bias gradients.
        dict(name="dense train bf16 16384", kind="dense_train", dtype="bf16", rows=16384, input_dim=768, output_dim=2304),
        # A long prompt at head width 128, written into an empty cache.
        dict(name="prefill d128 8192", kind="prefill", head_dim=128, length=8192, start=0),
        # A chat's next turn at the decoder's own head width: a ragged number of
        # new tokens behind those already cached.
        dict(name="prefill d256 1531+2309", kind="prefill", head_dim=256, length=1531, start=2309),
        # Training a grouped-query layer on a long sequence: forward with the
        # state for the backward kept, then backward.  The largest case.
        dict(name="gqa train d128 8192", kind="gqa_train", head_dim=128, length=8192),
        # The same layer at the decoder's own head width, on an ordinary sequence.
        dict(name="gqa train d256 1024", kind="gqa_train", head_dim=256, length=1024),
        # One decode step of an attention branch for a full batch of long contexts.
        dict(name="attention step 32 x 32768", kind="attention_step", head_dim=256, batch=32, storage="fp8", shortest=1024, longest=32768),
        # One decode step for one user with a short context: the smallest call.
        dict(name="attention step 1 x 777", kind="attention_step", head_dim=256, batch=1, storage="fp8", shortest=777, longest=777),
        # One decode step of a delta-net branch for a full batch.
        dict(name="delta step 32", kind="delta_step", batch=32, storage="fp8"),
        # A long ragged prompt through a delta-net layer.
        dict(name="delta prefill 8191", kind="delta_prefill", batch=1, length=8191, key_heads=16, value_heads=48),
        # Backward of a delta-net layer with all its parameters training.
        dict(name="delta backward 2048", kind="delta_backward", batch=1, length=2048, key_heads=16, value_heads=48),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice([c["kind"] for c in listed()])
    if kind == "mha_train":
        heads, head_dim = rng.choice([(12, 64), (12, 64), (6, 128), (4, 64)])
        dtype = rng.choice(["f32", "bf16"])
        # FP32 at the lengths of the GPT-2 recipes, bf16 also at four times that
        length = _log(rng, 48, 1024 if dtype == "f32" else 4096)
        return dict(kind=kind, dtype=dtype, batch=_log(rng, 1, max(1, 16384 // length)) if length > 512 else _log(rng, 1, 24),
                    length=length, heads=heads, head_dim=head_dim)
    if kind == "dense_train":
        n_in, n_out = rng.choice([(768, 2304), (768, 768), (768, 3072), (3072, 768), (256, 768)])
        return dict(kind=kind, dtype=rng.choice(["bf16", "f32"]), rows=_log(rng, 64, 16384), input_dim=n_in, output_dim=n_out)
    if kind == "prefill":
        length = _log(rng, 16, 8192)
        return dict(kind=kind, head_dim=rng.choice([128, 256]), length=length,
                    start=rng.choice([0, rng.randrange(0, 8193 - length)]))
    if kind == "gqa_train":
        head_dim = rng.choice([128, 256])
        return dict(kind=kind, head_dim=head_dim, length=_log(rng, 64, 4096 if head_dim == 128 else 1024))
    if kind == "attention_step":
        longest = _log(rng, 64, 32768)
        return dict(kind=kind, head_dim=rng.choice([128, 256]), batch=_log(rng, 1, 32), storage=rng.choice(["fp8", "fp8", "bf16"]),
                    shortest=max(1, longest // 32), longest=longest)
    if kind == "delta_step":
        return dict(kind=kind, batch=_log(rng, 1, 64), storage=rng.choice(["fp8", "fp8", "bf16"]))
    key_heads, value_heads = rng.choice([(16, 48), (16, 16)])
    if kind == "delta_prefill":
        length = _log(rng, 32, 16384)
        return dict(kind=kind, batch=rng.randint(1, max(1, min(4, 16384 // length))), length=length,
                    key_heads=key_heads, value_heads=value_heads)
    return dict(kind=kind, batch=1, length=_log(rng, 64, 4096), key_heads=key_heads, value_heads=value_heads)


# ---- inputs -----------------------------------------------------------------

class _Source:
    """Values on the GPU, made from one seed."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, scale=1.0, dtype=torch.float32):
        x = torch.randn(shape, generator=self.gen, device="cuda", dtype=dtype)
        return x if scale == 1.0 else x.mul_(scale)

    def uniform(self, *shape, low=0.0, high=1.0):
        return low + (high - low) * torch.rand(shape, generator=self.gen, device="cuda")

    def matrix(self, storage, input_dim, output_dim):
        """A frozen checkpoint matrix: (weights [out, in], FP8 block scales or None)."""
        if storage == "bf16":
            return self.normal(output_dim, input_dim, scale=1 / math.sqrt(input_dim), dtype=BF16), None
        w = torch.randint(0, 0x7f, (output_dim, input_dim), generator=self.gen, device="cuda", dtype=torch.uint8)
        w |= torch.randint(0, 2, (output_dim, input_dim), generator=self.gen, device="cuda", dtype=torch.uint8) << 7
        blocks = ((output_dim + 127) // 128, (input_dim + 127) // 128)
        return w, self.uniform(*blocks, low=0.5, high=1.5) * (0.01 / math.sqrt(input_dim))


def _empty(*shape, dtype=BF16):
    return torch.empty(shape, dtype=dtype, device="cuda")


def _norm_weights(source, head_dim):
    return source.normal(head_dim, scale=0.3), source.normal(head_dim, scale=0.3)


def _contexts(case):
    """Context lengths of the batch, spread over [shortest, longest]."""
    span = case["longest"] - case["shortest"] + 1
    return [case["shortest"] + int(span * ((0.618034 * (i + 1)) % 1.0)) for i in range(case["batch"])]


def _delta_weights(source, p):
    channels = 2 * p.key_heads * p.key_head_dim + p.value_heads * p.value_head_dim
    step = torch.exp(source.uniform(p.value_heads, low=math.log(1e-3), high=math.log(0.1)))
    return dict(conv_weight=source.normal(channels, p.conv_kernel_dim, scale=0.5),
                a_log=torch.log(source.uniform(p.value_heads, low=1.0, high=16.0)),
                dt_bias=torch.log(torch.expm1(step)),
                norm=1.0 + source.normal(p.value_head_dim, scale=0.1))


class _Projection:
    """Frozen matrices applied to the same rows, and what a serving loop keeps for them."""

    def __init__(self, source, storage, tokens, input_dim, output_dims):
        self.storage = STORAGE[storage]
        made = [source.matrix(storage, input_dim, n) for n in output_dims]
        self.weights, self.scales = [m[0] for m in made], [m[1] for m in made]
        size = capi.lib().pluto_hip_dense_imported_batch_workspace_bytes(tokens, input_dim)
        self.workspace = _empty(max(size, 1), dtype=torch.uint8)
        self.outs = [_empty(tokens, n) for n in output_dims]

    def __call__(self, x):
        if len(self.weights) == 1:
            return capi.dense_imported_forward_batch(self.storage, self.weights[0], self.scales[0], x, self.workspace, self.outs[0])
        return capi.dense_imported_forward_many(self.storage, self.weights, self.scales, x, self.workspace, self.outs)


# ---- the kinds --------------------------------------------------------------

def _prepare_mha_train(case, source):
    rows, width = case["batch"] * case["length"], case["heads"] * case["head_dim"]
    dtype = BF16 if case["dtype"] == "bf16" else torch.float32
    qkv = source.normal(rows, 3 * width).to(dtype)
    stats = (case["batch"] * case["heads"], case["length"])
    return dict(qkv=qkv, d_out=source.normal(rows, width), length=case["length"], heads=case["heads"],
                forward=(_empty(rows, width, dtype=dtype), _empty(*stats, dtype=torch.float32), _empty(*stats, dtype=torch.float32)),
                workspace=capi.mha_backward_workspace(qkv, case["length"], case["heads"]),
                d_qkv=_empty(rows, 3 * width, dtype=torch.float32))


def _run_mha_train(s):
    out, maxima, normalizers = capi.mha_forward(s["qkv"], s["length"], s["heads"], into=s["forward"])
    grads = capi.mha_backward(s["qkv"], out, s["d_out"], maxima, normalizers, s["length"], s["heads"], s["workspace"], s["d_qkv"])
    return out, maxima, normalizers, grads


def _prepare_dense_train(case, source):
    rows, n_in, n_out = case["rows"], case["input_dim"], case["output_dim"]
    x = source.normal(rows, n_in).to(BF16 if case["dtype"] == "bf16" else torch.float32)
    return dict(x=x, matrix=source.normal(n_in, n_out, scale=1 / math.sqrt(n_in)), bias=source.normal(n_out, scale=0.1),
                d_out=source.normal(rows, n_out), workspace=capi.dense_workspace(x, n_out), out=_empty(rows, n_out, dtype=x.dtype))


def _run_dense_train(s):
    out = capi.dense_forward(s["x"], s["matrix"], s["bias"], workspace=s["workspace"], out=s["out"])
    return (out,) + tuple(capi.dense_backward(s["x"], s["matrix"], s["d_out"], workspace=s["workspace"]))


def _attention_inputs(case, source, capacity):
    d, length = case["head_dim"], case["length"]
    p = capi.attention_params(QUERY_HEADS, KV_HEADS, d, ROTARY[d], capacity=capacity)
    q_norm, k_norm = _norm_weights(source, d)
    size = capi.lib().pluto_hip_gqa_prefill_workspace_bytes(p, length)
    return dict(p=p, qg=source.normal(length, QUERY_HEADS, 2, d, scale=0.5, dtype=BF16),
                k=source.normal(length, KV_HEADS, d, scale=0.5, dtype=BF16),
                v=source.normal(length, KV_HEADS, d, scale=0.5, dtype=BF16), q_norm=q_norm, k_norm=k_norm,
                cache=capi.KvCache(capacity, KV_HEADS, d), out=_empty(length, QUERY_HEADS, d),
                workspace=_empty(max(size, 1), dtype=torch.uint8))


def _prepare_prefill(case, source):
    s = _attention_inputs(case, source, case["start"] + case["length"])
    s["start"] = case["start"]
    s["cache"].keys.normal_(generator=source.gen)
    s["cache"].values.normal_(generator=source.gen)
    return s


def _run_prefill(s):
    out = capi.gqa_prefill(s["p"], s["qg"], s["k"], s["v"], s["q_norm"], s["k_norm"], s["cache"], start_position=s["start"],
                           out=s["out"], workspace=s["workspace"])
    return out, s["cache"].keys, s["cache"].values


def _prepare_gqa_train(case, source):
    s = _attention_inputs(case, source, case["length"])
    d = case["head_dim"]
    s["saved"] = capi.gqa_prefill_saved(s["p"], case["length"], s["cache"])
    s["dy"] = source.normal(case["length"], QUERY_HEADS, d)
    s["norm_grads"] = torch.zeros(2, d, device="cuda")
    return s


def _run_gqa_train(s):
    s["norm_grads"].zero_()
    out = capi.gqa_prefill(s["p"], s["qg"], s["k"], s["v"], s["q_norm"], s["k_norm"], s["cache"], saved=s["saved"],
                           out=s["out"], workspace=s["workspace"])
    grads = capi.gqa_prefill_backward(s["p"], s["qg"], s["k"], s["v"], s["q_norm"], s["k_norm"], s["dy"],
                                      dq_norm=s["norm_grads"][0], dk_norm=s["norm_grads"][1], saved=s["saved"])
    return (out, s["norm_grads"]) + tuple(grads)


def _prepare_attention_step(case, source):
    d, batch = case["head_dim"], case["batch"]
    lengths = _contexts(case)
    capacity = max(lengths)
    p = capi.attention_params(QUERY_HEADS, KV_HEADS, d, ROTARY[d], capacity=capacity)
    # one pool of keys and one of values for all sequences, as a server keeps them
    keys = source.normal(batch, KV_HEADS, capacity, d, dtype=BF16)
    values = source.normal(batch, KV_HEADS, capacity, d, dtype=BF16)
    caches = []
    for i in range(batch):
        cache = capi.KvCache(capacity, KV_HEADS, d)
        cache.keys, cache.values = keys[i], values[i]
        caches.append(cache)
    positions = [n - 1 for n in lengths]
    q_norm, k_norm = _norm_weights(source, d)
    return dict(p=p, keys=keys, values=values, caches=caches, positions=positions, q_norm=q_norm, k_norm=k_norm,
                hidden=source.normal(batch, WIDTH, dtype=BF16), attended=_empty(batch, QUERY_HEADS, d),
                into=_Projection(source, case["storage"], batch, WIDTH, [2 * QUERY_HEADS * d, KV_HEADS * d, KV_HEADS * d]),
                onto=_Projection(source, case["storage"], batch, QUERY_HEADS * d, [WIDTH]),
                workspace=capi.gqa_decode_workspace(p, positions))


def _run_attention_step(s):
    q_gate, k, v = s["into"](s["hidden"])
    p, batch = s["p"], s["hidden"].shape[0]
    attended = capi.gqa_decode(p, q_gate.view(batch, p.query_heads, 2, p.head_dim), k.view(batch, p.key_value_heads, p.head_dim),
                               v.view(batch, p.key_value_heads, p.head_dim), s["q_norm"], s["k_norm"], s["caches"],
                               positions=s["positions"], workspace=s["workspace"], out=s["attended"], advance=False)
    return s["onto"](attended.view(batch, -1)), attended, s["keys"], s["values"]


def _prepare_delta_step(case, source):
    batch = case["batch"]
    p = capi.delta_params(KEY_HEADS, VALUE_HEADS, DELTA_DIM, DELTA_DIM, CONV_TAPS)
    values = VALUE_HEADS * DELTA_DIM
    channels = 2 * KEY_HEADS * DELTA_DIM + values
    states = capi.DeltaNetStep(p, batch=batch)
    states.conv.normal_(generator=source.gen)
    states.state.normal_(generator=source.gen).mul_(0.1)
    return dict(states=states, weights=_delta_weights(source, p), hidden=source.normal(batch, WIDTH, dtype=BF16),
                into=_Projection(source, case["storage"], batch, WIDTH, [channels, values, VALUE_HEADS, VALUE_HEADS]),
                onto=_Projection(source, case["storage"], batch, values, [WIDTH]))


def _run_delta_step(s):
    qkv, z, a, b = s["into"](s["hidden"])
    mixed = s["states"].step(qkv, z, a, b, **s["weights"])
    return s["onto"](mixed), mixed, s["states"].state, s["states"].conv


def _delta_inputs(case, source):
    batch, length = case["batch"], case["length"]
    p = capi.delta_params(case["key_heads"], case["value_heads"], DELTA_DIM, DELTA_DIM, CONV_TAPS)
    values = p.value_heads * DELTA_DIM
    channels = 2 * p.key_heads * DELTA_DIM + values
    args = dict(qkv=source.normal(batch, length, channels, dtype=BF16), z=source.normal(batch, length, values, dtype=BF16),
                a=source.normal(batch, length, p.value_heads, dtype=BF16), b=source.normal(batch, length, p.value_heads, dtype=BF16))
    args.update(_delta_weights(source, p))
    return p, args


def _prepare_delta_prefill(case, source):
    p, args = _delta_inputs(case, source)
    return dict(p=p, args=args, state=_empty(case["batch"], p.value_heads, DELTA_DIM, DELTA_DIM, dtype=torch.float32))


def _run_delta_prefill(s):
    s["state"].zero_()
    return capi.gdn_layer_forward(s["p"], **s["args"], state=s["state"]), s["state"]


def _prepare_delta_backward(case, source):
    p, args = _delta_inputs(case, source)
    sizes = {n: args[n].numel() for n in ("conv_weight", "a_log", "dt_bias", "norm")}
    # one flat buffer for the parameters' gradients, cleared once a step
    flat = torch.zeros(sum(sizes.values()), device="cuda")
    pieces = dict(zip(sizes, torch.split(flat, list(sizes.values()))))
    return dict(p=p, args=args, dy=source.normal(case["batch"], case["length"], p.value_heads * DELTA_DIM), flat=flat,
                grads={n: piece.view(args[n].shape) for n, piece in pieces.items()})


def _run_delta_backward(s):
    s["flat"].zero_()
    return tuple(capi.gdn_layer_backward(s["p"], **s["args"], dy=s["dy"], parameter_grads=s["grads"])) + (s["flat"],)


def prepare(case, seed):
    return dict(globals()["_prepare_" + case["kind"]](case, _Source(seed)), kind=case["kind"])


def run(state):
    return globals()["_run_" + state["kind"]](state)


# ---- what a pass cannot do without ---------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "mha_train":
        B, T, H, D = case["batch"], case["length"], case["heads"], case["head_dim"]
        size = 2 if case["dtype"] == "bf16" else 4
        one = B * T * H * D
        # two products forward, five backward, over the visible half
        return {"flops": 14.0 * B * H * D * (T * (T + 1) // 2), "bytes": one * (3 * size + size + 4 + 12) + 2.0 * B * H * T * 4}
    if kind == "dense_train":
        rows, n_in, n_out = case["rows"], case["input_dim"], case["output_dim"]
        size = 2 if case["dtype"] == "bf16" else 4
        return {"flops": 6.0 * rows * n_in * n_out,
                "bytes": rows * (n_in * size + n_out * size + n_out * 4.0 + n_in * 4) + 8.0 * n_in * n_out + 8.0 * n_out}
    if kind in ("prefill", "gqa_train"):
        T, d, start = case["length"], case["head_dim"], case.get("start", 0)
        pairs = T * start + T * (T + 1) // 2
        new = T * (QUERY_HEADS * 2 + 2 * KV_HEADS) * d
        moved = 2.0 * new + 2.0 * (T * QUERY_HEADS + 2 * (T + start) * KV_HEADS + 2 * T * KV_HEADS) * d
        if kind == "prefill":
            return {"flops": 4.0 * QUERY_HEADS * d * pairs, "bytes": moved - 2.0 * 2 * T * KV_HEADS * d}
        return {"flops": 14.0 * QUERY_HEADS * d * pairs, "bytes": moved + 4.0 * T * QUERY_HEADS * d + 4.0 * new}
    if kind == "attention_step":
        d, batch = case["head_dim"], case["batch"]
        total = sum(_contexts(case))
        into, onto = (2 * QUERY_HEADS + 2 * KV_HEADS) * d, QUERY_HEADS * d
        weights = WIDTH * (into + onto)
        return {"flops": 2.0 * batch * weights + 4.0 * QUERY_HEADS * d * total,
                "bytes": weights * (1.0 if case["storage"] == "fp8" else 2.0) + 4.0 * KV_HEADS * d * total
                + 2.0 * batch * (2 * WIDTH + onto)}
    if kind == "delta_step":
        batch, values = case["batch"], VALUE_HEADS * DELTA_DIM
        channels = 2 * KEY_HEADS * DELTA_DIM + values
        weights = WIDTH * (channels + values + 2 * VALUE_HEADS + values)
        state = VALUE_HEADS * DELTA_DIM * DELTA_DIM
        return {"flops": batch * (2.0 * weights + 7.0 * state),
                "bytes": weights * (1.0 if case["storage"] == "fp8" else 2.0) + 8.0 * batch * (state + channels * CONV_TAPS)
                + 2.0 * batch * (2 * WIDTH + values)}
    tokens, vh = case["batch"] * case["length"], case["value_heads"]
    values = vh * DELTA_DIM
    channels = 2 * case["key_heads"] * DELTA_DIM + values
    recurrence = float(tokens) * vh * DELTA_DIM * DELTA_DIM
    if kind == "delta_prefill":
        return {"flops": 7 * recurrence, "bytes": 2.0 * tokens * (channels + 2 * values + 2 * vh) + 8.0 * case["batch"] * values * DELTA_DIM}
    return {"flops": 22 * recurrence, "bytes": tokens * (6.0 * channels + 6.0 * values + 12.0 * vh + 4.0 * values)}


def tolerance(case):
    kind = case["kind"]
    if case.get("dtype") == "f32":
        # FP32 results of FP32 sums (the dense layer's operands are half precision by definition)
        return {"rel": 1e-5}
    if kind == "delta_backward":
        # FP32 sums; forward values that lie on a tie of their bf16 rounding may fall either way
        return {"rel": 1e-4, "max": 0.05}
    return {"rel": 1e-2}
