"""The work this framework is measured on: decode waves and prefill blocks of the hybrid
stack (G,G,G,A: three Gated DeltaNet layers to one full-attention layer, hidden 2048), the way
a host drives it - tatara_amd.stack over the backend's command buffers, projections from
affine 4-bit weights or plain bf16 matrices, lane state in pools that stay on the GPU.

Eight layers (two periods of the pattern) stand for the forty of the model, each with its own
weights, caches and state.  A decode wave is recorded once and replayed as a compiled graph,
one replay per token, as a serving loop does; a prefill block has a position and a row count
of its own and is recorded afresh by every pass."""
import math

import torch

from tatara_amd import backend, stack

LAYERS = 8
VOCAB = 1024
ATTENTION_LAYERS = stack.layer_kinds(LAYERS).count("A")
GDN_LAYERS = LAYERS - ATTENTION_LAYERS


def _decode(name, lanes, shallowest, deepest, capacity, weights="q4"):
    return {"name": name, "mode": "decode", "weights": weights, "lanes": lanes,
            "shallowest": shallowest, "deepest": deepest, "capacity": capacity}


def _prefill(name, rows, cached, capacity, weights="q4"):
    return {"name": name, "mode": "prefill", "weights": weights, "rows": rows, "cached": cached,
            "capacity": capacity}


def listed():
    return [
        # one conversation near its start: the least work a token can be, launches and latency
        _decode("decode-1-short", 1, 1000, 1000, 8192),
        # one conversation over a document: the deepest single lane that is swept
        _decode("decode-1-deep", 1, 99999, 99999, 100096),
        # a few chats of ordinary, unequal lengths in caches with room to grow
        _decode("decode-4-chats", 4, 700, 6001, 32768),
        # four lanes at 32768 visible keys: the headline decode shape, caches full
        _decode("decode-4-full", 4, 32767, 32767, 32768),
        # the widest wave there is: sixteen lanes, from just started to a long transcript
        _decode("decode-16-mixed", 16, 150, 12000, 16384),
        # a verified draft or a tool's short answer: a dozen rows into a running conversation
        _prefill("prefill-12-draft", 12, 5003, 8192),
        # a short prompt from nothing: most requests of a chat
        _prefill("prefill-100-prompt", 100, 0, 4096),
        # an ordinary follow-up turn, an odd number of rows at an odd position
        _prefill("prefill-777-turn", 777, 1501, 8192),
        # a full block of the blocked prefill, late in a 32k-token prompt
        _prefill("prefill-2048-late", 2048, 30720, 32768),
        # the same block size early in a prompt, over plain bf16 projections
        _prefill("prefill-2048-dense", 2048, 4096, 32768, "dense"),
        # a long document in one block: the largest block that is prefilled at once
        _prefill("prefill-16384-document", 16384, 0, 16384),
    ]


def _spread(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    weights = "dense" if rng.random() < 0.15 else "q4"
    if rng.random() < 0.5:
        deepest = _spread(rng, 200, 100000)
        shallowest = min(deepest, _spread(rng, 100, 100000)) if rng.random() < 0.7 else deepest
        capacities = [c for c in (4096, 8192, 16384, 32768, 65536, 131072) if c > deepest]
        lanes = rng.choice((1, 1, 2, 3, 4, 4, 6, 8, 11, 16))
        return {"mode": "decode", "weights": weights, "lanes": lanes, "shallowest": shallowest,
                "deepest": deepest, "capacity": rng.choice(capacities[:2])}
    rows = _spread(rng, 2, 8192)
    cached = 0 if rng.random() < 0.3 else _spread(rng, 20, 32768 - rows)
    return {"mode": "prefill", "weights": weights, "rows": rows, "cached": cached,
            "capacity": rng.choice([c for c in (4096, 8192, 16384, 32768) if c >= cached + rows])}


def _contexts(case):
    """Cached positions of every lane: from the shallowest to the deepest in equal ratios."""
    lanes, low, high = case["lanes"], case["shallowest"], case["deepest"]
    return [int(round(high * (low / high) ** (lane / max(lanes - 1, 1)))) for lane in range(lanes)]


# ---- what a host keeps: one device, one queue and one kernel library per process ----
_process = {}


def _backend():
    if not _process:
        device = backend.Device()
        _process.update(device=device, queue=device.create_queue(), library=device.create_library())
    return _process["device"], _process["queue"], _process["library"]


def _words(tensor, dtype=None):
    host = tensor.cpu().contiguous().view(torch.int16 if tensor.dtype == torch.bfloat16 else tensor.dtype)
    host = host.numpy().reshape(-1)
    return host.view(dtype) if dtype is not None else host


def _weights(gen, form):
    """The stack's weights as tatara_amd.stack.make_weights lays them out and scales them,
    made on the GPU: bf16 as uint16 host arrays, 4-bit as (words, scales, biases)."""
    def normal(n, sigma, mean=0.0):
        t = torch.randn(n, generator=gen, device="cuda") * sigma + mean
        return _words(t.to(torch.bfloat16), "uint16")

    def uniform(n, low, high):
        t = torch.rand(n, generator=gen, device="cuda") * (high - low) + low
        return _words(t.to(torch.bfloat16), "uint16")

    def quantized(rows, k, sigma):
        words = torch.randint(-2 ** 31, 2 ** 31, (rows * k // 8,), generator=gen, device="cuda",
                              dtype=torch.int64).to(torch.int32)
        scale = (torch.rand(rows * k // 64, generator=gen, device="cuda") * 0.4 + 0.8) * (sigma / 4.61)
        return (_words(words, "uint32"), _words(scale.to(torch.bfloat16), "uint16"),
                _words((-7.5 * scale).to(torch.bfloat16), "uint16"))

    hidden = stack.HIDDEN
    out = {"layers": [], "final_norm": normal(hidden, 0.05, 1.0),
           "vocab": normal(VOCAB * hidden, hidden ** -0.5)}
    for kind in stack.layer_kinds(LAYERS):
        gated = kind == "G"
        layer = {"kind": kind, "input_norm": normal(hidden, 0.05, 1.0)}
        if gated:
            layer.update(conv_w=normal(4 * 8192, 0.5), a_log=uniform(32, -4.0, -2.5),
                         dt_bias=normal(32, 0.3), norm_w=normal(128, 0.1, 1.0))
        else:
            layer.update(q_norm=normal(256, 0.1, 1.0), k_norm=normal(256, 0.1, 1.0))
        if form == "q4":
            segments = stack.GDN_SEGMENTS if gated else stack.ATTN_SEGMENTS
            layer["in_q4"] = [quantized(rows, hidden, hidden ** -0.5) for rows in segments]
            layer["out_q4"] = quantized(hidden, 4096, 0.5 * 4096 ** -0.5)
        else:
            width = stack.GDN_PROJ if gated else stack.ATTN_PROJ
            layer["w_in"] = normal(width * hidden, hidden ** -0.5)
            layer["w_out"] = normal(hidden * 4096, 0.5 * 4096 ** -0.5)
        out["layers"].append(layer)
    return out


class _DeviceMemory:
    """A backend buffer as torch sees it (its bytes, no copy)."""

    def __init__(self, buffer):
        self.buffer = buffer
        self.__cuda_array_interface__ = {"shape": (buffer.size_bytes // 2,), "typestr": "<i2",
                                         "data": (buffer.device_pointer, False), "version": 2}


def _bf16_view(buffer):
    return torch.as_tensor(_DeviceMemory(buffer), device="cuda").view(torch.bfloat16)


def prepare(case, seed):
    """The stack with its weights, the lanes' caches and states as they stand after the cached
    tokens (normed keys, values, conv windows and recurrent states of the magnitudes the path
    leaves), the new tokens' embeddings, and for a decode wave its compiled recording."""
    device, queue, library = _backend()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)

    def randn(*shape, dtype=torch.bfloat16, sigma=1.0):
        t = torch.randn(shape, generator=gen, device="cuda", dtype=dtype)
        return t.mul_(sigma) if sigma != 1.0 else t

    decode = case["mode"] == "decode"
    lanes = case["lanes"] if decode else 1
    contexts = _contexts(case) if decode else [case["cached"]]
    rows = lanes if decode else case["rows"]
    capacity = case["capacity"]
    st = stack.StubStack(device, library, _weights(gen, case["weights"]), lanes, capacity, VOCAB,
                         block_rows=16 if decode else max(2048, (rows + 31) // 32 * 32))
    # lane state in the host's own pools, adopted by the stack
    keys_values = randn(2, ATTENTION_LAYERS, lanes, 2, capacity, 256)
    conv = randn(GDN_LAYERS, 2 * lanes, 3, 8192, sigma=0.5)
    recurrent = randn(GDN_LAYERS, 2 * lanes, 32, 128, 128, dtype=torch.float32, sigma=0.02)
    tokens = randn(rows, stack.HIDDEN)

    def adopt(t):
        return device.wrap(t.data_ptr(), t.numel() * t.element_size(), keepalive=t)

    attention = gated = 0
    for layer in st.layers:
        if layer["kind"] == "A":
            layer["keys"], layer["values"] = adopt(keys_values[0, attention]), adopt(keys_values[1, attention])
            attention += 1
        else:
            layer["conv"], layer["rec"] = adopt(conv[gated]), adopt(recurrent[gated])
            gated += 1
    st.context = list(contexts)
    st._write_tables()
    state = {"stack": st, "queue": queue, "decode": decode, "rows": rows, "tokens": adopt(tokens),
             "recordings": []}
    # what a pass leaves: the rows behind the last layer, the appended cache rows, the new planes
    out = {"hidden": _bf16_view(st.x)[:rows * stack.HIDDEN].view(rows, stack.HIDDEN),
           "conv": conv[:, 1::2], "recurrent": recurrent[:, 1::2]}
    if decode:
        out["logits"] = _bf16_view(st.logits)[:rows * VOCAB].view(rows, VOCAB)
        out["appended"] = [keys_values[:, :, lane, :, context] for lane, context in enumerate(contexts)]
        graph = queue.create_command_buffer()
        _record(state, graph)
        state["graph"] = graph.compile()
    else:
        out["appended"] = keys_values[:, :, 0, :, contexts[0]:contexts[0] + rows]
    state["out"] = out
    torch.cuda.synchronize()
    return state


def _record(state, recording):
    st, rows = state["stack"], state["rows"]
    recording.copy_buffer(state["tokens"], 0, st.x, 0, rows * stack.HIDDEN * 2)
    recording.begin_compute_pass()
    if state["decode"]:
        st.record_token_wave(recording)
    else:
        st.record_prefill_block(recording, 0, rows)
    recording.end_compute_pass()


def run(state):
    """One token of every lane, or one block of rows of a lane, through the stack."""
    if state["decode"]:
        state["graph"].commit()
    else:
        recording = state["queue"].create_command_buffer()
        _record(state, recording)
        recording.commit()
        # the block before this one may still be running while this one is recorded
        state["recordings"] = state["recordings"][-1:] + [recording]
    return state["out"]


def work(case):
    decode = case["mode"] == "decode"
    lanes = case["lanes"] if decode else 1
    rows = lanes if decode else case["rows"]
    contexts = _contexts(case) if decode else [case["cached"]]
    hidden = stack.HIDDEN
    matrices = (GDN_LAYERS * stack.GDN_PROJ + ATTENTION_LAYERS * stack.ATTN_PROJ) * hidden \
        + LAYERS * 4096 * hidden
    head = VOCAB * hidden if decode else 0
    cached = sum(contexts)
    pairs = cached + lanes if decode else rows * cached + rows * (rows + 1) // 2
    moved = matrices * (0.5 + 4.0 / 64.0 if case["weights"] == "q4" else 2.0) + head * 2
    moved += 2 * rows * hidden * 2 + (rows * VOCAB * 2 if decode else 0)
    moved += ATTENTION_LAYERS * 2048 * (cached + rows)
    moved += GDN_LAYERS * (lanes * 2 * (32 * 128 * 128 * 4 + 3 * 8192 * 2) + 4 * 8192 * 2)
    flops = 2.0 * rows * (matrices + head)
    flops += ATTENTION_LAYERS * 16 * 1024.0 * pairs
    flops += GDN_LAYERS * rows * (32 * 7 * 128.0 * 128.0 + 8 * 8192)
    return {"bytes": float(moved), "flops": float(flops)}


def tolerance(case):
    """Eight layers of bf16 stages: every projection, norm, cache row and layer output is
    rounded to bf16 once, and the next layer starts from the rounded sum.  The same passes with
    their sums in another order (the reference's order in the projections of a wave, attention
    in three dispatches; the token loop instead of chunks and unshared key walks in a block)
    were 0.0087 apart at most, and 0.19 in the single worst value of a recurrent state."""
    return {"rel": 0.03, "max": 0.7}
