"""Timed workloads of the decoder path: what a program that generates text, fills prompts or multiplies by quantized
matrices has the library do, through the C ABI and the loader's Model.

Every size is one of the repository's own decoder shapes (neura_amd.synth.SHAPES), at the planes, contexts and prompt
lengths its tests and its benchmark use, and odd ones between them.  Weights are random-init blocks made on the GPU:
uniform codes, one super scale a block, and minimums (or signs of the sub-scales) that centre the values, so a matrix has
mean 0 and a deviation of 0.02 whatever its element.
"""
import ctypes
import math

import numpy as np
import torch

import neura_amd
from neura_amd import NH_F16, NH_F32, NH_Q3_K, NH_Q4_K, NH_Q5_K, NH_Q6_K, NH_Q8_0, synth
from neura_amd.loader import ALIGNMENT, Model, Weights

NH_BF16 = 30
ELEMENTS = {"q8_0": NH_Q8_0, "q3_k": NH_Q3_K, "q4_k": NH_Q4_K, "q5_k": NH_Q5_K, "q6_k": NH_Q6_K}
STATES = {"half": NH_F16, "bfloat16": NH_BF16, "single": NH_F32}
SPREAD = 0.02  # standard deviation of a random-init weight


def listed():
    return [
        # the four products of one layer of a small decoder, one token: the smallest calls, where launches and latency count
        {"name": "products_1_5b_q4_k", "kind": "products", "shape": "qwen2.5-1.5b", "element": "q4_k", "rows": 1},
        # one projection over a 512-token chunk with half activations: the plain wide product
        {"name": "wide_q4_k_512", "kind": "wide", "element": "q4_k", "n": 18944, "k": 3584, "m": 512, "half": True},
        # interactive generation, one sequence: the smallest decoder, the headline decoder, the mix of elements its files ship in
        {"name": "decode_0_5b_q8_0", "kind": "decode", "shape": "qwen2.5-0.5b", "mix": "q8_0", "planes": 1, "context": 1088,
         "states": "half", "sampled": False, "steps": 8},
        {"name": "decode_7b_q4_k", "kind": "decode", "shape": "qwen2.5-7b", "mix": "q4_k", "planes": 1, "context": 4096, "states": "half",
         "sampled": False, "steps": 8},
        {"name": "decode_7b_q4_k_m", "kind": "decode", "shape": "qwen2.5-7b", "mix": "q4_k_m", "planes": 1, "context": 4096,
         "states": "half", "sampled": False, "steps": 8},
        # several sequences stepping together, each at a position of its own
        {"name": "decode_7b_q4_k_8_planes", "kind": "decode", "shape": "qwen2.5-7b", "mix": "q4_k", "planes": 8, "context": 4096,
         "states": "half", "sampled": False, "steps": 8},
        {"name": "decode_7b_q4_k_m_5_planes", "kind": "decode", "shape": "qwen2.5-7b", "mix": "q4_k_m", "planes": 5, "context": 2048,
         "states": "half", "sampled": False, "steps": 8},
        # a small server: sixteen sequences, every token drawn
        {"name": "decode_1_5b_q4_k_16_planes", "kind": "decode", "shape": "qwen2.5-1.5b", "mix": "q4_k", "planes": 16, "context": 1088,
         "states": "half", "sampled": True, "steps": 8},
        # time to the first token: a long prompt, a short one of an odd length behind a kept prefix, prompts of several planes
        {"name": "fill_7b_q4_k_512", "kind": "fill", "shape": "qwen2.5-7b", "mix": "q4_k", "planes": 1, "rows": 512, "cursor": 0,
         "context": 1088, "states": "half"},
        {"name": "fill_7b_q4_k_m_37", "kind": "fill", "shape": "qwen2.5-7b", "mix": "q4_k_m", "planes": 1, "rows": 37, "cursor": 700,
         "context": 1088, "states": "half"},
        {"name": "fill_0_5b_q8_0_4x100", "kind": "fill", "shape": "qwen2.5-0.5b", "mix": "q8_0", "planes": 4, "rows": 100, "cursor": 0,
         "context": 1088, "states": "half"},
    ]


def spread(rng, low, high):
    """a whole number between low and high, even over its logarithm"""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    kind = rng.choice(("products", "wide", "decode", "decode", "decode", "fill", "fill", "fill"))
    if kind == "products":
        shape = rng.choice(sorted(synth.SHAPES))
        element = "q8_0" if shape == "qwen2.5-0.5b" else rng.choice(("q8_0", "q3_k", "q4_k", "q4_k", "q5_k", "q6_k"))
        return {"kind": kind, "shape": shape, "element": element, "rows": rng.randint(1, 8)}
    if kind == "wide":
        _, n, k = rng.choice(synth.layer_matrices(synth.SHAPES[rng.choice(("qwen2.5-1.5b", "qwen2.5-7b"))]))
        return {"kind": kind, "element": rng.choice(("q8_0", "q3_k", "q4_k", "q4_k", "q5_k", "q6_k")), "n": n, "k": k,
                "m": spread(rng, 9, 512), "half": rng.random() < 0.5}
    shape = rng.choice(("qwen2.5-0.5b", "qwen2.5-1.5b", "qwen2.5-7b", "qwen2.5-7b"))
    case = {"kind": kind, "shape": shape, "mix": rng.choice({"qwen2.5-0.5b": ("q8_0",), "qwen2.5-1.5b": ("q4_k", "q4_k_m", "q8_0"),
                                                             "qwen2.5-7b": ("q4_k", "q4_k", "q4_k_m", "q5_k_m", "q3_k_m")}[shape])}
    states = rng.choice(("half", "half", "half", "bfloat16", "single"))
    if kind == "decode":
        planes = spread(rng, 1, 8 if shape == "qwen2.5-7b" else 16)
        return dict(case, planes=planes, context=spread(rng, 64, 4096), states=states, sampled=rng.random() < 0.25,
                    steps=rng.randint(4, 8) if planes < 3 else 4 if planes < 5 else 3)
    planes = rng.choice((1, 1, 2, 4))
    rows = spread(rng, 5, 480 // planes)
    cursor = rng.choice((0, rng.randint(1, 1500)))
    return dict(case, planes=planes, rows=rows, cursor=cursor, context=2048, states=states)


# ---- weights made on the GPU -------------------------------------------------------------------


def halves_at(raw, at, values):
    raw[:, at:at + 2] = values.to(torch.float16).reshape(-1, 1).view(torch.uint8)


def blocks(generator, element, rows, columns):
    """uint8 [rows * columns / block, block bytes] of a matrix with mean 0 and deviation SPREAD"""
    per, size = synth.BLOCK_BYTES[element]
    count = rows * columns // per
    raw = torch.randint(0, 256, (count, size), dtype=torch.uint8, device="cuda", generator=generator)
    scale = SPREAD * (0.75 + 0.5 * torch.rand(count, device="cuda", generator=generator))
    if element == NH_Q8_0:  # codes -127..127
        raw[:, 2:] = torch.where(raw[:, 2:] == 128, 0, raw[:, 2:])
        halves_at(raw, 0, scale / 73.3)
    elif element in (NH_Q4_K, NH_Q5_K):  # d * sc * code - dmin * m, with m = sc and dmin = d * the middle code
        steps = 16 if element == NH_Q4_K else 32
        d = scale / (48.4 * math.sqrt((steps * steps - 1) / 12.0))
        halves_at(raw, 0, d)
        halves_at(raw, 2, d * (steps - 1) / 2)
        sc = 32 + (raw[:, 4:12] & 31)
        low = sc[:, :4] | ((sc[:, 4:] >> 4) << 6)
        raw[:, 4:8], raw[:, 8:12] = low, low
        raw[:, 12:16] = (sc[:, 4:] & 15) | ((sc[:, 4:] & 15) << 4)
    elif element == NH_Q6_K:  # sub-scales of either sign, 32..127 in magnitude
        sc = 32 + torch.randint(0, 96, (count, 16), dtype=torch.int16, device="cuda", generator=generator)
        sc = torch.where(raw[:, 192:208] >= 128, -sc, sc)
        raw[:, 192:208] = sc.to(torch.int8).view(torch.uint8)
        halves_at(raw, 208, scale / (84.3 * 18.5))
    else:  # Q3_K: any bytes are sub-scales, -32..31 once read
        halves_at(raw, 108, scale / (18.5 * 2.35))
    return raw


def mixture(shape, mix):
    """(element, matrices stored otherwise, layers with q/k/v biases): the recipes of the K-quant files, as the benchmark has them"""
    if mix in ELEMENTS:
        return ELEMENTS[mix], {}, ()
    count = shape["layers"]
    base = {"q4_k_m": NH_Q4_K, "q5_k_m": NH_Q5_K, "q3_k_m": NH_Q3_K}[mix]
    held = {"output.weight": NH_Q6_K}
    if shape["tied"]:
        held = {"token_embd.weight": NH_Q6_K}
    for i in range(count):
        more = i < count // 8 or i >= 7 * count // 8 or (i - count // 8) % 3 == 2
        if base == NH_Q3_K:
            held["blk.%d.attn_output.weight" % i] = NH_Q4_K
            held["blk.%d.attn_v.weight" % i] = held["blk.%d.ffn_down.weight" % i] = NH_Q5_K if more else NH_Q4_K
        elif more:
            held["blk.%d.attn_v.weight" % i] = held["blk.%d.ffn_down.weight" % i] = NH_Q6_K
    return base, held, tuple(range(count))


def matrices(shape, mix):
    """(name, element, rows, columns) of every matrix of a decoder"""
    base, held, _ = mixture(shape, mix)
    names = [("token_embd.weight", shape["vocab"], shape["hidden"])]
    for i in range(shape["layers"]):
        names += [("blk.%d.%s.weight" % (i, name), rows, columns) for name, rows, columns in synth.layer_matrices(shape)]
    if not shape["tied"]:
        names.append(("output.weight", shape["vocab"], shape["hidden"]))
    return [(name, held.get(name, base), rows, columns) for name, rows, columns in names]


def load_weights(device, shape, mix, generator):
    """one arena filled on the GPU, tensor by tensor"""
    _, _, biased = mixture(shape, mix)
    hidden, kv = shape["hidden"], shape["kv_heads"] * shape["head_dim"]
    vectors = [("output_norm.weight", hidden)]
    for i in range(shape["layers"]):
        vectors += [("blk.%d.attn_norm.weight" % i, hidden), ("blk.%d.ffn_norm.weight" % i, hidden)]
        if i in biased:
            vectors += [("blk.%d.attn_q.bias" % i, shape["heads"] * shape["head_dim"]), ("blk.%d.attn_k.bias" % i, kv), ("blk.%d.attn_v.bias" % i, kv)]

    def aligned(nbytes):
        return -(-nbytes // ALIGNMENT) * ALIGNMENT

    wanted = matrices(shape, mix)
    total = sum(aligned(synth.matrix_bytes(element, rows, columns)) for _, element, rows, columns in wanted)
    total += sum(aligned(4 * n) for _, n in vectors)
    weights = Weights(device, (), total_bytes=total)

    def put(name, element, tensor):
        weights.offsets[name], weights.elements[name] = weights.used, element
        torch.cuda.synchronize()
        nbytes = tensor.numel() * tensor.element_size()
        checked(device, device.lib.nh_copy(device.handle, weights.pointer(name), tensor.data_ptr(), nbytes))
        device.sync()
        weights.used += aligned(nbytes)

    for name, element, rows, columns in wanted:
        put(name, element, blocks(generator, element, rows, columns))
    for name, n in vectors:
        values = torch.randn(n, device="cuda", generator=generator)
        put(name, NH_F32, 1.0 + 0.1 * values if "norm" in name else 0.5 * values)
    return weights


# ---- states --------------------------------------------------------------------------------------


def checked(device, status):
    if status != 0:
        raise neura_amd.NeuraError(status, device.lib.nh_last_error().decode())


class State:
    """what a program holds between calls; the handles go with it"""

    def __init__(self, case):
        self.case, self.device, self.weights, self.model = case, neura_amd.Device(0), None, None

    def __del__(self):
        for held in (self.model, self.weights):
            if held is not None:
                held.release()
        self.device.close()


def fill_states(state, generator):
    """N(0, 1) keys and values in every position, as the benchmark's caches hold"""
    model, element = state.model, STATES[state.case["states"]]
    kind = {NH_F16: torch.float16, NH_BF16: torch.bfloat16, NH_F32: torch.float32}[element]
    for layer in range(model.layers):
        for which in (0, 1):
            values = torch.randn(model.cache_shape, device="cuda", generator=generator).to(kind).cpu()
            model.cache_write(layer, which, values.numpy() if element == NH_F32 else values.view(torch.int16).numpy().view(np.uint16))


def prepare(case, seed):
    state = State(case)
    generator = torch.Generator(device="cuda").manual_seed(seed)
    rng = np.random.default_rng(seed)
    if case["kind"] == "products":
        shape, element = synth.SHAPES[case["shape"]], ELEMENTS[case["element"]]
        hidden, ffn, rows = shape["hidden"], shape["ffn"], case["rows"]
        width = (shape["heads"] + 2 * shape["kv_heads"]) * shape["head_dim"]
        state.calls = []
        # q|k|v, attn_output onto the residual stream, gate|up with SwiGLU, ffn_down onto the residual stream
        for n, k, swiglu in ((width, hidden, 0), (hidden, shape["heads"] * shape["head_dim"], 0), (2 * ffn, hidden, 1), (hidden, ffn, 0)):
            y = torch.empty((rows, n // 2 if swiglu else n), device="cuda")
            residual = torch.randn((rows, n), device="cuda", generator=generator) if n == hidden else None
            epilogue = neura_amd.Epilogue(residual.data_ptr() if residual is not None else None, swiglu)
            state.calls.append((element, blocks(generator, element, n, k), n, k, torch.randn((rows, k), device="cuda", generator=generator), rows, y,
                                residual, epilogue))
        return state
    if case["kind"] == "wide":
        element = ELEMENTS[case["element"]]
        state.w = blocks(generator, element, case["n"], case["k"])
        state.x = torch.randn((case["m"], case["k"]), device="cuda", generator=generator).to(torch.float16 if case["half"] else torch.float32)
        state.y = torch.empty((case["m"], case["n"]), device="cuda")
        return state
    shape, planes = synth.SHAPES[case["shape"]], case["planes"]
    state.weights = load_weights(state.device, shape, case["mix"], generator)
    state.model = Model(state.device, state.weights, shape, mixture(shape, case["mix"])[0], batch=planes, context=case["context"],
                        max_rows=case.get("rows", 1), cache_element=STATES[case["states"]])
    fill_states(state, generator)
    if case["kind"] == "decode":
        steps = case["steps"]
        last = case["context"] - steps
        # every plane at its own place in the second half of the context, the first one at its end
        state.cursors = np.array([last] + [int(c) for c in rng.integers(last // 2, last + 1, planes - 1)], dtype=np.uint32)
        state.tokens = rng.integers(0, shape["vocab"], (steps, planes)).astype(np.uint32)
        state.draws = np.empty((steps, planes), dtype=neura_amd.DRAW)
        state.draws["seed"] = 0x3F800000 | rng.integers(0, 1 << 23, (steps, planes))
        state.draws["temperature"], state.draws["keep"], state.draws["cumulative"] = 0.8, 40, 0.95
    else:
        state.prompt = rng.integers(0, shape["vocab"], (case["rows"], planes)).astype(np.uint32)
        state.last = rng.integers(0, shape["vocab"], planes).astype(np.uint32)
        state.cursors = np.full(planes, case["cursor"], dtype=np.uint32)
    return state


def run(state):
    case, device = state.case, state.device
    lib = device.lib
    if case["kind"] == "products":
        for element, w, n, k, x, rows, y, _, epilogue in state.calls:
            checked(device, lib.nh_gemv(device.handle, element, w.data_ptr(), n, k, x.data_ptr(), rows, y.data_ptr(), ctypes.byref(epilogue)))
        return [call[6] for call in state.calls]
    if case["kind"] == "wide":
        checked(device, lib.nh_gemm(device.handle, ELEMENTS[case["element"]], state.w.data_ptr(), case["n"], case["k"], state.x.data_ptr(),
                                    NH_F16 if case["half"] else NH_F32, case["m"], state.y.data_ptr(), None))
        return state.y
    if case["kind"] == "decode":
        # the next tokens of sequences whose text is known: the answer of every step is the model's own choice after it
        chosen = []
        for step in range(case["steps"]):
            if case["sampled"]:
                chosen.append(state.model.decode_step_sampled(state.tokens[step], state.cursors + step, state.draws[step]))
            else:
                chosen.append(state.model.decode_step(state.tokens[step], state.cursors + step))
        return {"chosen": np.stack(chosen), "logits": state.model.logits()}
    # a prompt: all but its last token as one chunk, the last one through the step that answers
    state.model.prefill(state.prompt.reshape(-1), case["rows"], state.cursors)
    chosen = state.model.decode_step(state.last, state.cursors + case["rows"])
    return {"chosen": chosen, "logits": state.model.logits()}


def work(case):
    if case["kind"] == "products":
        shape, rows = synth.SHAPES[case["shape"]], case["rows"]
        sizes = [(n, k) for _, n, k in synth.layer_matrices(shape)]
        weights = sum(synth.matrix_bytes(ELEMENTS[case["element"]], n, k) for n, k in sizes)
        hidden, ffn = shape["hidden"], shape["ffn"]
        wide = (shape["heads"] + 2 * shape["kv_heads"]) * shape["head_dim"]
        # the activation rows in, the residual rows in, the outputs out
        moved = 2 * hidden + shape["heads"] * shape["head_dim"] + ffn + 2 * hidden + wide + 2 * hidden + ffn
        return {"bytes": weights + 4 * rows * moved, "flops": 2.0 * rows * sum(n * k for n, k in sizes)}
    if case["kind"] == "wide":
        n, k, m = case["n"], case["k"], case["m"]
        return {"bytes": synth.matrix_bytes(ELEMENTS[case["element"]], n, k) + m * k * (2 if case["half"] else 4) + 4 * m * n, "flops": 2.0 * m * n * k}
    shape, planes = synth.SHAPES[case["shape"]], case["planes"]
    layer_bytes = layer_weights = head_bytes = 0
    for name, element, rows, columns in matrices(shape, case["mix"]):
        if name.startswith("blk."):
            layer_bytes += synth.matrix_bytes(element, rows, columns)
            layer_weights += rows * columns
        elif name == ("token_embd.weight" if shape["tied"] else "output.weight"):
            head_bytes = synth.matrix_bytes(element, rows, columns)
    head_weights = shape["vocab"] * shape["hidden"]
    per_key = 2 * shape["layers"] * shape["kv_heads"] * shape["head_dim"] * (4 if case["states"] == "single" else 2)  # bytes a position
    key_flops = 4.0 * shape["layers"] * shape["heads"] * shape["head_dim"]  # of one query against one position
    logits = 4 * planes * shape["vocab"]
    if case["kind"] == "decode":
        steps = case["steps"]
        keys = (0.75 * (planes - 1) + 1.0) * case["context"]  # of all planes, on average
        return {"bytes": steps * (layer_bytes + head_bytes + keys * per_key + logits),
                "flops": steps * (2.0 * planes * (layer_weights + head_weights) + keys * key_flops)}
    rows, cursor = case["rows"], case["cursor"]
    seen = sum(cursor + row + 1 for row in range(rows))
    return {"bytes": 2 * layer_bytes + head_bytes + 2 * planes * (cursor + rows) * per_key + logits,
            "flops": 2.0 * planes * ((rows + 1) * layer_weights + head_weights) + planes * (seen + cursor + rows) * key_flops}


def tolerance(case):
    # a product against its matrix in 64 bits: 2-norm 4.3e-7 apart at most, a single output 3.4e-6
    if case["kind"] in ("products", "wide"):
        return {"rel": 2e-6, "max": 1.5e-5}
    # a decode step with its sums in another order (vector products for the matrix cores, another attention): logits 2.3e-5
    # apart, mostly keys and values whose rounding to half fell the other way, one logit 1.7e-4
    if case["kind"] == "decode":
        return {"rel": 1e-4, "max": 7e-4, "differ": 0.01}
    # a fill with its products in fp32 sums of another order: 2.6e-4 and 1.2e-3 (every row's keys and values are rounded again
    # in every layer)
    return {"rel": 1e-3, "max": 5e-3, "differ": 0.01}
