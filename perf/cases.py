"""The calls that a user of gla_jax_amd makes, as cases that can be timed and compared.

A case is a dict of plain values.  `op` names the call:
    chunk_train      chunk_gla, forward and the gradients of all five arrays (a training step of a GLA layer)
    chunk_forward    chunk_gla without gradients (prefill, evaluation)
    recurrent_train  recurrent_gla, forward and gradients
    recurrent_forward  recurrent_gla without gradients; T = 1 is a decode step, the state in float32 as a serving loop
                     carries it from one call to the next
    scans            cumsum_recursive of the log gates within chunks and, from its end, along the whole sequence (as the
                     gates' gradient is formed), and rnn_recursive over the chunk states
Sizes are B sequences of T steps with H heads of D key and D value features; gates are log_sigmoid(shift + N(0,1)).
"""
import math

import torch

from gla_jax_amd import chunk_gla, cumsum_recursive, recurrent_gla, rnn_recursive

# the largest listed case holds this many elements in each of its row arrays; drawn cases stay at or below it
MOST_ELEMENTS = 4 * 4096 * 16 * 128


def _case(op, B, T, H, D, dtype="bf16", shift=5.0, chunk=0, reverse=False):
    return {"op": op, "B": B, "T": T, "H": H, "D": D, "dtype": dtype, "shift": shift, "chunk": chunk, "reverse": reverse}


def listed():
    def named(name, *args, **more):
        return dict(_case(*args, **more), name=name)

    return [
        # serving: one token of one sequence through a 16-head layer: latency, host path and launches
        named("decode_b1", "recurrent_forward", 1, 1, 16, 128, shift=3.0),
        # serving: one token of a batch of 64 sequences: the states' traffic
        named("decode_b64", "recurrent_forward", 64, 1, 16, 128, shift=3.0),
        # serving: the prompt of one sequence
        named("chunk_prefill", "chunk_forward", 1, 8192, 16, 128, chunk=128),
        # training: the benchmark's own step (the reference's headline sizes)
        named("chunk_train", "chunk_train", 4, 4096, 6, 128, chunk=128),
        # training on one long sequence under strong decay (the benchmark's long workload)
        named("chunk_train_long", "chunk_train", 1, 32768, 8, 128, shift=0.0, chunk=128),
        # training at a length that is a multiple of 32 only
        named("chunk_train_ragged", "chunk_train", 3, 1120, 6, 128, chunk=32),
        # a small float32 step: unit tests, gradient checks and research code
        named("chunk_train_fp32", "chunk_train", 1, 512, 2, 64, dtype="fp32", chunk=64),
        # training with the recurrent form on many sequences (the benchmark's recurrent workload)
        named("recurrent_train", "recurrent_train", 16, 2048, 16, 64, shift=3.0),
        # the sizes of the reference's own script: fewer sequences than compute units, 128 features
        named("recurrent_train_few", "recurrent_train", 4, 4096, 16, 128, shift=3.0),
        # an odd length, scanned from its end (the second direction of a bidirectional layer)
        named("recurrent_train_odd", "recurrent_train", 2, 777, 8, 64, shift=3.0, reverse=True),
        # the two scan operators at the sizes that chunked code of a user's own gives them
        named("scans", "scans", 4, 4096, 6, 128, dtype="fp32", chunk=128),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    op = rng.choices(["chunk_train", "chunk_forward", "recurrent_train", "recurrent_forward", "scans"], [6, 3, 5, 4, 2])[0]
    dtype = "fp32" if op == "scans" else rng.choice(["bf16", "bf16", "bf16", "fp32"])
    # head dimensions of trained models; the chunk form in float32 is built up to 128
    D = rng.choice([64, 128, 128] if dtype == "fp32" else [64, 128, 128, 256])
    shift = rng.choice([5.0, 5.0, 3.0, 0.0])
    H = rng.choice([1, 2, 4, 5, 6, 8, 12, 16])
    B = _log_int(rng, 1, 32)
    if op.startswith("chunk") or op == "scans":
        # half of the lengths are multiples of 128, the others of 32 or 64 only
        unit = rng.choice([128, 128, 64, 32])
        T = unit * max(1, _log_int(rng, 128, 32768) // unit)
        chunk = min(128, T & -T)
    else:
        chunk = 0
        T = 1 if op == "recurrent_forward" and rng.random() < 0.5 else _log_int(rng, 16, 8192)
        if T == 1:
            B = _log_int(rng, 1, 64)
    most = MOST_ELEMENTS // (2 if dtype == "fp32" or D == 256 else 1)  # no more bytes or operations than the largest listed case
    while B * T * H * D > most:
        if B > 1:
            B = max(1, B // 2)
        else:
            T = max(1, T // (2 * (chunk or 1))) * (chunk or 1)
    return _case(op, B, T, H, D, dtype, shift, chunk, rng.random() < 0.3 if op.startswith("recurrent") and T > 1 else False)


def prepare(case, seed):
    B, T, H, D = case["B"], case["T"], case["H"], case["D"]
    dt = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, generator=gen, device="cuda")

    g = torch.nn.functional.logsigmoid(case["shift"] + normal(B, T, H, D))
    if case["op"] == "scans":
        C = case["chunk"]
        return {"op": "scans", "gates": g.reshape(B * (T // C), C, H * D), "dgates": normal(B, T, H * D),
                # per chunk: total log decay and the key-value product of its rows
                "decay": g.reshape(B, T // C, C, H, D).sum(2).permute(0, 2, 1, 3).reshape(B * H, T // C, D).contiguous(),
                "products": normal(B * H, T // C, D, D) * math.sqrt(C), "decay_init": torch.zeros(B * H, D, device="cuda"), "init": normal(B * H, D, D)}
    train = case["op"].endswith("train")
    h0 = normal(B, H, D, D).to(torch.float32 if case["op"] == "recurrent_forward" else dt)
    v, k, q = (normal(B, T, H, D).to(dt) for _ in range(3))
    state = {"op": case["op"], "chunk": case["chunk"], "reverse": case["reverse"], "arrays": [t.requires_grad_(train) for t in (h0, g, v, k, q)]}
    if train:
        state["cotangents"] = [normal(B, H, D, D).to(dt), normal(B, T, H, D).to(dt)]
    return state


def run(state):
    op = state["op"]
    if op == "scans":
        sums = cumsum_recursive(state["gates"], 1)
        dgates = cumsum_recursive(state["dgates"], 1, reverse=True)
        decay, states = rnn_recursive(state["decay"], state["products"], state["decay_init"], state["init"])
        return sums, dgates, decay, states
    arrays = state["arrays"]

    def layer():
        return chunk_gla(*arrays, state["chunk"]) if op.startswith("chunk") else recurrent_gla(*arrays, reverse=state["reverse"])

    if not op.endswith("train"):
        with torch.no_grad():
            return layer()
    outputs = layer()
    return outputs + torch.autograd.grad(outputs, arrays, state["cotangents"])


def work(case):
    B, T, H, D = case["B"], case["T"], case["H"], case["D"]
    e = 2 if case["dtype"] == "bf16" else 4
    rows, states = B * T * H * D, B * H * D * D
    if case["op"] == "scans":
        n = B * H * (T // case["chunk"])
        return {"bytes": 16 * rows + 8 * n * (D * D + D) + 4 * states, "flops": 2 * rows + 2 * n * D * D}
    # the recurrence: a rank-1 update and a product with the state in the forward, the states formed again and four more
    # such products (dq, dk, dv, dstate) in the backward, 2 D^2 operations each
    if case["op"].endswith("train"):  # read gates, v, k, q, dout; write out, dv, dk, dq, dgates; four state arrays
        return {"bytes": rows * (8 + 8 * e) + 4 * states * e, "flops": 14 * rows * D}
    e_state = 4 if case["op"] == "recurrent_forward" else e
    return {"bytes": rows * (4 + 4 * e) + 2 * states * e_state, "flops": 4 * rows * D}


def tolerance(case):
    # four times what the outputs differ by from the recurrence in float64 (2-norm), measured over listed and drawn cases;
    # the largest single difference reads larger in the gates' gradient under strong decay, a sum that cancels
    if case["op"] == "scans":  # 5e-7; a single value 5e-6 of the root mean square
        return {"rel": 2e-6, "max": 2e-5}
    if case["dtype"] == "fp32":  # 8e-7; 5e-5
        return {"rel": 3e-6, "max": 1e-4}
    if case["op"].startswith("chunk"):  # operands and states in bf16: 3.4e-3; 0.12
        return {"rel": 1.3e-2, "max": 0.5}
    return {"rel": 7e-3, "max": 0.12}  # the results' own rounding to bf16: 1.7e-3; 0.04
