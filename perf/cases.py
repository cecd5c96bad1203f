"""The work a serving program hands to this package, as timed cases.

One pass is what a program does per generated token - one `DynamicDecodeLayer.forward` over the logits of a batch - or,
for beam search, a short request from its first token to the ranked hypotheses, or, for prompts, one scoring call.
Sizes are those of bench.py's workloads where it has one, and ordinary ones of the same kinds elsewhere.
"""
import ctypes
import math

import numpy as np
import torch

import fastertransformer_amd as fa
from fastertransformer_amd import ops

_TYPES = {"f32": fa.F32, "f16": fa.F16, "bf16": fa.BF16}
_WIDTH = {"f32": 4, "f16": 2, "bf16": 2}

# What a sampling step is asked for when a case does not say otherwise. `top_k` lists the values rows choose from (0: a
# row sampled by top-p alone); every lo/hi pair is a range that each row draws its own value from.
_STEP = dict(kind="step", history=64, top_k="64", top_p_lo=0.9, top_p_hi=0.9, top_p_decay=1.0, temperature_lo=1.0,
             temperature_hi=1.0, repetition_lo=1.0, repetition_hi=1.0, presence=0.0, frequency=0.0, min_length=0,
             bad_words=0, stop_words=0, log_probs=False, length_limit=False, logits="normal")


def _step(name, dtype, batch, vocab, pitch=None, **more):
    case = dict(_STEP, dtype=dtype, batch=batch, vocab=vocab, pitch=pitch or vocab, **more)
    return dict(case, name=name) if name else case


def _beam(name, dtype, batch, beams, vocab, steps):
    case = dict(kind="beam", dtype=dtype, batch=batch, beams=beams, vocab=vocab, steps=steps)
    return dict(case, name=name) if name else case


def _score(name, dtype, batch, length, vocab, pitch=None):
    case = dict(kind="score", dtype=dtype, batch=batch, length=length, vocab=vocab, pitch=pitch or vocab)
    return dict(case, name=name) if name else case


def listed():
    return [
        # one interactive user: a single short row, where only latency counts
        _step("one_request_b1_v32000_f16_k40", "f16", 1, 32000, top_k="40", temperature_lo=0.7, temperature_hi=0.7,
              repetition_lo=1.1, repetition_hi=1.1),
        # a handful of users of a GPT-2 size vocabulary, rows of odd length, log-probs returned, stop at a length limit
        _step("small_loop_b8_v50257_f32_k40_logprobs", "f32", 8, 50257, top_k="40", top_p_lo=0.0, top_p_hi=0.0,
              repetition_lo=1.2, repetition_hi=1.2, log_probs=True, length_limit=True),
        # a ragged batch of the same vocabulary in half precision: rows that start between the vectors of the memory
        _step("ragged_b77_v50257_f16_k50", "f16", 77, 50257, top_k="50", temperature_lo=0.7, temperature_hi=1.1,
              repetition_lo=1.1, repetition_hi=1.1, history=301),
        # the headline: a full batch over a large vocabulary
        _step("headline_b256_v128256_f32_k64", "f32", 256, 128256, temperature_lo=0.8, temperature_hi=0.8,
              repetition_lo=1.1, repetition_hi=1.1),
        # every request with a k of its own, from greedy to the largest
        _step("per_row_k_b256_v51200_f16_k1-1024", "f16", 256, 51200, top_k="1,4,16,40,64,1024", temperature_lo=0.8,
              temperature_hi=0.8, repetition_lo=1.1, repetition_hi=1.1),
        # long conversations: 2048 tokens of history, additive penalties, a minimum length, word lists, a length limit
        _step("long_history_b128_v32000_bf16_k50_words", "bf16", 128, 32000, history=2048, top_k="50", top_p_lo=0.0,
              top_p_hi=0.0, presence=0.5, frequency=0.3, min_length=4096, bad_words=64, stop_words=16,
              length_limit=True),
        # the largest batch: log-probs kept for every token of every row
        _step("largest_b1024_v152064_f16_k64_logprobs", "f16", 1024, 152064, history=8, temperature_lo=0.8,
              temperature_hi=0.8, repetition_lo=1.1, repetition_hi=1.1, log_probs=True, length_limit=True),
        # nucleus sampling over whole rows, every row with a p of its own that decays
        _step("top_p_b256_v128256_f32", "f32", 256, 128256, history=1, top_k="0", top_p_lo=0.5, top_p_hi=0.99,
              top_p_decay=0.9, logits="zipf"),
        # a chat service's defaults: nucleus sampling with a temperature and a repetition penalty, log-probs returned
        _step("chat_b64_v128256_bf16_top_p", "bf16", 64, 128256, history=700, top_k="0", top_p_lo=0.9, top_p_hi=0.95,
              temperature_lo=0.6, temperature_hi=1.0, repetition_lo=1.05, repetition_hi=1.2, log_probs=True,
              length_limit=True, logits="zipf"),
        # requests of every kind in one batch: greedy, top-k and nucleus rows, each with its own values
        _step("mixed_b128_v152064_bf16", "bf16", 128, 152064, history=300, top_k="0,0,1,20,50", top_p_lo=0.8,
              top_p_hi=0.99, temperature_lo=0.6, temperature_hi=1.2, repetition_lo=1.0, repetition_hi=1.2,
              logits="zipf"),
        # translation-style beam search, from the first token to the ranked hypotheses
        _beam("beams_b32_k4_v50257_f16", "f16", 32, 4, 50257, 6),
        # prompts scored token by token
        _score("score_b32_t64_v50257_f16", "f16", 32, 64, 50257),
    ]


def _spread(rng, lo, hi):
    """a whole number, its logarithm spread evenly over the range"""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _vocab(rng, most):
    """(columns, pitch): sizes in use, or any size; rows as they are or padded to a multiple of 8, as for a GEMM"""
    known = [v for v in (32000, 50257, 51200, 128256, 152064) if v <= most]
    vocab = rng.choice(known) if known and rng.random() < 0.5 else _spread(rng, 8192, most)
    return vocab, vocab if rng.random() < 0.5 else -(-vocab // 8) * 8


def _batch(rng, vocab, dtype, most_rows, most_bytes):
    return _spread(rng, 1, max(1, min(most_rows, most_bytes // (vocab * _WIDTH[dtype]))))


def draw(rng):
    kind = rng.choice(["top_k", "top_k", "top_k", "log_probs", "log_probs", "per_row_k", "long_history", "top_p",
                       "chat", "mixed", "beam", "score"])
    dtype = rng.choice(["f32", "f16", "bf16"])
    vocab, pitch = _vocab(rng, 152064)
    t_lo = round(rng.uniform(0.5, 1.0), 2)
    values = dict(temperature_lo=t_lo, temperature_hi=round(t_lo + rng.choice([0.0, 0.3]), 2),
                  repetition_lo=rng.choice([1.0, 1.1]), repetition_hi=rng.choice([1.1, 1.2]))
    if kind == "top_k":
        batch = _batch(rng, vocab, dtype, 1024, 300_000_000)
        return _step(None, dtype, batch, vocab, pitch, top_k=rng.choice(["1", "10", "40", "64", "100", "1,20,50"]),
                     top_p_lo=0.8, top_p_hi=1.0, history=_spread(rng, 1, 2000), **values)
    if kind == "log_probs":
        batch = _batch(rng, vocab, dtype, 1024, 250_000_000)
        return _step(None, dtype, batch, vocab, pitch, top_k=rng.choice(["1", "20", "50", "64", "1,20,100"]),
                     history=_spread(rng, 1, 2000), log_probs=True, length_limit=rng.random() < 0.5, **values)
    if kind == "per_row_k":
        batch = _batch(rng, vocab, dtype, 384, 60_000_000)
        return _step(None, dtype, batch, vocab, pitch, top_k=rng.choice(["1,40,200", "1,4,16,40,64,1024", "300"]),
                     history=_spread(rng, 1, 500), **values)
    if kind == "long_history":
        batch = _batch(rng, vocab, dtype, 256, 40_000_000)
        return _step(None, dtype, batch, vocab, pitch, history=_spread(rng, 500, 4000), top_k="50",
                     top_p_lo=0.95, top_p_hi=0.95, presence=0.5, frequency=rng.choice([0.0, 0.3]),
                     min_length=rng.choice([0, 8192]), bad_words=rng.choice([0, 16, 64]),
                     stop_words=rng.choice([0, 4, 16]), length_limit=True)
    if kind == "top_p":
        batch = _batch(rng, vocab, dtype, 256, 100_000_000)
        return _step(None, dtype, batch, vocab, pitch, history=1, top_k="0", top_p_lo=0.5, top_p_hi=0.95,
                     top_p_decay=rng.choice([1.0, 0.9]), log_probs=rng.random() < 0.3, logits="zipf")
    if kind == "chat":
        batch = _batch(rng, vocab, dtype, 256, 40_000_000)
        return _step(None, dtype, batch, vocab, pitch, history=_spread(rng, 10, 2000), top_k="0", top_p_lo=0.8,
                     top_p_hi=0.95, log_probs=rng.random() < 0.5, length_limit=rng.random() < 0.5, logits="zipf",
                     **values)
    if kind == "mixed":
        batch = _batch(rng, vocab, dtype, 256, 40_000_000)
        return _step(None, dtype, batch, vocab, pitch, history=_spread(rng, 10, 2000),
                     top_k=rng.choice(["0,1", "0,50", "0,0,1,20,50"]), top_p_lo=0.8, top_p_hi=0.95, logits="zipf",
                     **values)
    if kind == "beam":
        beams = rng.choice([2, 3, 4, 5, 8])
        vocab, _ = _vocab(rng, 60000)
        return _beam(None, dtype, _spread(rng, 1, 128 // beams), beams, vocab, rng.choice([4, 6]))
    length = _spread(rng, 8, 128)
    batch = max(1, min(32, 200_000_000 // (length * pitch * _WIDTH[dtype])))
    return _score(None, dtype, _spread(rng, 1, batch), length, vocab, pitch)


def _generator(seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    return gen


def _logits(gen, case, rows, end_id):
    """rows of logits as a model leaves them: ordinary columns around zero or falling off like word frequencies
    (Zipf), the end token unlikely in the middle of a text"""
    vocab, pitch = case["vocab"], case.get("pitch", case["vocab"])
    x = torch.randn((rows, pitch), generator=gen, device="cuda")
    if case.get("logits") == "zipf":
        rank = torch.rand((rows, pitch), generator=gen, device="cuda").mul_(vocab).floor_().add_(1.0)
        x.mul_(0.5).sub_(rank.log_().mul_(1.1))
    else:
        x.mul_(2.5)
    if end_id is not None:
        x[:, end_id] = -20.0
    return x.to(fa.torch_dtype(_TYPES[case["dtype"]]))


def _words(rng, batch, vocab, words, longest):
    """word lists [batch, 2, words * longest]: ids one after the other, then where each word ends (-1: no more)"""
    lists = np.zeros((batch, 2, words * longest), np.int32)
    lists[:, 1] = -1
    for row in lists:
        lengths = rng.integers(1, longest + 1, words)
        ends = np.cumsum(lengths)
        row[0, :ends[-1]] = rng.integers(1, vocab, ends[-1])
        row[1, :words] = ends
    return torch.from_numpy(lists).cuda()


def _prepare_step(case, seed):
    gen, rng = _generator(seed), np.random.default_rng(seed)
    batch, vocab, pitch, history = case["batch"], case["vocab"], case["pitch"], case["history"]
    end_id = vocab - 1
    logits = _logits(gen, case, batch, end_id).reshape(batch, 1, pitch)
    top_ks = rng.choice(np.array([int(k) for k in case["top_k"].split(",")], np.uint32), batch).astype(np.uint32)

    def per_row(lo, hi):
        return rng.uniform(lo, hi, batch).astype(np.float32)

    args = {"runtime_top_k": top_ks, "runtime_top_p": per_row(case["top_p_lo"], case["top_p_hi"]),
            "temperature": per_row(case["temperature_lo"], case["temperature_hi"]),
            "random_seed": rng.integers(0, 1 << 62, batch).astype(np.uint64)}
    plain = case["temperature_hi"] == case["temperature_lo"] == 1.0
    if case["presence"] or case["frequency"]:
        args["presence_penalty"] = np.array([case["presence"]], np.float32)
        args["frequency_penalty"] = np.array([case["frequency"]], np.float32)
        plain = False
    elif case["repetition_hi"] != 1.0:
        args["repetition_penalty"] = per_row(case["repetition_lo"], case["repetition_hi"])
        plain = False
    if case["min_length"]:
        args["min_length"] = np.array([case["min_length"]], np.int32)
    if case["top_p_decay"] != 1.0:
        args["top_p_decay"] = torch.full((batch,), case["top_p_decay"], device="cuda")
        args["top_p_min"] = torch.full((batch,), 0.3, device="cuda")
        args["top_p_reset_ids"] = torch.full((batch,), 13, dtype=torch.int32, device="cuda")
    layer = fa.DynamicDecodeLayer(_TYPES[case["dtype"]], vocab, pitch)
    layer.setup(batch, 1, args)

    output_ids = torch.zeros((history + 2, batch), dtype=torch.int32, device="cuda")
    tokens = np.minimum(rng.zipf(1.2, (history, batch)), vocab - 2).astype(np.int32)
    output_ids[:history] = torch.from_numpy(tokens).cuda()
    outputs = {"output_ids": output_ids, "finished": torch.zeros(batch, dtype=torch.bool, device="cuda"),
               "sequence_length": torch.full((batch,), history - 1, dtype=torch.int32, device="cuda")}
    inputs = {"logits": logits, "step": np.array([history], np.int32), "max_input_length": np.array([history], np.int32),
              "ite": np.array([0], np.uint32), "local_batch_size": np.array([batch], np.int32),
              "end_id": torch.full((batch,), end_id, dtype=torch.int32, device="cuda")}
    if case["log_probs"]:
        outputs["cum_log_probs"] = torch.zeros(batch, device="cuda")
        outputs["output_log_probs"] = torch.zeros((2, batch), device="cuda")
    if case["length_limit"]:
        inputs["sequence_limit_length"] = torch.full((batch,), history + 4096, dtype=torch.int32, device="cuda")
        outputs["should_stop"] = np.zeros(1, np.bool_)
    if case["bad_words"]:
        inputs["bad_words_list"] = _words(rng, batch, vocab, case["bad_words"], 4)
    if case["stop_words"]:
        inputs["stop_words_list"] = _words(rng, batch, vocab, case["stop_words"], 3)
        outputs["parent_ids"] = torch.zeros(1, dtype=torch.int32, device="cuda")
    # A step may leave its penalties in the logits (windows of nucleus rows, and the frequency penalty), so there the
    # logits are written anew before each step, as the model's last projection does.
    projected = None
    if not plain and (not top_ks.any() or case["frequency"]):
        projected = logits.clone()
    return dict(case=case, layer=layer, inputs=inputs, outputs=outputs, projected=projected)


def _run_step(state):
    if state["projected"] is not None:
        state["inputs"]["logits"].copy_(state["projected"])
    state["layer"].forward(state["outputs"], state["inputs"])
    return {name: value for name, value in state["outputs"].items() if name != "parent_ids"}


def _prepare_beam(case, seed):
    gen, rng = _generator(seed), np.random.default_rng(seed)
    batch, beams, vocab, steps = case["batch"], case["beams"], case["vocab"], case["steps"]
    rows, prompt, dtype = batch * beams, 1, _TYPES[case["dtype"]]
    length = prompt + steps
    end_ids = torch.from_numpy(rng.integers(0, vocab, batch).astype(np.int32)).cuda()
    logits = []
    for _ in range(steps):
        x = _logits(gen, case, rows, None)
        ending = torch.rand(rows, generator=gen, device="cuda") < 0.1   # some beams are about to end
        at = torch.arange(rows, device="cuda")
        x[at[ending], end_ids.repeat_interleave(beams).long()[ending]] = 12.0
        logits.append(x.reshape(batch, beams, vocab))

    def zeros(*shape, dtype=torch.float32):
        return torch.zeros(shape, dtype=dtype, device="cuda")

    first = torch.from_numpy(rng.integers(0, vocab, rows).astype(np.int32)).cuda()
    hypotheses = {"output_ids_tgt": zeros(batch, 2 * beams, length, dtype=torch.int32),
                  "sequence_lengths_tgt": zeros(batch, 2 * beams, dtype=torch.int32),
                  "cum_log_probs": zeros(batch, 2 * beams), "normed_scores": zeros(batch, 2 * beams),
                  "log_probs": zeros(batch, 2 * beams, length), "min_normed_scores": zeros(batch),
                  "num_beams": zeros(batch, dtype=torch.int32), "is_done": zeros(batch, dtype=torch.bool)}
    packed = ops.BeamHypotheses()
    for name, tensor in hypotheses.items():
        setattr(packed, name, tensor.data_ptr())
    packed.early_stopping, packed.is_return_normed_score = True, True
    outputs = {"output_ids": zeros(length, batch, beams, dtype=torch.int32),
               "parent_ids": zeros(length, batch, beams, dtype=torch.int32), "finished": zeros(rows, dtype=torch.bool),
               "sequence_length": zeros(rows, dtype=torch.int32), "cum_log_probs": zeros(rows),
               "output_log_probs": zeros(length, batch, beams), "beam_hyps": np.frombuffer(packed, np.uint8)}
    caches = [zeros(batch, beams, length, dtype=torch.int32), zeros(batch, beams, length, dtype=torch.int32)]
    inputs = {"max_input_length": np.array([prompt], np.int32), "ite": np.array([0], np.uint32),
              "local_batch_size": np.array([batch], np.int32), "end_id": end_ids,
              "len_penalty": np.array([0.6], np.float32), "beam_search_diversity_rate": np.array([0.0], np.float32)}
    # one dictionary of inputs and one of outputs per step, as a decode loop fills them
    per_step = []
    for i in range(steps):
        ins = dict(inputs, logits=logits[i], step=np.array([prompt + i], np.int32), src_cache_indirection=caches[i % 2])
        per_step.append((ins, dict(outputs, tgt_cache_indirection=caches[1 - i % 2])))
    best = {"output_ids": zeros(batch, beams, length - 1, dtype=torch.int32),
            "sequence_lengths": zeros(batch, beams, dtype=torch.int32), "cum_log_probs": zeros(batch, beams),
            "output_log_probs": zeros(batch, beams, length - 1)}
    layer = fa.DynamicDecodeLayer(dtype, vocab, vocab)
    layer.setup(batch, beams, {"len_penalty": np.array([0.6], np.float32)})
    return dict(case=case, layer=layer, per_step=per_step, outputs=outputs, hypotheses=hypotheses, packed=packed,
                first=first, caches=caches, best=best, prompt=prompt, length=length)


def _run_beam(state):
    case, out, hyps, best, lib = state["case"], state["outputs"], state["hypotheses"], state["best"], fa.ftk()
    batch, beams, stream = case["batch"], case["beams"], ops.current_stream()
    ops.check(lib.ftk_invoke_decoding_initialize(
        fa.F32, out["finished"].data_ptr(), out["sequence_length"].data_ptr(), out["output_ids"].data_ptr(),
        out["cum_log_probs"].data_ptr(), state["first"].data_ptr(), batch, beams, state["prompt"], stream))
    hyps["num_beams"].zero_()
    hyps["is_done"].zero_()
    for inputs, outputs in state["per_step"]:
        state["layer"].forward(outputs, inputs)
    ops.check(lib.ftk_invoke_finalize(
        best["output_ids"].data_ptr(), best["sequence_lengths"].data_ptr(), best["cum_log_probs"].data_ptr(),
        best["output_log_probs"].data_ptr(), hyps["output_ids_tgt"].data_ptr(),
        hyps["sequence_lengths_tgt"].data_ptr(), hyps["normed_scores"].data_ptr(), hyps["cum_log_probs"].data_ptr(),
        hyps["log_probs"].data_ptr(), hyps["num_beams"].data_ptr(), beams, state["length"] - 1, batch, stream))
    return {"best": best, "output_ids": out["output_ids"], "parent_ids": out["parent_ids"],
            "finished": out["finished"], "sequence_length": out["sequence_length"],
            "cum_log_probs": out["cum_log_probs"], "output_log_probs": out["output_log_probs"],
            "num_beams": hyps["num_beams"], "normed_scores": hyps["normed_scores"], "caches": state["caches"]}


def _prepare_score(case, seed):
    gen, rng = _generator(seed), np.random.default_rng(seed)
    batch, length, vocab = case["batch"], case["length"], case["vocab"]
    logits = torch.stack([_logits(gen, case, batch, None) for _ in range(length)])
    ids = torch.from_numpy(rng.integers(0, vocab, (length, batch)).astype(np.int32)).cuda()
    lengths = rng.integers(max(1, length // 2), length + 1, batch).astype(np.int32)
    lengths[0] = length
    return dict(case=case, logits=logits, ids=ids, lengths=torch.from_numpy(lengths).cuda(),
                result=torch.zeros(batch, device="cuda"), workspace=torch.zeros(length * batch, device="cuda"))


def _run_score(state):
    case, workspace = state["case"], state["workspace"]
    ops.check(fa.ftk().ftk_invoke_log_prob_from_logits(
        _TYPES[case["dtype"]], state["result"].data_ptr(), state["logits"].data_ptr(), state["ids"].data_ptr(),
        state["lengths"].data_ptr(), case["length"], case["batch"], case["vocab"], case["pitch"],
        workspace.data_ptr(), workspace.numel() * 4, ops.current_stream(), False))
    return state["result"]


def prepare(case, seed):
    return {"step": _prepare_step, "beam": _prepare_beam, "score": _prepare_score}[case["kind"]](case, seed)


def run(state):
    return {"step": _run_step, "beam": _run_beam, "score": _run_score}[state["case"]["kind"]](state)


def work(case):
    """every logit read once, the token history where a penalty follows it, and a few words per row; the operations
    are one comparison per logit and, where the whole row is summed, an exponential's worth of arithmetic"""
    width, vocab = _WIDTH[case["dtype"]], case["vocab"]
    if case["kind"] == "beam":
        values = case["batch"] * case["beams"] * vocab * case["steps"]
        return {"bytes": values * width, "flops": 10 * values}
    if case["kind"] == "score":
        # (on average a quarter of the positions lies behind the end of a prompt)
        values = int(0.75 * case["batch"] * case["length"]) * vocab
        return {"bytes": values * width, "flops": 10 * values}
    values = case["batch"] * vocab
    penalised = case["repetition_hi"] != 1.0 or case["presence"] or case["frequency"]
    summed = case["log_probs"] or "0" in case["top_k"].split(",")
    return {"bytes": values * width + (case["batch"] * case["history"] * 4 if penalised else 0) + 64 * case["batch"],
            "flops": (10 if summed else 1) * values}


def tolerance(case):
    """Token ids, lengths and flags are whole numbers that every implementation agrees on. Log-probs carry the rounding
    of a 32-bit sum (against sums in 64 bits: 5e-8) and, where the step rounds logits and probabilities to a 16-bit
    type, of that type (f16: 5e-4, bf16: 1.2e-3)."""
    if case["kind"] == "score":
        return {"rel": 1e-6, "max": 1e-5}
    if case["kind"] == "step" and not case["log_probs"]:
        return "exact"
    return {"f32": {"rel": 1e-6, "max": 1e-5}, "f16": {"rel": 2e-3, "max": 5e-3},
            "bf16": {"rel": 5e-3, "max": 1e-2}}[case["dtype"]]
