"""The fused top-k step with log-probs has several launch forms (csrc/ftk_logprob.cuh): row maxima and rows in two
launches, or one launch with 1024, 512 or 256 threads per row, of which short rows have one of their own. All of them add the row's exponentials in the
reference's order (src/fastertransformer/kernels/sampling_topp_kernels.cu:1308-1344: thread t of 1024 adds columns
t, t + 1024, ... one after the other, then butterflies), so ids, lengths, finished flags and both log-prob outputs
must agree bit for bit between the forms, whatever the batch; parity of the product's own choice with the oracle is
what the layer tests check. The test build of the library selects the form."""
import numpy as np
import pytest

import ft_oracle as O
from helpers import DTYPE_NAMES

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(600)]

FORMS = (1, 1024, 512, 256, -1024, -512, -256)  # ftk_test_set_lp_form


def _case(torch, dt, B, V, Vp, H, k, seed, kind):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    tdt = {O.F32: torch.float32, O.F16: torch.float16, O.BF16: torch.bfloat16}[dt]
    x = torch.randn((B, Vp), generator=gen, device="cuda") * 2.5
    if kind == "grid":  # a coarse grid: many equal values around the k-th largest
        x = torch.round(x * 2.0) / 2.0
    elif kind == "flat":  # constant rows with a few larger columns, some rows with a NaN or an infinity
        x[:] = 0.25
        x[:, ::211] = 1.5
        x[1, 5] = float("nan")
        x[2, 7] = float("inf")
        x[3, :] = float("-inf")
        x[3, 11] = 0.0
    elif kind == "far":  # columns up to a hundred below the maximum, and masked ones of three kinds
        x *= 4.0
        masks = torch.rand((B, Vp), generator=gen, device="cuda") < 0.03
        lows = torch.tensor([float("-inf"), -1e4, -O.max_t(dt), -60.0], device="cuda")
        x = torch.where(masks, lows[torch.arange(B, device="cuda") % 4][:, None], x)
        x[:, 3 * Vp // 4:] -= 25.0
    history = torch.randint(0, V, (H, B), generator=gen, device="cuda", dtype=torch.int32)
    if kind == "edges":  # the largest values in the row's first and last columns, all of them in the history
        x[:, :8] += 20.0
        x[:, V - 8:V] += 20.0
        history[0:8] = torch.arange(8, dtype=torch.int32, device="cuda")[:, None]
        history[8:16] = torch.arange(V - 8, V, dtype=torch.int32, device="cuda")[:, None]
    logits = x.to(tdt)
    draws = torch.rand(B, generator=gen, device="cuda").clamp_(min=1e-6)
    finished0 = torch.zeros(B, dtype=torch.bool, device="cuda")
    finished0[B // 3] = True
    seqlen0 = torch.full((B,), H - 1, dtype=torch.int32, device="cuda")
    return logits, history, draws, finished0, seqlen0


CASES = [
    (O.F32, 40, 50257, 50257, 64, 40, "normal"),    # rows at every 4-byte offset of a 16-byte vector
    (O.F16, 300, 32000, 32004, 300, 50, "normal"),  # padded rows, more rows than compute units
    (O.BF16, 24, 9001, 9001, 16, 128, "grid"),      # one whole batch of columns per thread and a ragged rest
    (O.F32, 9, 1024, 1024, 8, 7, "normal"),         # the shortest row the step takes
    (O.F32, 12, 8192, 8192, 8, 33, "grid"),         # exactly one batch, nothing behind it
    (O.F16, 16, 16500, 16504, 2000, 64, "normal"),  # a long history
    (O.F32, 8, 30011, 30011, 32, 20, "flat"),       # rows the candidates' bound cannot separate, NaN, infinities
    (O.F16, 520, 152064, 152064, 64, 64, "normal"),  # two rounds of 512-thread workgroups
    (O.BF16, 13, 1024, 1027, 16, 8, "edges"),       # rows off 16-byte boundaries whose maxima lie in the columns in
    (O.F32, 11, 4999, 5001, 16, 30, "edges"),       # front of the first whole vector and behind the last
    (O.F16, 19, 33001, 33003, 16, 64, "edges"),
    (O.BF16, 12, 50257, 50257, 16, 40, "far"),
    (O.BF16, 12, 9001, 9001, 16, 40, "far"),        # less than one batch of columns per thread
    (O.BF16, 300, 33001, 33002, 16, 20, "far"),
    (O.F16, 12, 50257, 50257, 16, 40, "far"),
]


@pytest.mark.parametrize("dt,B,V,Vp,H,k,kind", CASES,
                         ids=["%s-%dx%d-%s" % (DTYPE_NAMES[c[0]], c[1], c[2], c[6]) for c in CASES])
def test_forms_of_the_log_prob_step_agree_bit_for_bit(dt, B, V, Vp, H, k, kind):
    import torch
    from fastertransformer_amd import ops
    from helpers import run_fused_step
    hooks = ops.ftk_hooks()
    logits, history, draws, finished0, seqlen0 = _case(torch, dt, B, V, Vp, H, k, 1000 + B + V, kind)
    cum0 = np.linspace(-3.0, 0.0, B).astype(np.float32)
    results = {}
    try:
        for form in FORMS:
            hooks.ftk_test_set_lp_form(form)
            lp = {"cum": cum0.copy()}
            out = run_fused_step("caller", torch, dt, B, V, H, k, logits, history, draws, finished0, seqlen0,
                                 lib=hooks, log_probs=lp, Vp=Vp)
            assert out[3] == 0 and hooks.ftk_test_last_fused_path() == 4
            results[form] = (out[0], out[1], out[2], lp["cum"].view(np.uint32), lp["out"].view(np.uint32))
    finally:
        hooks.ftk_test_set_lp_form(0)
    ref = results[FORMS[0]]
    assert ((ref[0] >= 0) & (ref[0] < V)).all()
    live = ~finished0.cpu().numpy()
    assert (ref[3][live] != cum0.view(np.uint32)[live]).any()  # log-probs were written
    for form in FORMS[1:]:
        for name, a, b in zip(("ids", "sequence_length", "finished", "cum_log_probs", "output_log_probs"), ref,
                              results[form]):
            assert np.array_equal(a, b), "%s differ between the two-launch form and form %d" % (name, form)


RAISING = [
    (O.F16, 300, 33001, 33003, 600, 50, 0.7),   # a penalty that raises: columns of the history reach the bound from below
    (O.F32, 9, 4999, 5001, 30, 30, 0.6),
    (O.BF16, 5, 170000, 170000, 16, 64, 0.8),   # the history's bitmaps in memory; groups of sixteen vectors
    (O.F16, 7, 20000, 20000, 5000, 40, 1.5),    # every fourth column or so in the history, more ids than threads hold
]


@pytest.mark.parametrize("dt,B,V,Vp,H,k,penalty", RAISING,
                         ids=["%s-%dx%d-%g" % (DTYPE_NAMES[c[0]], c[1], c[2], c[6]) for c in RAISING])
def test_forms_agree_whatever_the_penalty_does_to_the_largest_values(dt, B, V, Vp, H, k, penalty):
    """The one-launch form takes a row's maximum from raw values and corrects it for the columns of the history."""
    import torch
    from fastertransformer_amd import ops
    from helpers import run_fused_step
    hooks = ops.ftk_hooks()
    logits, history, draws, finished0, seqlen0 = _case(torch, dt, B, V, Vp, H, k, 77 + V, "normal")
    order = logits[:, :V].float().argsort(dim=1, descending=True)
    history[:H // 2] = order[:, 1::3][:, :H // 2].t().int()  # among the largest, but not all of them
    history[0, ::2] = order[::2, 0].int()                    # and in every other row the largest itself
    results = {}
    try:
        for form in FORMS:
            hooks.ftk_test_set_lp_form(form)
            lp = {}
            out = run_fused_step("caller", torch, dt, B, V, H, k, logits, history, draws, finished0, seqlen0,
                                 lib=hooks, log_probs=lp, Vp=Vp, penalty=penalty)
            assert out[3] == 0 and hooks.ftk_test_last_fused_path() == 4
            results[form] = (out[0], out[1], out[2], lp["cum"].view(np.uint32), lp["out"].view(np.uint32))
    finally:
        hooks.ftk_test_set_lp_form(0)
    for form in FORMS[1:]:
        for a, b in zip(results[FORMS[0]], results[form]):
            assert np.array_equal(a, b), "form %d" % form


PEAKED = [
    (O.F16, 6, 9001, 9001, 64, "sharp"),    # k-th probability below binary16's normal range
    (O.F16, 4, 9001, 9008, 128, "sharper"),  # ... below its smallest number: zeros are picked, pads among them
    (O.F16, 5, 5003, 5003, 40, "plateau"),  # small probabilities in long runs of ties under a large denominator
    (O.F32, 4, 5003, 5008, 16, "level"),    # nothing but ties; the short first stage (thread numbers below 128)
    (O.BF16, 4, 3001, 3001, 128, "level"),
    (O.F32, 4, 2050, 2056, 128, "alone"),   # one column, every other probability exactly zero
    (O.BF16, 4, 2050, 2050, 100, "few"),    # fewer numbers than k
    (O.F16, 4, 40003, 40003, 64, "sharp"),  # the same in rows that are not short
    (O.F16, 4, 40003, 40008, 128, "sharper"),
    (O.F16, 4, 40003, 40003, 40, "plateau"),
    (O.F32, 3, 20483, 20488, 16, "level"),
    (O.BF16, 3, 40003, 40003, 128, "level"),
    (O.F32, 4, 20050, 20056, 128, "alone"),
    (O.BF16, 4, 40050, 40050, 100, "few"),
]


@pytest.mark.parametrize("dt,B,V,Vp,k,kind", PEAKED, ids=["%s-%d-%s" % (DTYPE_NAMES[c[0]], c[2], c[5]) for c in PEAKED])
def test_rows_whose_candidates_are_gathered_again(dt, B, V, Vp, k, kind):
    """Rows that one bound on e cannot settle: ids and log-probs of the oracle's full sequence."""
    from decode_harness import Case, OracleRunner, ProductRunner, compare
    from helpers import uniforms
    rng = np.random.default_rng(len(kind) * 1000 + V)
    H = 12
    c = Case(dt, B, V, Vp, max_input_length=H, gen_len=2, runtime_top_k=[k], runtime_top_p=[1.0], temperature=[0.9],
             repetition_penalty=[1.2], prompt=rng.integers(0, V, (H, B)).astype(np.int32), with_cum=True,
             with_out_lp=True)
    p, o = ProductRunner(c), OracleRunner(c)
    for i in range(2):
        x = rng.standard_normal((B, Vp)).astype(np.float32)
        if kind == "sharp":
            x *= 6.0
            x[:, 17] = 28.0
        elif kind == "sharper":
            x[:, 17] = 40.0
        elif kind == "plateau":
            x = np.round(x * 2.0) / 2.0
            x[:, 100:160] = 14.0
        elif kind == "level":
            x[:] = 0.5
            x[:, 7::701] = 0.75
        elif kind == "alone":
            x[:] = -300.0
            x[:, 1234] = 5.0
        else:
            x[:] = -np.inf
            x[:, ::97] = 1.0
        x = O.to_storage(x, dt)
        u = uniforms(rng, B)
        p.step(H + i, x, u)
        o.step(H + i, x, u)
        compare(p.snapshot(), o.snapshot(), dt, check_logits=False, where="%s step %d" % (kind, i))


@pytest.mark.parametrize("dt", [O.F32, O.F16, O.BF16], ids=lambda d: DTYPE_NAMES[d])
@pytest.mark.parametrize("B,V,Vp,k", [(6, 1452, 1459, 5), (300, 1030, 1040, 20), (5, 2100, 3200, 130), (4, 9001, 9008, 8),
                                      (6, 40001, 40009, 5), (300, 13001, 13013, 20)])
def test_masked_rows_count_their_pads(dt, B, V, Vp, k):
    """Rows masked throughout, with -inf or the type's lowest number: the pad columns hold -MAX_T and carry the softmax."""
    from decode_harness import Case, OracleRunner, ProductRunner, compare
    from helpers import uniforms
    rng = np.random.default_rng(V + dt)
    H = 4
    c = Case(dt, B, V, Vp, max_input_length=H, gen_len=2, runtime_top_k=[k], runtime_top_p=[1.0],
             end_ids=np.full(B, V - 1), prompt=rng.integers(0, V, (H, B)).astype(np.int32), with_cum=True,
             with_out_lp=True)
    p, o = ProductRunner(c), OracleRunner(c)
    for i in range(2):
        x = rng.standard_normal((B, Vp)).astype(np.float32)
        x[0] = -np.inf
        x[1] = -O.max_t(dt)
        x[2], x[2, rng.integers(0, V, 3)] = -np.inf, -O.max_t(dt)
        x[3], x[3, rng.integers(0, V, V // 2)] = -O.max_t(dt), -np.inf
        x, u = O.to_storage(x, dt), uniforms(rng, B)
        print("masked rows", DTYPE_NAMES[dt], B, V, Vp, k, i, flush=True)
        p.step(H + i, x, u)
        o.step(H + i, x, u)
        compare(p.snapshot(), o.snapshot(), dt, check_logits=False, where="step %d" % i)


@pytest.mark.parametrize("dt", [O.F32, O.F16, O.BF16], ids=lambda d: DTYPE_NAMES[d])
@pytest.mark.parametrize("B,V,Vp,k", [(8, 1452, 1459, 5), (8, 9001, 9001, 30), (264, 1030, 1041, 20), (1032, 1100, 1101, 8),
                                      (8, 40001, 40003, 30), (264, 13001, 13008, 20), (1032, 4101, 4101, 8)])
def test_masked_end_ids_count_in_masked_rows(dt, B, V, Vp, k):
    """Below the minimum length the end id has the type's lowest number, also where its logit is -inf or NaN: in rows without
    anything larger it is one of the largest. Short rows and others, with 1024, 512 and 256 threads per row; end ids in the
    whole vectors of a row and in front of and behind them."""
    from decode_harness import Case, OracleRunner, ProductRunner, compare
    from helpers import uniforms
    rng = np.random.default_rng(V + dt)
    H = 4
    ends = np.where(np.arange(B) % 4 == 3, rng.integers(0, V, B), np.array([0, V - 1, V // 2])[np.arange(B) % 3])
    c = Case(dt, B, V, Vp, max_input_length=H, gen_len=3, runtime_top_k=[k], runtime_top_p=[1.0], min_length=[100],
             end_ids=ends, prompt=rng.integers(0, V, (H, B)).astype(np.int32), with_cum=True, with_out_lp=True)
    p, o = ProductRunner(c), OracleRunner(c)
    rows = np.arange(B)
    for i in range(3):
        x = np.full((B, Vp), -np.inf, np.float32)
        for r in rows:
            some = V // 2 if r % 2 == 0 else 8 * k
            x[r, rng.integers(0, V, some)] = -O.max_t(dt)
        x[rows % 5 == 4] = rng.standard_normal((1, Vp))     # ordinary rows among them
        x[rows, ends] = (-np.inf, np.nan, 3.0)[i]
        x, u = O.to_storage(x, dt), uniforms(rng, B)
        u[rows % 3 == 0] = 0.999                            # (the order of ties puts late columns first or last)
        print("masked end ids", DTYPE_NAMES[dt], B, V, Vp, k, i, flush=True)
        p.step(H + i, x, u)
        o.step(H + i, x, u)
        compare(p.snapshot(), o.snapshot(), dt, check_logits=False, where="step %d" % i)
