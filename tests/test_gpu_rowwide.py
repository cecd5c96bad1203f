"""The one-launch steps (a 1024-thread workgroup per row: csrc/ftk_rowwide.cuh, k <= 192, up to 256 rows, or up to 1023
in nearly full rounds of 256 with rows of at least 16384 16-byte vectors; csrc/ftk_largek.cuh, larger k; no bias, no
log-probs) against the CPU oracle, through DynamicDecodeLayer with injected draws: ids / finished / sequence_length
bit-exact. Where the test build of the library is asked which kernel a launch took, that kernel is compared with
the launches it replaces. The last tests are of selections that the log-prob step shares."""
import numpy as np
import pytest

import ft_oracle as O
from decode_harness import Case, OracleRunner, ProductRunner, compare
from helpers import DTYPES, DTYPE_NAMES, uniforms

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(900)]


def _normal(rng, dt, B, Vp, sigma):
    return O.to_storage(rng.standard_normal((B, Vp), dtype=np.float32) * np.float32(sigma), dt)


def _run(c, rng, steps, logits_fn):
    p, o = ProductRunner(c), OracleRunner(c)
    for i in range(steps):
        step = c.max_input_length + i
        logits = logits_fn(i)
        u = uniforms(rng, c.batch)
        p.step(step, logits, u)
        o.step(step, logits, u)
        compare(p.snapshot(), o.snapshot(), c.dt, False, where="step %d" % step)
    return p.snapshot()


@pytest.mark.parametrize("dt", DTYPES, ids=lambda d: DTYPE_NAMES[d])
def test_rowwide_mixed_rows(dt):
    """Per-row k from 1 to 192, per-row top_p and temperature, a repetition penalty that lowers values in some rows
    and raises them in others (below 1), padded vocabulary, min_length masking the end id, rows that finish on the
    way; two steps."""
    rng = np.random.default_rng(300 + dt)
    B = 256
    V, Vp = (70001, 70004) if dt == O.F32 else (131101, 131104)
    H = 48
    ks = rng.choice([1, 2, 7, 40, 64, 100, 192], B).astype(np.uint32)
    pen = rng.choice([0.7, 1.0, 1.1, 1.5], B).astype(np.float32)
    c = Case(dt, B, V, Vp, max_input_length=H, gen_len=2, runtime_top_k=ks, runtime_top_p=rng.uniform(0.3, 1.0, B),
             temperature=rng.uniform(0.5, 1.5, B), repetition_penalty=pen, min_length=[H + 5],
             end_ids=rng.integers(0, V, B).astype(np.int32), prompt=rng.integers(0, V, (H, B)).astype(np.int32))

    def logits_fn(i):
        x = rng.standard_normal((B, Vp), dtype=np.float32) * np.float32(2.5)
        for b in range(0, B, 9):
            x[b, c.end_ids[b]] = 30.0  # the masked end id would win if it were not masked
        return O.to_storage(x, dt)

    _run(c, rng, 2, logits_fn)


def test_rowwide_ties_flat_and_masked_rows():
    """Rows the bound cannot separate: a handful of distinct values (thousands of ties around the k-th: lists longer
    than 256 after the cut, lists that outgrow LDS and are walked again), constant rows, rows that rise towards
    their end (every late column beats what came before), rows where fewer than k columns are valid; presence
    penalty, no temperature."""
    rng = np.random.default_rng(17)
    dt, B, V = O.F32, 256, 66000
    x = rng.standard_normal((B, V), dtype=np.float32) * np.float32(2.0)
    x[0:40] = rng.integers(0, 4, (40, V)).astype(np.float32)                 # four distinct values
    x[40:60] = 1.5                                                            # constant
    x[60:90] = np.sort(x[60:90], axis=1)                                      # ascending
    x[90:110] = -np.inf
    for b in range(90, 110):
        x[b, rng.integers(0, V, 5 + b % 50)] = rng.standard_normal(5 + b % 50)  # fewer valid columns than k
    x[110:130] = np.round(x[110:130] * 4.0) / 4.0                            # a coarse grid: many ties
    H = 20
    c = Case(dt, B, V, V, max_input_length=H, gen_len=1, runtime_top_k=rng.choice([1, 30, 64, 150], B),
             runtime_top_p=[0.95], presence_penalty=[0.4], prompt=rng.integers(0, V, (H, B)).astype(np.int32))
    _run(c, rng, 1, lambda i: x)


def test_rowwide_long_history_and_second_round():
    """512 rows (two full rounds of workgroups), a
    history of 3000 tokens per row with prompt padding skipped, additive penalty that raises (negative)."""
    rng = np.random.default_rng(23)
    dt, B, V, H = O.F32, 512, 65600, 3000
    prompt = np.minimum(rng.zipf(1.2, (H, B)), V - 1).astype(np.int32)
    lengths = rng.integers(H - 500, H + 1, B).astype(np.int32)
    c = Case(dt, B, V, V, max_input_length=H, gen_len=1, runtime_top_k=[50], runtime_top_p=[0.8],
             temperature=[0.9], presence_penalty=[-0.5], input_lengths=lengths, prompt=prompt)
    _run(c, rng, 1, lambda i: _normal(rng, dt, B, V, 2.0))


def test_rowwide_generated_draws_are_reproducible():
    """Without injected draws the kernel takes them from the layer's generator states: the same seed gives the same
    ids, and the states advance (a second step with the same logits differs from the first somewhere)."""
    import torch
    rng = np.random.default_rng(5)
    dt, B, V = O.F32, 256, 65600
    logits = _normal(rng, dt, B, V, 2.0)
    outs = []
    for rep in range(2):
        c = Case(dt, B, V, V, gen_len=2, runtime_top_k=[64], runtime_top_p=[0.9], temperature=[0.8],
                 random_seed=[1234])
        p = ProductRunner(c)
        p.step(0, logits, None)
        p.step(1, logits, None)
        torch.cuda.synchronize()
        outs.append(p.snapshot()["output_ids"].copy())
    assert np.array_equal(outs[0], outs[1])
    assert (outs[0][0] != outs[0][1]).any()
    assert ((outs[0] >= 0) & (outs[0] < V)).all()


def test_rowwide_kernel_is_what_these_shapes_take():
    """the test build of the library reports the path of its last fused step: 3 = one 1024-thread workgroup per row;
    the same rows in two launches (hook) do not take it, nor does a batch between one round of workgroups and a
    nearly full second one (300 rows); any batch of up to 256 rows does; and all agree on the ids"""
    import torch
    from fastertransformer_amd import ops
    from helpers import run_fused_step
    hooks = ops.ftk_hooks()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(9)
    H, k = 16, 64
    for B, V, want in ((256, 65600, 3), (300, 65600, 1), (100, 128256, 3), (100, 32000, 3)):
        logits = torch.randn((B, V), generator=gen, device="cuda") * 2.0
        history = torch.randint(0, V, (H, B), generator=gen, device="cuda", dtype=torch.int32)
        draws = torch.rand(B, generator=gen, device="cuda").clamp_(min=1e-6)
        finished0 = torch.zeros(B, dtype=torch.bool, device="cuda")
        finished0[3] = True
        seqlen0 = torch.full((B,), H - 1, dtype=torch.int32, device="cuda")
        one = run_fused_step("caller", torch, O.F32, B, V, H, k, logits, history, draws, finished0, seqlen0, lib=hooks)
        assert one[3] == 0 and hooks.ftk_test_last_fused_path() == want
        hooks.ftk_test_set_fused_two_launches(1)
        try:
            two = run_fused_step("caller", torch, O.F32, B, V, H, k, logits, history, draws, finished0, seqlen0,
                                 lib=hooks)
            assert two[3] == 0 and hooks.ftk_test_last_fused_path() == 1
        finally:
            hooks.ftk_test_set_fused_two_launches(0)
        for a, b in zip(one[:3], two[:3]):
            assert np.array_equal(a, b)


def test_rowwide_rows_walked_again_do_not_depend_on_the_workspace():
    """Rows whose list outgrows LDS are walked again by the four waves that are left of the workgroup, with the
    history bitmap rebuilt in the workspace: constant rows with a few larger columns, some of them in the history
    (so the penalty decides which win), a workspace full of ones. Same ids as the two-launch step."""
    import torch
    from fastertransformer_amd import ops
    from helpers import run_fused_step
    hooks = ops.ftk_hooks()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(3)
    B, V, H, k = 32, 149544, 300, 150
    logits = torch.full((B, V), 0.75, device="cuda")
    logits[:, ::997] = 1.0
    history = torch.randint(0, V // 997, (H, B), generator=gen, device="cuda", dtype=torch.int32) * 997
    draws = torch.rand(B, generator=gen, device="cuda").clamp_(min=1e-6)
    finished0 = torch.zeros(B, dtype=torch.bool, device="cuda")
    seqlen0 = torch.full((B,), H - 1, dtype=torch.int32, device="cuda")
    one = run_fused_step("caller", torch, O.F32, B, V, H, k, logits, history, draws, finished0, seqlen0, lib=hooks,
                         ws_fill=0xFF)
    assert one[3] == 0 and hooks.ftk_test_last_fused_path() == 3
    hooks.ftk_test_set_fused_two_launches(1)
    try:
        two = run_fused_step("caller", torch, O.F32, B, V, H, k, logits, history, draws, finished0, seqlen0, lib=hooks,
                             ws_fill=0xFF)
    finally:
        hooks.ftk_test_set_fused_two_launches(0)
    for a, b in zip(one[:3], two[:3]):
        assert np.array_equal(a, b)
    assert (one[0] % 997 == 0).all()  # only the larger columns can be sampled (k = 150 of them, all tied)


def test_large_k_lists_in_one_launch_agree_with_the_two_launches():
    """With a largest k beyond 192 one 1024-thread workgroup per row does the step in one launch (csrc/ftk_largek.cuh; path
    5) where the lean gather takes three (maxima, gather, selection); the test build can keep those (path 1). Same ids, lengths and flags on rows of three types:
    vocabularies that end inside a 16-byte vector, histories, rows with fewer valid columns than k, constant rows
    (lists that overflow and send the row to the exact replay)."""
    import torch
    from fastertransformer_amd import ops
    from helpers import run_fused_step
    hooks = ops.ftk_hooks()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(21)
    tdt = {O.F32: torch.float32, O.F16: torch.float16, O.BF16: torch.bfloat16}
    for dt, B, V, Vp, H, k, kind in ((O.F16, 256, 50257, 51200, 64, 1024, "normal"), (O.F32, 130, 50261, 50264, 16, 700, "normal"),
                                     (O.BF16, 100, 32000, 32000, 300, 300, "grid"), (O.F32, 24, 20000, 20000, 8, 1024, "sparse"),
                                     (O.F16, 16, 40000, 40000, 8, 512, "flat")):
        x = torch.randn((B, Vp), generator=gen, device="cuda") * 3.0
        if kind == "grid":
            x = torch.round(x * 2.0) / 2.0
        elif kind == "sparse":  # fewer valid columns than k in some rows
            x[::3] = float("-inf")
            for b in range(0, B, 3):
                cols = torch.randint(0, V, (200,), generator=gen, device="cuda")
                x[b, cols] = torch.randn(200, generator=gen, device="cuda")
        elif kind == "flat":
            x[::2] = 0.5
        logits = x.to(tdt[dt])
        history = torch.randint(0, V, (H, B), generator=gen, device="cuda", dtype=torch.int32)
        draws = torch.rand(B, generator=gen, device="cuda").clamp_(min=1e-6)
        finished0 = torch.zeros(B, dtype=torch.bool, device="cuda")
        finished0[1] = True
        seqlen0 = torch.full((B,), H - 1, dtype=torch.int32, device="cuda")
        one = run_fused_step("caller", torch, dt, B, V, H, k, logits, history, draws, finished0, seqlen0, lib=hooks,
                             Vp=Vp, ws_fill=0xFF)
        assert one[3] == 0 and hooks.ftk_test_last_fused_path() == 5, (dt, B, V)
        hooks.ftk_test_set_largek_two_launches(1)
        try:
            two = run_fused_step("caller", torch, dt, B, V, H, k, logits, history, draws, finished0, seqlen0, lib=hooks,
                                 Vp=Vp, ws_fill=0xFF)
            assert two[3] == 0 and hooks.ftk_test_last_fused_path() == 1
        finally:
            hooks.ftk_test_set_largek_two_launches(0)
        for name, a, b in zip(("ids", "sequence_length", "finished"), one[:3], two[:3]):
            assert np.array_equal(a, b), (name, DTYPE_NAMES[dt], B, V, kind)
        assert ((one[0] >= 0) & (one[0] < V)).all()


@pytest.mark.parametrize("dt", DTYPES, ids=lambda d: DTYPE_NAMES[d])
@pytest.mark.parametrize("B,V,Vp,offset,k", [(3, 1025, 1025, 1, 64), (9, 8193, 8193, 0, 192), (77, 50257, 50257, 3, 50),
                                             (33, 131069, 131071, 1, 40), (24, 152063, 152063, 0, 64), (5, 4097, 4099, 5, 1)])
def test_rowwide_rows_off_the_vector_grid(dt, B, V, Vp, offset, k):
    """Rows that start anywhere: the vectors begin at a row's first 128-byte line. Every row has its largest values in
    the columns in front of that line, behind the last whole vector, in the first and last vectors or anywhere, some
    of them in the history (so the penalty decides). Same ids, lengths and flags as gather and selection."""
    import torch
    from fastertransformer_amd import ops
    from helpers import run_fused_step
    hooks = ops.ftk_hooks()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(31 * V + dt)
    tdt = {O.F32: torch.float32, O.F16: torch.float16, O.BF16: torch.bfloat16}[dt]
    H = 40
    buf = (torch.randn(offset + B * Vp, generator=gen, device="cuda") * 2.0).to(tdt)
    logits = buf[offset:].view(B, Vp)
    history = torch.randint(0, V, (H, B), generator=gen, device="cuda", dtype=torch.int32)
    edges = [0, 1, 5, 20, 62, 63, 64, 65, 72, V - 70, V - 9, V - 8, V - 3, V - 2]
    for b in range(B):
        for i, v in enumerate(edges[b % 3::2] if b % 4 else []):
            logits[b, v] = 9.0 + 0.25 * ((i * 5 + b) % 7)
            if (i + b) % 3 == 0:
                history[i, b] = v
    draws = torch.rand(B, generator=gen, device="cuda").clamp_(min=1e-6)
    finished0 = torch.zeros(B, dtype=torch.bool, device="cuda")
    seqlen0 = torch.full((B,), H - 1, dtype=torch.int32, device="cuda")
    one = run_fused_step("caller", torch, dt, B, V, H, k, logits, history, draws, finished0, seqlen0, lib=hooks, Vp=Vp)
    assert one[3] == 0 and hooks.ftk_test_last_fused_path() == 3
    hooks.ftk_test_set_fused_two_launches(1)
    try:
        two = run_fused_step("caller", torch, dt, B, V, H, k, logits, history, draws, finished0, seqlen0, lib=hooks, Vp=Vp)
        assert two[3] == 0 and hooks.ftk_test_last_fused_path() == 1
    finally:
        hooks.ftk_test_set_fused_two_launches(0)
    for a, b in zip(one[:3], two[:3]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("dt", DTYPES, ids=lambda d: DTYPE_NAMES[d])
@pytest.mark.parametrize("B,V,Vp,k", [(9, 1025, 1025, 64), (40, 9001, 9003, 50), (30, 50257, 50257, 192)])
def test_rows_off_the_vector_grid_in_the_reference_order(dt, B, V, Vp, k):
    """The same kind of rows against the oracle: the largest values in front of a row's first 128-byte line, behind its last whole
    vector, in the vectors beside them or anywhere, some of them equal, some in the history, one of them the masked end id."""
    rng = np.random.default_rng(41 * V + dt)
    H = 40
    x = (rng.standard_normal((B, Vp)) * 2.0).astype(np.float32)
    prompt = rng.integers(0, V, (H, B)).astype(np.int32)
    end_ids = rng.integers(0, V, B).astype(np.int32)
    edges = [0, 1, 5, 20, 31, 32, 62, 63, 64, 65, 72, V - 70, V - 9, V - 8, V - 5, V - 4, V - 3, V - 2, V - 1]
    for b in range(B):
        for i, v in enumerate(edges[b % 3::2] if b % 4 else []):
            x[b, v] = 9.0 + 0.25 * ((i * 5 + b) % 7)
            if (i + b) % 3 == 0:
                prompt[i, b] = v
        end_ids[b] = edges[b % len(edges)]
    x = O.to_storage(x, dt)
    c = Case(dt, B, V, Vp, max_input_length=H, gen_len=1, runtime_top_k=np.resize(np.array([k, 1, k // 2], np.uint32), B),
             runtime_top_p=[0.9], temperature=[0.8], repetition_penalty=[1.15], prompt=prompt, end_ids=end_ids, min_length=[H + 5])
    _run(c, rng, 1, lambda i: x)


@pytest.mark.parametrize("dt,B,V,Vp,offset,H,k,kind", [
    (O.F32, 5, 1161, 1161, 1, 8, 193, "normal"),        # as few vectors as the rule allows
    (O.F16, 9, 12289, 12289, 3, 40, 1024, "normal"),
    (O.BF16, 7, 73729, 73729, 0, 40, 600, "normal"),    # one column more than the registers of a row hold
    (O.F32, 6, 36864, 36864, 0, 40, 1000, "normal"),
    (O.F16, 3, 20001, 20003, 1, 5000, 257, "normal"),   # a history longer than one request
    (O.BF16, 6, 50257, 50257, 1, 40, 1024, "grid"),     # many equal values in a bucket
    (O.F16, 6, 50257, 50257, 0, 40, 700, "few values"),
    (O.F32, 6, 50257, 50257, 0, 40, 500, "one slice"),  # more than k of the best in one of the eight slices
    (O.F32, 6, 50257, 50257, 0, 40, 1024, "outlier"),
    (O.F16, 6, 50257, 50257, 0, 40, 300, "not finite"),
    (O.F16, 300, 16385, 16385, 0, 40, 400, "edges"),
])
def test_large_k_in_one_launch(dt, B, V, Vp, offset, H, k, kind):
    """largek_step_kernel (path 5) against the launches that shapes outside its rule take, whose selection orders slices and
    merges them: every k from 1 on in one batch, rows that start anywhere, values that the buckets of the order separate
    badly or not at all, maxima in the columns outside the vectors, a masked end id."""
    import ctypes as C
    import torch
    from fastertransformer_amd import ops
    hooks = ops.ftk_hooks()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(V + k)
    x = torch.randn(offset + B * Vp, generator=gen, device="cuda") * 2.5
    rows = x[offset:].view(B, Vp)
    if kind == "grid":
        rows.copy_(torch.round(rows * 4.0) / 4.0)
    elif kind == "few values":
        rows[::2] = torch.randint(0, 30, (len(rows[::2]), Vp), generator=gen, device="cuda").float() ** 2 * 0.01
    elif kind == "one slice":
        rows[::2] += 20.0 * ((torch.arange(Vp, device="cuda") // 256) % 8 == 3)
    elif kind == "outlier":
        rows[::2, 777] = 3.0e4
        rows[1::2, 778] = 60.0
    elif kind == "not finite":
        rows[0, ::3] = float("nan")
        rows[1, 5] = float("inf")
        rows[2] = float("-inf")
        rows[3, 200:] = float("-inf")
        rows[4] = -65504.0
    elif kind == "edges":
        for i, v in enumerate([0, 1, 30, 63, 64, V - 65, V - 8, V - 2, V - 1]):
            rows[i % 3::3, v] = 20.0 + i
    logits = x.to({O.F32: torch.float32, O.F16: torch.float16, O.BF16: torch.bfloat16}[dt])
    dev = dict(device="cuda")
    top_ks = torch.randint(1, k + 1, (B,), generator=gen, dtype=torch.int32, **dev)
    top_ks[::2] = k
    history = torch.randint(0, V, (H, B), generator=gen, dtype=torch.int32, **dev)
    draws = torch.rand(B, generator=gen, **dev).clamp_(min=1e-6)
    top_ps, temps, pens = torch.full((B,), 0.97, **dev), torch.full((B,), 0.9, **dev), torch.full((B,), 1.15, **dev)
    end_ids = torch.randint(0, V, (B,), generator=gen, dtype=torch.int32, **dev)
    min_lengths = torch.full((B,), H + 9, dtype=torch.int32, **dev)
    results = []
    for two_launches in (0, 1):
        ids = torch.full((B,), -7, dtype=torch.int32, **dev)
        seq, finished = torch.full((B,), H, dtype=torch.int32, **dev), torch.zeros(B, dtype=torch.bool, **dev)
        finished[1] = B > 5
        a = ops.FusedTopkArgs()
        a.dtype, a.logits, a.embedding_bias = dt, logits.data_ptr() + offset * logits.element_size(), None
        a.vocab_size, a.vocab_size_padded, a.batch_size, a.local_batch_size = V, Vp, B, B
        a.step, a.max_input_length = H, H
        a.temperatures, a.penalties, a.penalty_type = temps.data_ptr(), pens.data_ptr(), ops.PENALTY_MULTIPLICATIVE
        a.end_ids, a.output_ids, a.min_lengths = end_ids.data_ptr(), history.data_ptr(), min_lengths.data_ptr()
        a.top_ks, a.top_ps, a.max_top_k, a.uniform_draws = top_ks.data_ptr(), top_ps.data_ptr(), k, draws.data_ptr()
        a.ids, a.sequence_length, a.finished = ids.data_ptr(), seq.data_ptr(), finished.data_ptr()
        hooks.ftk_test_set_largek_two_launches(two_launches)
        try:
            a.workspace = None
            ops.check(hooks.ftk_fused_topk_step(C.addressof(a), ops.current_stream()))
            ws = torch.full((a.workspace_size,), 0xFF, dtype=torch.uint8, **dev)
            a.workspace = ws.data_ptr()
            ops.check(hooks.ftk_fused_topk_step(C.addressof(a), ops.current_stream()))
            assert (hooks.ftk_test_last_fused_path() == 5) == (two_launches == 0)
        finally:
            hooks.ftk_test_set_largek_two_launches(0)
        torch.cuda.synchronize()
        results.append([v.cpu().numpy() for v in (ids, seq, finished)])
    for a, b in zip(*results):
        assert np.array_equal(a, b)
    assert ((results[0][0] >= 0) & (results[0][0] < V)).all()


@pytest.mark.parametrize("dt", DTYPES, ids=lambda d: DTYPE_NAMES[d])
def test_large_k_in_the_reference_order(dt):
    """largek_step_kernel against the oracle: lists whose buckets are as they should be, that lie in one bucket of the first
    count (fewer valid columns than k, a maximum far ahead, a heap in the middle), with buckets that stay full (equal values)
    and with most candidates in one slice."""
    rng = np.random.default_rng(91 + dt)
    kinds = ["plain", "grid", "one slice", "valid 257", "valid 300", "valid 800", "valid 1000", "ahead 60", "ahead 200", "ahead 30000",
             "heap", "equal 90", "equal 600", "lowest", "both"]
    V, B = 12345, len(kinds)
    x = (rng.standard_normal((B, V)) * 2.5).astype(np.float32)
    for b, kind in enumerate(kinds):
        if kind == "grid":
            x[b] = np.round(x[b] * 4.0) / 4.0
        elif kind == "one slice":
            x[b, (np.arange(V) // 256) % 8 == 3] += 20.0
        elif kind.startswith("valid"):
            x[b, rng.permutation(V)[int(kind[5:]):]] = -np.inf
        elif kind.startswith("ahead"):
            x[b, 777] = float(kind[5:])
        elif kind == "heap":
            x[b, rng.permutation(V)[:700]] = 30.0 + rng.uniform(0.0, 0.01, 700)
            x[b, rng.permutation(V)[:3]] = 300.0
        elif kind.startswith("equal"):
            x[b, rng.permutation(V)[:int(kind[5:])]] = 4.0
        elif kind == "lowest":
            x[b, rng.permutation(V)[500:]] = -65504.0 if dt == O.F16 else -3.3e38
        elif kind == "both":
            x[b, rng.permutation(V)[400:]] = -np.inf
            x[b, :5] = 1.0e4
    x = O.to_storage(x, dt)
    for ks in ([1024], [600], [257, 1024, 40]):
        c = Case(dt, B, V, V, gen_len=1, runtime_top_k=np.resize(np.array(ks, np.uint32), B), runtime_top_p=[0.95], temperature=[0.9])
        _run(c, rng, 1, lambda i: x)
    for k, v in ((193, 1161), (1024, 6151)):  # as few vectors as the rule allows
        if v // (4 if dt == O.F32 else 8) * 2 < 3 * k:
            continue
        c = Case(dt, B, v, v, gen_len=1, runtime_top_k=[k], runtime_top_p=[0.95])
        _run(c, rng, 1, lambda i: np.ascontiguousarray(x[:, :v]))


@pytest.mark.parametrize("dt", DTYPES, ids=lambda d: DTYPE_NAMES[d])
@pytest.mark.parametrize("log_probs", [False, True], ids=["ids", "log_probs"])
def test_short_lists_of_equal_values_in_the_reference_order(dt, log_probs):
    """Lists of 1 to 300 candidates (around the sizes at which the ranking is split differently or gives way to another)
    of a few distinct values, spread over the eight slices or all in one of them, which then keeps k of its entries only."""
    rng = np.random.default_rng(77 + dt)
    sizes = [1, 2, 3, 15, 16, 17, 63, 64, 65, 127, 128, 129, 200, 255, 256, 257, 300]
    B, V = 2 * len(sizes), 17000
    x = np.full((B, V), -np.inf, np.float32)
    for b in range(B):
        n = sizes[b // 2]
        columns = np.arange(V) if b % 2 == 0 else np.flatnonzero((np.arange(V) // 256) % 8 == 3)
        at = rng.choice(columns, n, replace=False)
        x[b, at] = rng.choice([2.0, 2.5, 3.0, 3.25, 6.0], n)
    x = O.to_storage(x, dt)
    for k in (1, 5, 30, 64, 100):
        c = Case(dt, B, V, V, gen_len=1, runtime_top_k=[k], runtime_top_p=[0.95], with_cum=log_probs, with_out_lp=log_probs)
        _run(c, rng, 1, lambda i: x)


@pytest.mark.parametrize("V,Vp", [(4097, 4104), (30011, 30011)])
def test_fp32_rows_of_16_bit_values_with_log_probs(V, Vp):
    """fp32 rows that hold binary16 or bfloat16 values (their lists go straight to the ranking that expects equal values), the
    same with finer values at the row's start or anywhere else, and finer values with equal ones among the candidates."""
    rng = np.random.default_rng(V)
    B = 24
    x = (rng.standard_normal((B, Vp)) * 2.5).astype(np.float32)
    x[::4] = x[::4].astype(np.float16)
    x[1::4] = (x[1::4].view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32)
    x[4, 3] = x[5, 200] = x[8, 5] = x[9, 9] = 0.1
    x[12, 3000] = x[13, 4000] = np.float32(7.1)
    for b in range(2, B, 4):
        x[b, rng.permutation(V)[:200]] = rng.choice(np.array([8.1, 8.3, 9.7], np.float32), 200)
    x[3, :] = np.round(x[3, :])
    x = np.ascontiguousarray(x)
    for ks in ([1], [40], [64, 20, 100, 1]):
        c = Case(O.F32, B, V, Vp, gen_len=1, runtime_top_k=np.resize(np.array(ks, np.uint32), B), runtime_top_p=[0.95],
                 temperature=[0.8], with_cum=True, with_out_lp=True)
        _run(c, rng, 1, lambda i: x)


@pytest.mark.parametrize("dt", DTYPES, ids=lambda d: DTYPE_NAMES[d])
@pytest.mark.parametrize("V,Vp,ks", [(20011, 20011, [50]), (32000, 32000, [16, 1, 7]), (20011, 20016, [181, 64, 192]), (120001, 120001, [192])])
def test_more_equal_columns_than_a_list_holds(dt, V, Vp, ks):
    """Rows whose k-th largest value thousands of columns share, so that the reference's tie orders alone decide: flat rows, fewer
    columns than k above a finite mask, two values, ties in one slice or above k in some of them, negative and zero ties; with a
    history that takes columns out of the tie. (192 of 120001 columns: more than a list holds even so, the literal replay.)"""
    rng = np.random.default_rng(V + dt + ks[0])
    H, kinds = 30, ["flat", "zero", "mask", "mask few", "two", "one slice", "above", "steps"]
    B = len(kinds)
    x = (rng.standard_normal((B, Vp)) * 2.0).astype(np.float32)
    slices = (np.arange(Vp) // (128 if max(ks) <= 16 else 256)) % 8
    for b, kind in enumerate(kinds):
        if kind in ("flat", "zero"):
            x[b] = 0.7 if kind == "flat" else 0.0
        elif kind.startswith("mask"):
            x[b, rng.permutation(Vp)[30 if kind == "mask" else 3:]] = -1.0e4
        elif kind == "two":
            x[b] = np.where(rng.uniform(size=Vp) < 0.4, 3.0, -2.5)
        elif kind == "one slice":
            x[b] = np.where(slices == 5, 1.25, -np.inf)
        elif kind == "above":
            x[b] = 1.0
            x[b, np.flatnonzero(slices == 2)[:max(ks) // 2]] = 4.0
        else:
            x[b] = np.minimum(np.round(x[b]), 1.0)
    x = O.to_storage(x, dt)
    c = Case(dt, B, V, Vp, max_input_length=H, gen_len=2, runtime_top_k=np.resize(np.array(ks, np.uint32), B), runtime_top_p=[0.97],
             temperature=[0.9], repetition_penalty=[1.2], prompt=rng.integers(0, V, (H, B)).astype(np.int32),
             end_ids=np.full(B, V - 1, np.int32), min_length=[H + 9])
    _run(c, rng, 2, lambda i: x)
