"""The top-p step with its penalties folded in (ftk_fused_topp_penalty_step, what the top-p layer takes): edges of the
kernels' tiles and of the rules that split a row, against the oracle's kernel-by-kernel layer. Ids, flags and lengths bit
for bit; log-probs within the harness's tolerance."""
import ctypes as C

import numpy as np
import pytest

import ft_oracle as O
from decode_harness import Case, OracleRunner, ProductRunner, compare, kernel_sequence
from helpers import DTYPE_NAMES, DTYPES, make_logits, to_numpy, to_torch, uniforms

pytestmark = pytest.mark.gpu


def _zipf(rng, dt, B, V, Vp, spread):
    x = -1.1 * np.log(rng.integers(1, V + 1, (B, Vp))) + 0.3 * rng.standard_normal((B, Vp))
    x[rng.random((B, Vp)) < 0.02] = -np.inf          # masked columns
    x[:, 0] += spread                                # a spike far above the rest
    return O.to_storage(x.astype(np.float32), dt)


# (rows, columns, pitch): one stretch of 1024 columns and its neighbours, rows off the 16-byte grid, blocks of 512, both
# sides of the row counts at which a row is split differently
SHAPES = [(3, 1024, 1024), (2, 1025, 1031), (5, 2047, 2048), (2, 8193, 8193), (1, 50257, 50257), (2, 33000, 33008),
          (64, 1536, 1536), (71, 1100, 1101), (72, 1100, 1104), (95, 1100, 1101), (96, 1100, 1104),
          (191, 1100, 1101), (192, 1100, 1104), (256, 1030, 1032), (2, 152063, 152064)]


@pytest.mark.parametrize("dt", DTYPES, ids=lambda d: DTYPE_NAMES[d])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "%dx%d_%d" % s)
def test_penalised_nucleus_rows(dt, shape):
    B, V, Vp = shape
    rng = np.random.default_rng(V + B + dt)
    H = 11
    ks = np.where(rng.random(B) < 0.2, 3, 0).astype(np.uint32)   # a few rows of the other layer among them
    kind = "repetition_penalty" if rng.random() < 0.5 else "presence_penalty"
    c = Case(dt, B, V, Vp, max_input_length=H, gen_len=3, runtime_top_k=ks, runtime_top_p=rng.uniform(0.2, 1.0, B),
             temperature=rng.uniform(0.5, 1.5, B), min_length=rng.integers(0, 3, B), end_ids=rng.integers(0, V, B),
             input_lengths=rng.integers(1, H + 1, B), prompt=rng.integers(0, V, (H, B)).astype(np.int32),
             top_p_decay=rng.uniform(0.5, 1.0, B), top_p_min=rng.uniform(0.1, 0.4, B),
             top_p_reset_ids=rng.integers(0, V, B), with_cum=True, with_out_lp=True, **{kind: rng.uniform(0.5, 1.5, B)})
    p, o = ProductRunner(c), OracleRunner(c)
    for i in range(3):
        print("topp penalty", DTYPE_NAMES[dt], shape, kind, i, flush=True)
        x = (_zipf(rng, dt, B, V, Vp, 30.0 * (i == 1)) if i < 2 else make_logits(rng, dt, B, V, Vp, 2.0))
        u = uniforms(rng, B)
        u[0] = 1.0 if i == 2 else u[0]                # a draw at the very end of the row
        p.step(H + i, x, u)
        o.step(H + i, x, u)
        compare(p.snapshot(), o.snapshot(), dt, check_logits=False, where="step %d" % i)


@pytest.mark.parametrize("dt", DTYPES, ids=lambda d: DTYPE_NAMES[d])
@pytest.mark.parametrize("H", [1, 511, 2049, 4096, 4097, 9000])
def test_long_histories_of_nucleus_rows(dt, H):
    """Histories around the number of ids that a stage requests at once, with vectors whose columns are all in the history,
    the masked end id among them, and ids on both sides of where workgroups share a row out."""
    B, V, Vp = 3, 20011, 20016
    rng = np.random.default_rng(H + dt)
    prompt = rng.integers(0, V, (H, B)).astype(np.int32)
    near = rng.random((H, B)) < 0.5
    prompt[near] = (4090 + rng.integers(0, 24, int(near.sum()))).astype(np.int32)
    c = Case(dt, B, V, Vp, max_input_length=H, gen_len=2, runtime_top_k=np.zeros(B, np.uint32),
             runtime_top_p=rng.uniform(0.5, 1.0, B), temperature=rng.uniform(0.5, 1.5, B), min_length=np.full(B, H + 9),
             end_ids=np.array([4095, V - 1, 4100]), input_lengths=np.array([H, max(1, H // 2), 1]), prompt=prompt,
             repetition_penalty=rng.uniform(0.8, 1.5, B), with_cum=True, with_out_lp=True)
    p, o = ProductRunner(c), OracleRunner(c)
    for i in range(2):
        print("long history", DTYPE_NAMES[dt], H, i, flush=True)
        x = _zipf(rng, dt, B, V, Vp, 0.0)
        u = uniforms(rng, B)
        p.step(H + i, x, u)
        o.step(H + i, x, u)
        compare(p.snapshot(), o.snapshot(), dt, check_logits=False, where="step %d" % i)


def _sample_step(dt, x, V, p_arr, end_ids, draws=None, states=None, gathered=None, finished=None, hooks=False):
    """One ftk_fused_topp_sample_step over rows of `x`: (ids, finished, lengths, cumulative log-probs). The draws are
    `draws`, or generated from `states` (advanced in place). `gathered` (fp32; an int32 array) gets the number of entries
    in each row's ordered prefix."""
    import torch
    from fastertransformer_amd import ops
    lib = ops.ftk_hooks() if hooks or gathered is not None else ops.ftk()
    B, Vp = x.shape
    d_x, d_p, d_end, d_u = to_torch(x, dt), to_torch(p_arr), to_torch(end_ids), to_torch(draws)
    ids = torch.full((B,), -7, dtype=torch.int32, device="cuda")
    fin = torch.zeros(B, dtype=torch.bool, device="cuda") if finished is None else to_torch(finished)
    seq = torch.zeros(B, dtype=torch.int32, device="cuda")
    cum = torch.zeros(B, dtype=torch.float32, device="cuda")
    size = C.c_size_t(0)
    ops.check(lib.ftk_fused_topp_sample_step(dt, None, C.addressof(size), None, V, Vp, B, *(None,) * 8, 1.0, *(None,) * 7))
    ws = torch.empty(size.value, dtype=torch.uint8, device="cuda")
    ops.check(lib.ftk_fused_topp_sample_step(
        dt, ws.data_ptr(), C.addressof(size), d_x.data_ptr(), V, Vp, B, d_end.data_ptr(), fin.data_ptr(), seq.data_ptr(),
        ids.data_ptr(), cum.data_ptr(), None, ops.ptr(states), ops.ptr(d_u), 1.0, d_p.data_ptr(), None, None, None, None,
        None, ops.current_stream()))
    torch.cuda.synchronize()
    if gathered is not None:
        ops.check(lib.ftk_test_topp_prefix_lengths(ws.data_ptr(), B, V, Vp, 0, gathered.ctypes.data))
    return tuple(to_numpy(a) for a in (ids, fin, seq, cum))


def _oracle_step(dt, x, V, p_arr, end_ids, draws, finished=None):
    B, Vp = x.shape
    probs, fin, seq = x.copy(), np.zeros(B, np.bool_) if finished is None else finished.copy(), np.zeros(B, np.int32)
    O.add_bias_softmax(dt, probs, None, end_ids, fin, B, Vp, V)
    ids, cum, out = np.full(B, -7, np.int32), np.zeros(B, np.float32), np.zeros(B, np.float32)
    O.batch_topp_sampling(dt, probs, ids, seq, fin, cum, out, draws, B, Vp, end_ids, 0.0, p_arr, None)
    return ids, fin, seq, cum


def _same(got, want, dt):
    for a, b in zip(got[:3], want[:3]):
        assert np.array_equal(a, b)
    np.testing.assert_allclose(got[3], want[3], rtol=1e-5 if dt == O.F32 else 2e-3, atol=1e-6)


@pytest.mark.parametrize("dt,V,kind", [(O.F16, 20011, "signs"), (O.BF16, 20011, "signs"), (O.F16, 30000, "levels"),
                                       (O.BF16, 70001, "levels"), (O.BF16, 300000, "levels")])
def test_deep_draws_into_long_runs(dt, V, kind):
    """16-bit rows whose draws lie behind whole scan tiles of one value, tiles of many and both in turn, up to more tiles
    than one round of the scan holds; the column that is picked is one of thousands of equal probabilities, whose logits
    may be of both signs."""
    B = 6
    rng = np.random.default_rng(V + len(kind))
    if kind == "signs":  # e is 1 / e^3 for all of them, whatever their sign
        x = (rng.choice([-1.0, 1.0], (B, V)) * 2.0 ** rng.uniform(-22.0, -16.0, (B, V))).astype(np.float32)
        x[:, ::97] = 3.0
    else:
        x = rng.choice(np.array([0.0, -0.25, -0.5, -1.0], np.float32), (B, V))
        some = rng.random((B, V)) < 0.05
        x = np.where(some, rng.standard_normal((B, V)) * 0.5 - 0.5, x).astype(np.float32)
        x[:, :400] = rng.standard_normal((B, 400)) * 1.5 + 1.0
    x = O.to_storage(x, dt)
    p = np.array([1.0, 1.0, 0.97, 0.9, 1.0, 0.6], np.float32)
    draws = np.array([0.05, 0.5, 0.999, 0.7, 0.92, 0.8], np.float32)
    end_ids = np.full(B, -1, np.int32)
    _same(_sample_step(dt, x, V, p, end_ids, draws), _oracle_step(dt, x, V, p, end_ids, draws), dt)


@pytest.mark.parametrize("dt", [O.F16, O.BF16], ids=["f16", "bf16"])
@pytest.mark.parametrize("head", [600, 2048, 2049, 8191, 8193, 16384, 16640])
@pytest.mark.parametrize("V", [20011, 19969])
def test_draws_around_the_end_of_the_short_runs(dt, head, V):
    """16-bit rows of `head` columns of hundreds of values in front of long runs whose probabilities are half a last place
    of the running sum and less: draws on both sides of where the scan's values lie position by position, and picks in the
    last columns, of which 43 or one fill no block."""
    B = 8
    rng = np.random.default_rng(V + head + dt)
    x = np.full((B, V), -6.0, np.float32) + rng.choice(np.array([0.0, 0.03125, 0.0625], np.float32), (B, V))
    for row in x:
        at = rng.permutation(V)[:head]
        row[at] = rng.standard_normal(head) * 1.2 - 0.5
    x[6:, :] = -9.0
    x[6:, -30:] = rng.standard_normal((2, 30))
    x[7, -1] = 5.0
    x = O.to_storage(x, dt)
    p = np.ones(B, np.float32)
    draws = np.array([0.02, 0.6, 0.9, 0.97, 0.995, 0.9999, 0.7, 0.3], np.float32)
    end_ids = np.full(B, -1, np.int32)
    _same(_sample_step(dt, x, V, p, end_ids, draws), _oracle_step(dt, x, V, p, end_ids, draws), dt)


@pytest.mark.parametrize("dt", [O.F16, O.BF16], ids=["f16", "bf16"])
@pytest.mark.parametrize("runs", [[1, 127, 128, 129, 130, 135, 136, 137, 143, 144, 145, 301, 1001], [5000, 5003, 5001], [3, 16379, 9],
                                  [8191, 127, 140], [16384, 1, 133], [129] * 140, [1]], ids=lambda r: "%dx%d" % (len(r), r[0]))
def test_draws_from_long_runs_at_the_head(dt, runs):
    """16-bit rows of few distinct values, whose first runs are around the lengths at which their positions are written by
    different threads, end anywhere in a vector of eight and reach over the end of the array; draws from all over the row."""
    V, B = 20011, 24
    rng = np.random.default_rng(sum(runs) + dt)
    value = np.concatenate([np.full(n, -0.0625 * i) for i, n in enumerate(runs)] + [np.full(V - sum(runs), -0.0625 * len(runs))])
    x = O.to_storage(np.stack([value[rng.permutation(V)] for _ in range(B)]).astype(np.float32), dt)
    p = np.ones(B, np.float32)
    draws = rng.uniform(0.0, 1.0, B).astype(np.float32)
    draws[:4] = [1e-7, 0.9999, 0.01, 0.02]
    end_ids = np.full(B, -1, np.int32)
    _same(_sample_step(dt, x, V, p, end_ids, draws), _oracle_step(dt, x, V, p, end_ids, draws), dt)


@pytest.mark.parametrize("dt", [O.F16, O.BF16], ids=["f16", "bf16"])
@pytest.mark.parametrize("V,Vp", [(9001, 9001), (9001, 9008), (2000, 2003)])
@pytest.mark.parametrize("first", [-0.0, 0.0])
def test_largest_values_are_zeros_of_both_signs(dt, V, Vp, first):
    """The largest value of a row is zero: -0 and +0 have one probability, and a draw picks among all of them."""
    zeros = np.array([0, 100, 513, 1024, V - 1])
    B = len(zeros) + 2
    rng = np.random.default_rng(V + dt)
    x = rng.uniform(-14.0, -11.0, (B, Vp)).astype(np.float32)
    x[:, zeros] = np.where(np.arange(len(zeros)) % 2 == 0, first, -first)
    x[-1, zeros[1:]] = first     # a row of one sign
    x = O.to_storage(x, dt)
    p = np.full(B, 1.0, np.float32)
    draws = np.append((np.arange(len(zeros)) + 0.5) / (len(zeros) + 0.2), [0.02, 0.4]).astype(np.float32)
    end_ids = np.full(B, -1, np.int32)
    want = _oracle_step(dt, x, V, p, end_ids, draws)
    assert set(want[0][:len(zeros)]) == set(zeros)
    _same(_sample_step(dt, x, V, p, end_ids, draws), want, dt)


@pytest.mark.parametrize("B,V", [(24, 20011), (256, 14000)])   # sixteen and four workgroups per row
def test_long_fp32_prefixes(B, V):
    """Draws so deep into flat fp32 rows that the prefix in front of them (most of the row, more than 5632 entries) is
    ordered in segments that the whole launch shares out."""
    rng = np.random.default_rng(B + V)
    x = rng.standard_normal((B, V)).astype(np.float32) * rng.uniform(0.2, 1.0, (B, 1)).astype(np.float32)
    p_arr, end_ids = np.full(B, 1.0, np.float32), rng.integers(0, V, B).astype(np.int32)
    for step in range(2):
        u = rng.uniform(0.8, 0.999, B).astype(np.float32)
        print("long prefixes", B, V, step, flush=True)
        _same(_sample_step(O.F32, x, V, p_arr, end_ids, u), _oracle_step(O.F32, x, V, p_arr, end_ids, u), O.F32)


@pytest.mark.parametrize("dt", DTYPES, ids=lambda d: DTYPE_NAMES[d])
@pytest.mark.parametrize("B,V", [(40, 14000), (300, 2051)])
def test_generated_draws_are_the_injected_ones(dt, B, V):
    """Three steps that draw for themselves from per-row generators against the same draws injected: ids, flags, lengths
    and log-probs bit for bit, and generators that have gone on by one draw a step."""
    import torch
    from fastertransformer_amd import ops
    hooks = ops.ftk_hooks()
    rng = np.random.default_rng(V + dt)
    states = torch.zeros(B * 2, dtype=torch.int64, device="cuda")
    seeds = to_torch(rng.integers(0, 1 << 62, B).astype(np.uint64))
    ops.check(hooks.ftk_invoke_curand_batch_initialize(states.data_ptr(), B, seeds.data_ptr(), ops.current_stream()))
    drawn, ahead = torch.empty(B * 3, dtype=torch.float32, device="cuda"), states.clone()
    ops.check(hooks.ftk_test_rng_uniform(ahead.data_ptr(), drawn.data_ptr(), B, 3, ops.current_stream()))
    torch.cuda.synchronize()
    draws = to_numpy(drawn).reshape(B, 3)
    p_arr, end_ids = rng.uniform(0.3, 1.0, B).astype(np.float32), rng.integers(0, V, B).astype(np.int32)
    for i, spread in enumerate((0.3, 2.0, 8.0)):    # from draws deep into flat rows to one token that is all there is
        x = make_logits(rng, dt, B, V, V, spread)
        print("generated draws", DTYPE_NAMES[dt], B, V, i, flush=True)
        own = _sample_step(dt, x, V, p_arr, end_ids, states=states)
        for a, b in zip(own, _sample_step(dt, x, V, p_arr, end_ids, np.ascontiguousarray(draws[:, i]))):
            assert np.array_equal(a, b)
        assert (to_numpy(states).reshape(B, 2)[:, 1] == i + 1).all()
    assert np.array_equal(to_numpy(states), to_numpy(ahead))


def _prefix_bound(y, draw):
    """The most entries a row's ordered prefix may need. Buckets are 1/64 wide: the sum bounds a prefix's mass from below
    and what lies behind it from above by a factor of e^(1/64) each, and takes two more buckets than the one that covers
    the draw (with the margin of 1/1024 on it). Beyond that, the buckets' open top, 8 above the largest of a sample of
    1024 columns, may hold columns that the sample missed: 200 are allowed for here."""
    y = np.sort(y.astype(np.float64))[::-1]
    mass = np.cumsum(np.exp(y - y[0]))
    behind = np.maximum(mass[-1] - mass, 0.0) + 1e-6
    q = draw * (1 + 1 / 1024)
    if q >= 1:
        return len(y)
    enough = np.nonzero(mass * (1 - q) >= 1.001 * np.exp(2 / 64) * q * behind)[0]
    return len(y) if len(enough) == 0 else int((y >= y[enough[0]] - 4 / 64).sum()) + 200


@pytest.mark.parametrize("kind", ["two_ahead", "five_ahead", "masked_head", "cold", "allowed_few", "peaked"])
@pytest.mark.parametrize("B,V", [(12, 40009), (256, 9001)])   # sixteen and four workgroups per row
def test_fp32_prefix_is_what_the_draw_needs(B, V, kind):
    """Rows whose columns are unlike each other: a few tokens far ahead of all others, an id range masked out, a low
    temperature, nearly everything masked. The prefix that is gathered and ordered follows the draw, not the layout."""
    rng = np.random.default_rng(V + len(kind))
    x = (rng.standard_normal((B, V)) * 2.5).astype(np.float32)
    if kind == "two_ahead":
        x[:, V // 25], x[:, V * 2 // 3] = 20.0, 19.5
    elif kind == "five_ahead":
        x[:, rng.integers(V // 25, V, 5)] = np.float32([20.0, 19.9, 19.8, 19.7, 19.6])
    elif kind == "masked_head":
        x[:, :1024] = -1e4
    elif kind == "cold":
        x *= 10.0
    elif kind == "allowed_few":
        keep = rng.random((B, V)) < 0.01
        x[~keep] = -1e4
        x[:, 5] = 3.0
    else:
        x[:, V // 2:V // 2 + 50] += 12.0
    p_arr, end_ids = np.ones(B, np.float32), rng.integers(0, V, B).astype(np.int32)
    u = rng.uniform(0.05, 0.995, B).astype(np.float32)
    u[:6] = [0.3, 0.6, 0.85, 0.98, 0.99, 0.995]
    got = np.zeros(B, np.int32)
    print("prefix", B, V, kind, flush=True)
    _same(_sample_step(O.F32, x, V, p_arr, end_ids, u, gathered=got), _oracle_step(O.F32, x, V, p_arr, end_ids, u),
          O.F32)
    bound = np.array([_prefix_bound(x[b], float(u[b])) for b in range(B)])
    assert (got >= 1).all() and (got <= bound).all(), (got[got > bound], bound[got > bound])


# (rows of the batch, of a window, columns, pitch): odd columns, padded and odd pitches, both splits of a row
@pytest.mark.parametrize("B,window,V,Vp", [(12, 6, 1501, 1504), (12, 6, 2050, 2051), (6, 6, 33001, 33008),
                                           (200, 100, 1030, 1030), (200, 200, 1025, 1032)])
@pytest.mark.parametrize("dt", DTYPES, ids=lambda d: DTYPE_NAMES[d])
def test_biased_nucleus_rows(dt, B, window, V, Vp):
    """An embedding bias under every other penalty, rows of both layers, windows of the batch; the second step's bias
    masks most columns."""
    rng = np.random.default_rng(V + dt)
    H = 7
    ks = np.where(rng.random(B) < 0.3, 4, 0).astype(np.uint32)
    kind = "repetition_penalty" if V % 2 else "presence_penalty"
    for masks in (False, True):
        bias = rng.standard_normal(Vp).astype(np.float32)
        if masks:
            bias[rng.random(Vp) < 0.9] = -1e4
        c = Case(dt, B, V, Vp, max_input_length=H, gen_len=2, local_batch=window, runtime_top_k=ks,
                 runtime_top_p=rng.uniform(0.2, 1.0, B), temperature=rng.uniform(0.5, 1.5, B),
                 min_length=rng.integers(0, 3, B), end_ids=rng.integers(0, V, B),
                 input_lengths=rng.integers(1, H + 1, B), prompt=rng.integers(0, V, (H, B)).astype(np.int32),
                 embedding_bias=O.to_storage(bias, dt), with_cum=True, with_out_lp=window == B, **{kind: rng.uniform(0.5, 1.5, B)})
        p, o = ProductRunner(c), OracleRunner(c)
        for i in range(2):
            x, u = make_logits(rng, dt, B, V, Vp, 2.0), uniforms(rng, B)
            for ite in range(B // window):
                print("biased", DTYPE_NAMES[dt], B, window, V, Vp, masks, i, ite, flush=True)
                p.step(H + i, x, u, ite=ite)
                o.step(H + i, x, u, ite=ite)
                compare(p.snapshot(), o.snapshot(), dt, check_logits=False, where="step %d window %d" % (i, ite))


@pytest.mark.parametrize("dt", [O.F16, O.BF16], ids=["f16", "bf16"])
@pytest.mark.parametrize("V,Vp,offset", [(1025, 1025, 1), (4103, 4104, 3), (20011, 20011, 0)])
def test_bias_anywhere_in_memory(dt, V, Vp, offset):
    """A bias that starts off the 16-byte grid, under rows whose last vector runs over the end, with a history and a masked
    end id in whole vectors and in that one."""
    import torch
    B, H = 4, 40
    rng = np.random.default_rng(V + dt)
    prompt = rng.integers(0, V, (H, B)).astype(np.int32)
    prompt[:8] = V - 1 - np.arange(8)[:, None]
    c = Case(dt, B, V, Vp, max_input_length=H, gen_len=1, runtime_top_k=np.zeros(B, np.uint32), runtime_top_p=np.full(B, 0.9),
             temperature=rng.uniform(0.5, 1.5, B), min_length=np.full(B, H + 9), end_ids=np.array([V - 1, V - 9, 8, 0]),
             prompt=prompt, embedding_bias=O.to_storage(rng.standard_normal(Vp).astype(np.float32) * 2, dt),
             repetition_penalty=rng.uniform(1.1, 1.5, B), with_cum=True, with_out_lp=True)
    p, o = ProductRunner(c), OracleRunner(c)
    p.bias = torch.cat([torch.zeros(offset, dtype=p.bias.dtype, device="cuda"), p.bias])[offset:]
    x, u = make_logits(rng, dt, B, V, Vp, 2.0), uniforms(rng, B)
    p.step(H, x, u)
    o.step(H, x, u)
    compare(p.snapshot(), o.snapshot(), dt, check_logits=False)


def _penalty_step(dt, x, V, p_arr, end_ids, draws, finished, temps, penalties, history):
    """_sample_step with a temperature and a repetition penalty over `history` [steps, rows]"""
    import torch
    from fastertransformer_amd import ops

    class Args(C.Structure):
        _fields_ = [("row", ops.FusedTopkArgs), ("max_top_p", C.c_float), ("runtime_top_p", C.c_void_p)] + [
            ("decay%d" % i, C.c_void_p) for i in range(4)]

    lib, (B, Vp) = ops.ftk_hooks(), x.shape
    d = dict(logits=to_torch(x, dt), temperatures=to_torch(temps), penalties=to_torch(penalties),
             end_ids=to_torch(end_ids), output_ids=to_torch(history), uniform_draws=to_torch(draws), finished=to_torch(finished),
             ids=torch.full((B,), -7, dtype=torch.int32, device="cuda"),
             sequence_length=torch.zeros(B, dtype=torch.int32, device="cuda"),
             cum_log_probs=torch.zeros(B, dtype=torch.float32, device="cuda"))
    a = Args(row=ops.FusedTopkArgs(dtype=dt, vocab_size=V, vocab_size_padded=Vp, batch_size=B, local_batch_size=B,
                                   step=len(history), max_input_length=len(history), penalty_type=1,
                                   **{k: v.data_ptr() for k, v in d.items()}))
    d["p"] = to_torch(p_arr)
    a.max_top_p, a.runtime_top_p = 1.0, d["p"].data_ptr()
    ops.check(lib.ftk_fused_topp_penalty_step(C.addressof(a), None))
    ws = torch.empty(a.row.workspace_size, dtype=torch.uint8, device="cuda")
    a.row.workspace = ws.data_ptr()
    ops.check(lib.ftk_fused_topp_penalty_step(C.addressof(a), ops.current_stream()))
    torch.cuda.synchronize()
    return tuple(to_numpy(d[k]) for k in ("ids", "finished", "sequence_length", "cum_log_probs"))


@pytest.mark.parametrize("B,V,Vp", [(7, 1027, 1027), (6, 4096, 4104), (200, 1100, 1101)])
@pytest.mark.parametrize("dt", DTYPES, ids=lambda d: DTYPE_NAMES[d])
def test_whole_row_fallback(dt, B, V, Vp):
    """The exact way out of the pick, every row sent there by the test build's switch, and without it: plain and
    penalised rows against the oracle. Among them finished rows with an end id inside and outside of the vocabulary."""
    from fastertransformer_amd import ops
    rng = np.random.default_rng(V + 10 * dt)
    hooks, H = ops.ftk_hooks(), 9
    end_ids = rng.integers(0, V, B).astype(np.int32)
    end_ids[1], end_ids[2], end_ids[3] = Vp + 5, -1, V - 1
    finished = np.zeros(B, np.bool_)
    finished[1:4] = True
    temps, pens = (rng.uniform(0.5, 1.5, B).astype(np.float32) for _ in range(2))
    history = rng.integers(0, V, (H, B)).astype(np.int32)
    for i, spread in enumerate((0.3, 2.0, 8.0)):
        x = make_logits(rng, dt, B, V, Vp, spread)
        p_arr, u = rng.uniform(0.3, 1.0, B).astype(np.float32), uniforms(rng, B)
        u[0], p_arr[0] = 1.0, 1.0
        y = x.copy()
        O.batch_apply_temperature_penalty(dt, y, None, temps, B, V, Vp)
        O.batch_apply_repetition_penalty(dt, y, pens, history, B, B, Vp, None, H, H, 1)
        for deep in (1, 0):
            hooks.ftk_test_set_topp_force_deep(deep)
            try:
                print("whole row", DTYPE_NAMES[dt], B, V, Vp, i, deep, flush=True)
                plain = _sample_step(dt, x, V, p_arr, end_ids, u, finished=finished, hooks=True)
                penalised = _penalty_step(dt, x, V, p_arr, end_ids, u, finished, temps, pens, history)
            finally:
                hooks.ftk_test_set_topp_force_deep(0)
            _same(plain, _oracle_step(dt, x, V, p_arr, end_ids, u, finished), dt)
            _same(penalised, _oracle_step(dt, y, V, p_arr, end_ids, u, finished), dt)


@pytest.mark.parametrize("dt", DTYPES, ids=lambda d: DTYPE_NAMES[d])
@pytest.mark.parametrize("V,Vp,sequence", [(500, 500, False), (333, 336, False), (2050, 2050, True), (2050, 2056, True),
                                           (2050, 2050, False)])
def test_rows_without_an_ordinary_denominator(dt, V, Vp, sequence):
    """Rows with a NaN, with an infinity, all masked and all at the lowest number, without a bias: through the step that
    writes the probabilities (fewer than 1024 columns, or asked for) and through the one that does not."""
    rng = np.random.default_rng(V + dt)
    B, H = 9, 3
    c = Case(dt, B, V, Vp, max_input_length=H, gen_len=2, runtime_top_k=[0], runtime_top_p=rng.uniform(0.2, 1.0, B),
             end_ids=np.full(B, V - 1), prompt=rng.integers(0, V, (H, B)).astype(np.int32), with_cum=True)
    with kernel_sequence(sequence):
        p, o = ProductRunner(c), OracleRunner(c)
        for i in range(2):
            x = rng.standard_normal((B, Vp)).astype(np.float32)
            x[1, rng.integers(0, V)], x[2, rng.integers(0, V)] = np.nan, np.inf
            x[3], x[4], x[5], x[6] = -np.inf, np.nan, O.max_t(dt) * -1.0, 0.0
            x = O.to_storage(x, dt)
            u = uniforms(rng, B)
            print("denominators", DTYPE_NAMES[dt], V, Vp, sequence, i, flush=True)
            p.step(H + i, x, u)
            o.step(H + i, x, u)
            compare(p.snapshot(), o.snapshot(), dt, check_logits=False, where="step %d" % i)


@pytest.mark.parametrize("sequence", [False, True])
@pytest.mark.parametrize("dt", DTYPES, ids=lambda d: DTYPE_NAMES[d])
def test_crossings_behind_the_last_column(dt, sequence):
    """Draws of 1.0: where rounding lets the running sum reach them only among the zeros that fill the last tile, the last
    entry in order of probabilities is emitted."""
    rng = np.random.default_rng(dt)
    B, V = 300, 1526
    x = np.round(rng.standard_normal((B, V)) * 5.0).astype(np.float32) / 2
    x = O.to_storage(x, dt)
    c = Case(dt, B, V, V, gen_len=1, runtime_top_k=[0], runtime_top_p=[1.0])
    with kernel_sequence(sequence):
        p, o = ProductRunner(c), OracleRunner(c)
        print("behind the last column", DTYPE_NAMES[dt], sequence, flush=True)
        p.step(0, x, np.ones(B, np.float32))
        o.step(0, x, np.ones(B, np.float32))
    compare(p.snapshot(), o.snapshot(), dt, check_logits=False)
    if dt == O.F32:
        last = np.argsort(-x, axis=1, kind="stable")[:, -1]
        assert ((o.snapshot()["output_ids"][0] == last) & (last != V - 1)).any()
