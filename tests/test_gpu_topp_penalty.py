"""The top-p step with its penalties folded in (ftk_fused_topp_penalty_step, what the top-p layer takes): edges of the
kernels' tiles and of the rules that split a row, against the oracle's kernel-by-kernel layer. Ids, flags and lengths bit
for bit; log-probs within the harness's tolerance."""
import numpy as np
import pytest

import ft_oracle as O
from decode_harness import Case, OracleRunner, ProductRunner, compare
from helpers import DTYPE_NAMES, DTYPES, make_logits, uniforms

pytestmark = pytest.mark.gpu


def _zipf(rng, dt, B, V, Vp, spread):
    x = -1.1 * np.log(rng.integers(1, V + 1, (B, Vp))) + 0.3 * rng.standard_normal((B, Vp))
    x[rng.random((B, Vp)) < 0.02] = -np.inf          # masked columns
    x[:, 0] += spread                                # a spike far above the rest
    return O.to_storage(x.astype(np.float32), dt)


# (rows, columns, pitch): one stretch of 1024 columns and its neighbours, rows off the 16-byte grid, blocks of 512, both
# sides of the row counts at which a row is split differently
SHAPES = [(3, 1024, 1024), (2, 1025, 1031), (5, 2047, 2048), (2, 8193, 8193), (1, 50257, 50257), (2, 33000, 33008),
          (64, 1536, 1536), (191, 1100, 1101), (192, 1100, 1104), (256, 1030, 1032), (2, 152063, 152064)]


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
