"""GPU: the layered decoder's kernels at the sizes where a variant or a split of the work changes, against the float64 oracle or
a float64 product."""
import pytest

import layered_models as lm
import layered_oracle as lo

pytestmark = pytest.mark.gpu
# bounds of tests/test_gpu_layered.py: root mean square over the vocabulary over the logits' standard deviation
TOL = {"float32": 3e-5, "bfloat16": 4e-2}


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("width,vocab,ff", [
    (70, 98309, 2050),    # one step of a row; two rows per wavefront by N (ff), 256 workgroups (vocab)
    (1700, 2049, 4100),   # bf16 four steps, f32 seven; the smallest N with two rows, the smallest above it with one
    (2200, 12301, 64),    # five and nine steps; two rows by N, four steps of each at a time
    (3600, 40, 900),      # bf16 eight steps
])
def test_decode_linear_splits(width, vocab, ff, dtype):
    cfg = lm.config([lm.attention(4, 2, 24, 24, 16, 4, ff=ff), lm.retention(2, 40, 32, 20)], width=width, vocab=vocab)
    w = lm.random_weights(cfg, seed=width)
    tokens = [7, 3, 11, 39]
    dec = lm.runner(cfg, w, dtype, max_seq=8)
    state = dec.new_state()
    ref = lo.forward(cfg, w, tokens)
    for i, t in enumerate(tokens):
        assert lm.errors(dec.forward(state, [t], i), ref[i:i + 1]).max() < TOL[dtype], i
