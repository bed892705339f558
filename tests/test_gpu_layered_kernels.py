"""GPU: the layered decoder's kernels at the sizes where a variant or a split of the work changes, against the float64 oracle or
a float64 product."""
import numpy as np
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


@pytest.mark.parametrize("H,taps,first,rest", [
    (64, 8, 3, 45),      # more workgroups than one would read the ring if each took a single row
    (1600, 4, 2, 40),
    (330, 4, 1, 3),
    (5100, 8, 9, 20),    # seven rows of halo and seven more do not fit the LDS: rows and tail in two launches
    (5100, 8, 4, 3),     # ... with a tail that keeps older rows
])
def test_norm_conv_leaves_its_tail_when_nobody_reads_the_ring(pkg, H, taps, first, rest):
    import torch

    rng = np.random.default_rng(H + taps)
    T, ld = first + rest + 5, (H + 63) // 64 * 64
    x, w, cw = rng.standard_normal((T, H)), rng.standard_normal(H), rng.standard_normal((H, taps)) * 0.5
    h = lo.layer_norm(x, w, 1e-5)
    ref = h + lo.causal_conv(h, cw)

    def dev(a):
        out = torch.zeros(a.shape[:-1] + (ld,), device="cuda")
        out[..., :H] = torch.tensor(a)
        return out
    for _ in range(20):
        ring, at = torch.full((taps, ld), float("nan"), device="cuda"), 0
        for n in (first, rest, 5):
            y, _ = pkg.op_layernorm_conv(dev(x[at:at + n]), dev(w), 1e-5, dev(cw.T), ring, H, at)
            # f32 sums of up to 5100 terms of size 1: a few 1e-6 of the largest value
            assert np.abs(y.double().cpu().numpy()[:, :H] - ref[at:at + n]).max() < 5e-6 * np.abs(ref).max(), (at, n)
            at += n
