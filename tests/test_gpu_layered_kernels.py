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


# sizes at which each tile shape is chosen, rows and columns just past a tile, one to ten tiles of k
# (the first two: 256 x 256 with the last bands of columns in 128 x 256)
@pytest.mark.parametrize("M,N,K", [(1025, 18001, 128), (515, 33091, 192),
                                   (1025, 8963, 64), (1100, 9001, 256), (1025, 4483, 320), (513, 8961, 128), (513, 4483, 192),
                                   (257, 4481, 640), (600, 3001, 128), (300, 2049, 192), (129, 2001, 64), (70, 130, 448), (1, 1, 64)])
def test_bf16_product_of_every_shape(pkg, M, N, K):
    import torch

    g = torch.Generator(device="cuda").manual_seed(M)
    a = torch.randn((M, K), generator=g, device="cuda").bfloat16()
    b = torch.randn((N, K), generator=g, device="cuda").bfloat16()
    ref = a.double() @ b.double().t()
    scale = float(ref.abs().max())
    ldc = N + 5
    for parts, c_bf16 in [(p, False) for p in sorted({1, min(2, K // 64), K // 64})] + [(1, True)]:
        c = torch.full((parts * M + 1, ldc), 7.0, dtype=torch.bfloat16 if c_bf16 else torch.float32, device="cuda")
        rc = pkg.lib().w4a32_op_matmul_bf16_nt(a.data_ptr(), b.data_ptr(), c.data_ptr(), M, N, K, ldc, int(c_bf16), parts,
                                               torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        got = c[:parts * M, :N].double().view(parts, M, N).sum(0)
        # exact products, f32 sums of up to 640 terms: 640 x 2^-24 at most, a sixth of it seen; bf16 results: half a step
        assert float((got - ref).abs().max()) / scale < (4e-3 if c_bf16 else 4e-6), (parts, c_bf16)
        assert bool((c[:parts * M, N:] == 7).all()) and bool((c[parts * M:] == 7).all())


@pytest.mark.parametrize("rows,hidden,experts,top,ff", [
    (190, 64, 2, 1, 64),      # 95 rows per expert: tiles of 64 rows; one tile of columns, half full
    (200, 130, 2, 1, 130),    # 100: 128 rows
    (1540, 72, 4, 2, 100),    # 770
    (12400, 70, 128, 1, 900),   # 96, about 160 tiles of rows
    (12400, 1800, 128, 1, 60),  # ... column counts that are no multiple of a tile
    (1900, 1530, 40, 3, 60),    # 142
    (1100, 1530, 8, 2, 1500),   # 275
    (2500, 1800, 40, 2, 310),   # 125
    (2500, 1800, 4, 2, 900),    # 1250
])
def test_grouped_products_of_every_height(pkg, rows, hidden, experts, top, ff):
    grouped_products(pkg, rows, hidden, experts, top, ff)


# bf16: every pair of tiles that two products take, by their costs; row and column counts that are no multiples of them
@pytest.mark.parametrize("rows,hidden,experts,top,ff,up,down", [
    (578, 123, 3, 1, 81, (128, 128), (128, 128)),
    (2517, 258, 40, 4, 432, (128, 128), (128, 256)),
    (4459, 2725, 3, 1, 259, (128, 128), (256, 256)),   # an expert's last rows in 128 x 256, here and below
    (3884, 826, 40, 4, 85, (128, 256), (128, 128)),
    (5280, 880, 4, 1, 386, (128, 256), (128, 256)),
    (3739, 1577, 4, 2, 260, (128, 256), (256, 256)),
    (5819, 273, 40, 4, 210, (256, 256), (128, 128)),
    (3596, 290, 8, 4, 448, (256, 256), (128, 256)),
    (4132, 700, 40, 4, 257, (256, 256), (256, 256)),
])
def test_grouped_products_of_every_pair_of_tiles(pkg, rows, hidden, experts, top, ff, up, down):
    for which, tile in ((0, up), (1, down)):
        assert pkg.lib().w4a32_op_experts_tile(pkg.LAYERED_BF16, rows, hidden, experts, top, ff, which) == tile[0] << 16 | tile[1]
    grouped_products(pkg, rows, hidden, experts, top, ff)


def grouped_products(pkg, rows, hidden, experts, top, ff):
    import torch

    g = torch.Generator(device="cuda").manual_seed(rows)
    rnd = lambda *s, std=1.0: (torch.randn(s, generator=g, device="cuda") * std).bfloat16()
    pad = lambda n: (n + 63) // 64 * 64
    h, gate, up = rnd(rows, hidden), rnd(experts, ff, hidden, std=hidden ** -0.5), rnd(experts, ff, hidden, std=hidden ** -0.5)
    down = rnd(experts, hidden, ff, std=ff ** -0.5)
    # experts of unequal use, no close calls
    logits = torch.stack([torch.randperm(experts, generator=g, device="cuda") for _ in range(rows)]).float()
    logits[:rows // 3, 0] += 100
    _, chosen = logits.topk(top, 1)
    share = torch.softmax(logits.gather(1, chosen).double(), 1)
    ref = torch.zeros((top, rows, hidden), dtype=torch.float64, device="cuda")
    for e in range(experts):
        r, slot = (chosen == e).nonzero(as_tuple=True)
        x = h[r].double()
        gg = (x @ gate[e].double().t()).clamp(max=0.9)
        uu = (x @ up[e].double().t()).clamp(-0.9, 0.9)
        ref[slot, r] = share[r, slot, None] * ((gg * torch.sigmoid(1.702 * gg) * (uu + 1)) @ down[e].double().t())
    # tolerances of tests/test_gpu_lesarax.py::test_experts_alone, whose operands these are
    for dtype, tol in ((torch.float32, 3e-6), (torch.bfloat16, 1e-2)):
        hp = torch.zeros((rows, pad(hidden)), dtype=dtype, device="cuda")
        hp[:, :hidden] = h
        dp = torch.zeros((experts, pad(hidden), pad(ff)), dtype=dtype, device="cuda")
        dp[:, :hidden, :ff] = down
        parts = pkg.op_experts(hp, logits, pkg.pack_gate_up(gate.to(dtype), up.to(dtype)), dp, hidden, top, ff, 0.9).double()
        assert bool((parts[:, :, hidden:] == 0).all())
        assert float((parts[:, :, :hidden] - ref).abs().max()) < tol * float(ref.abs().max())


# rows of results of 2396745 f32, 4793490 bf16 values are the longest whose stores have 32-bit offsets; of operands 8388607 bf16,
# 4194303 f32 (in whole steps of 64 and 32)
@pytest.mark.parametrize("M,N,K,kinds", [(9, 2396745, 64, "bf16 f32"), (67, 2396746, 64, "bf16 f32"), (9, 4793491, 64, "bf16 bf16"),
                                         (67, 2396746, 32, "f32 f32"), (67, 70, 8388544, "bf16 f32"), (67, 70, 8388608, "bf16 f32"),
                                         (9, 70, 8388608, "bf16 bf16"), (67, 70, 4194304, "f32 f32")])
def test_products_of_rows_of_millions(pkg, M, N, K, kinds):
    import torch

    types = {"bf16": torch.bfloat16, "f32": torch.float32}
    dtype, out = (types[t] for t in kinds.split())
    g = torch.Generator(device="cuda").manual_seed(N)
    # 0 and +-1: sums below 2^24 in size, exact in f32 in any order
    a, b = (torch.randint(-1, 2, (n, K), generator=g, device="cuda", dtype=torch.int8).to(dtype) for n in (M, N))
    ref = torch.zeros((M, N), device="cuda")
    for k in range(0, K, 1 << 18):
        ref += a[:, k:k + (1 << 18)].float() @ b[:, k:k + (1 << 18)].float().t().contiguous()
    c = torch.full((M + 1, N), 7.0, dtype=out, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    if dtype == torch.float32:
        rc = pkg.lib().w4a32_op_matmul_f32_nt(a.data_ptr(), b.data_ptr(), c.data_ptr(), M, N, K, stream)
    else:
        rc = pkg.lib().w4a32_op_matmul_bf16_nt(a.data_ptr(), b.data_ptr(), c.data_ptr(), M, N, K, N, int(out == dtype), 1, stream)
    assert rc == 0
    assert torch.equal(c[:M], ref.to(out)) and bool((c[M] == 7).all())


@pytest.mark.parametrize("rows,hidden,ff,kind", [(67, 40, 4793450, "bfloat16"), (67, 40, 2396740, "float32"),
                                                 (67, 8388600, 40, "bfloat16")])
def test_experts_of_rows_of_millions(pkg, rows, hidden, ff, kind):
    import torch

    dtype = getattr(torch, kind)
    g = torch.Generator(device="cuda").manual_seed(ff)
    rnd = lambda *s, std=1.0: (torch.randn(s, generator=g, device="cuda") * std).bfloat16().to(dtype)
    pad = lambda n: (n + 63) // 64 * 64
    h, gate, up, down = rnd(rows, hidden), rnd(1, ff, hidden, std=hidden ** -0.5), rnd(1, ff, hidden, std=hidden ** -0.5), \
        rnd(1, hidden, ff, std=ff ** -0.5)
    hp = torch.zeros((rows, pad(hidden)), dtype=dtype, device="cuda")
    hp[:, :hidden] = h
    dp = torch.zeros((1, pad(hidden), pad(ff)), dtype=dtype, device="cuda")
    dp[:, :hidden, :ff] = down
    logits = torch.zeros((rows, 1), device="cuda")
    parts = pkg.op_experts(hp, logits, pkg.pack_gate_up(gate, up), dp, hidden, 1, ff, 0.9)
    del hp, dp
    gg = (h.double() @ gate[0].double().t().contiguous()).clamp(max=0.9)
    uu = (h.double() @ up[0].double().t().contiguous()).clamp(-0.9, 0.9)
    act = gg * torch.sigmoid(1.702 * gg) * (uu + 1)
    del gg, uu, gate, up
    assert bool((parts[:, :, hidden:] == 0).all())
    ref = act @ down[0].double().t().contiguous()
    # f32 sums of n = 2.4 to 8.4 million terms, one after the other: each addition rounds the sum so far, sqrt(n) 2^-24 of the result
    # in all, 1.7e-4 at the most; bf16 as in test_grouped_products_of_every_height
    assert float((parts[0, :, :hidden] - ref).abs().max()) < (2e-4 if kind == "float32" else 1e-2) * float(ref.abs().max())


@pytest.mark.parametrize("kind", ["float32", "bfloat16"])
def test_experts_gates_of_any_size(pkg, kind):
    """Each result is one gate and one up value's, the other terms are 0: every value for itself, from where the sigmoid is 0 up."""
    import torch

    dtype, n = getattr(torch, kind), 192
    g = torch.Generator(device="cuda").manual_seed(3)
    eye = torch.eye(n, device="cuda", dtype=dtype)
    gate = (torch.rand((n, n), generator=g, device="cuda") * 59.5 - 50.5).to(dtype)
    gate[0, :8] = torch.tensor([-51.5, -52.5, -60.0, -100.0, -1000.0, -3e30, -0.0, 1e30], device="cuda")
    up = (torch.randn((n, n), generator=g, device="cuda") * 3).to(dtype)
    parts = pkg.op_experts(eye, torch.zeros((n, 1), device="cuda"), pkg.pack_gate_up(gate[None], up[None]), eye[None].contiguous(), n,
                           1, n, 7.0)[0].double()
    gg, uu = gate.double().clamp(max=7.0).t(), up.double().clamp(-7.0, 7.0).t()
    ref = gg * torch.sigmoid(1.702 * gg) * (uu + 1)
    # 1.702 g rounded, up to 86: 86 x 2^-24 = 5.1e-6 in the exponential; a rounding to bf16: 2^-9. Below 2^-126 sigmoids may be 0
    assert bool((((parts - ref).abs() - 51.5 * 2.0 ** -126 * 22) <= ref.abs() * (1e-5 if kind == "float32" else 2.0 ** -8)).all())


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("width,taps", [(2050, 4), (2500, 8), (4200, 3)])
def test_norm_of_wide_rows_in_two_launches(width, taps, dtype):
    """Portions of one to 40 rows (strips of 16), behind each other and in front of position 0."""
    cfg = lm.config([lm.retention(1, 16, 16, 8, ff=70), lm.attention(2, 1, 16, 16, 64, 8)], width=width, taps=taps)
    w = lm.random_weights(cfg, seed=width)
    tokens = np.random.default_rng(width).integers(0, cfg["vocab"], 40)
    ref = lo.forward(cfg, w, tokens)
    dec = lm.runner(cfg, w, dtype, max_seq=41)
    state = dec.new_state()
    for portions in ([40], [2] * 20, [17, 3, 1, 16, 3], [33, 7]):
        at = 0
        for n in portions:
            got = dec.forward(state, tokens[at:at + n], at)
            assert lm.errors(got, ref[at:at + n]).max() < TOL[dtype], (portions, at)
            at += n


@pytest.mark.parametrize("F,ld", [(2049, 2112), (4097, 4160), (6200, 6208), (10241, 10304), (20481, 20544), (39930, 39936)])
def test_polynorm_of_every_row_length(pkg, F, ld):
    import torch

    g = torch.Generator(device="cuda").manual_seed(F)
    act = torch.tensor([0.7, -0.4, 0.3, 0.05], device="cuda")
    for dtype, tol in ((torch.float32, 3e-6), (torch.bfloat16, 4e-3)):
        z = torch.randn((3, ld), generator=g, device="cuda").to(dtype)
        x = z[:, :F].double()
        rms = lambda t: t / torch.sqrt((t * t).mean(-1, keepdim=True) + 1e-5)
        ref = 0.7 * rms(x) - 0.4 * rms(x ** 2) + 0.3 * rms(x ** 3) + 0.05
        y = pkg.op_polynorm(z, F, act, 1e-5).double()
        # f32 sums of up to 39930 positive terms by 512 threads: far below 1e-6; bf16: half a step of the largest result
        assert float((y[:, :F] - ref).abs().max() / ref.abs().max()) < tol
        assert bool((y[:, F:] == 0).all())


@pytest.mark.parametrize("F,ld", [(3, 4), (9, 12), (33, 36), (97, 100), (2050, 2052), (4099, 4100), (6150, 6156), (20480, 20484)])
def test_polynorm_of_rows_that_end_in_half_a_piece(pkg, F, ld):
    """bf16 rows of an odd number of four elements, starting on eight bytes only: no row touches another, or what lies around all."""
    import torch

    g = torch.Generator(device="cuda").manual_seed(ld)
    act = torch.tensor([0.7, -0.4, 0.3, 0.05], device="cuda")
    rms = lambda t: t / torch.sqrt((t * t).mean(-1, keepdim=True) + 1e-5)
    for dtype, tol in ((torch.float32, 3e-6), (torch.bfloat16, 4e-3)):  # as above
        for rows, front in ((1, 0), (300, 4)):
            z = torch.randn(front + rows * ld + ld, generator=g, device="cuda").to(dtype)
            before, body = z.clone(), slice(front, front + rows * ld)
            x = before[body].view(rows, ld)[:, :F].double()
            ref = 0.7 * rms(x) - 0.4 * rms(x ** 2) + 0.3 * rms(x ** 3) + 0.05
            y = pkg.op_polynorm(z[body].view(rows, ld), F, act, 1e-5).double()
            assert float((y[:, :F] - ref).abs().max() / ref.abs().max()) < tol, (rows, dtype)
            assert bool((y[:, F:] == 0).all())
            assert torch.equal(z[:front], before[:front]) and torch.equal(z[front + rows * ld:], before[front + rows * ld:])


@pytest.mark.parametrize("M,N,K", [(2000, 3001, 256), (1985, 2945, 288), (65, 3003, 96), (9, 65, 32)])
def test_f32_products_in_one_part(pkg, M, N, K):
    """64 x 128 (the first two) and 64 x 64, from one to nine tiles of k."""
    import torch

    g = torch.Generator(device="cuda").manual_seed(M)
    a, b = (torch.randn((n, K), generator=g, device="cuda") for n in (M, N))
    ref = a.double() @ b.double().t().contiguous()
    # f32 products and sums of K terms of size 1: sqrt(K) roundings of 2^-24 of a sum of up to 5 sqrt(K), K = 288
    assert float((pkg.op_matmul_f32_nt(a, b).double() - ref).abs().max()) < 288 * 5 * 2.0 ** -24


@pytest.mark.parametrize("rows", [9, 63, 65, 130])
@pytest.mark.parametrize("width,ff,vocab", [(70, 100, 130), (1030, 2100, 65)])
def test_f32_products_of_a_prompt(width, ff, vocab, rows):
    """The f32 product's tiles through a model of one layer, where the norm behind takes parts; every token's logits."""
    cfg = lm.config([lm.retention(2, 24, 24, 8, ff=ff)], width=width, vocab=vocab)
    w = lm.random_weights(cfg, seed=rows)
    tokens = np.random.default_rng(rows).integers(0, vocab, rows)
    dec = lm.runner(cfg, w, "float32", max_seq=rows)
    assert lm.errors(dec.forward(dec.new_state(), tokens, 0), lo.forward(cfg, w, tokens)).max() < TOL["float32"]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("width,experts,top", [(70, 1, 1), (250, 9, 2), (700, 33, 16), (700, 64, 64 // 8), (1600, 64, 4), (64, 65, 3),
                                               (70, 13, 1), (70, 16, 1), (130, 32, 2), (130, 33, 2), (200, 49, 3), (200, 56, 3)])
def test_router_inside_and_in_front_of_the_experts(width, experts, top, dtype):
    # up to 64 experts, and 18 for each that is chosen less 4, by counting, else by rounds; up to 96 KB of router in the experts'
    # launch; rows that agree: the lower expert is chosen
    cfg = lm.lesarax([lm.rotary(1, 1, 16, 8, mlp=lm.moe(24, experts, top))], width=width, vocab=50)
    w = lm.lesarax_weights(cfg, seed=experts)
    router = next(k for k in w if k.endswith("router"))
    w[router][experts // 2:experts // 2 * 2] = w[router][:experts // 2]
    tokens = [3, 41, 7, 22, 9]
    dec = lm.runner(cfg, w, dtype, max_seq=8)
    state, ref = dec.new_state(), lo.forward(cfg, w, tokens)
    for i, t in enumerate(tokens):
        assert lm.errors(dec.forward(state, [t], i), ref[i:i + 1]).max() < TOL[dtype], i


@pytest.mark.parametrize("heads,dim,vdim", [(9, 24, 23), (17, 40, 64), (1, 70, 130)])
def test_recurrences_of_any_number_of_heads(heads, dim, vdim):
    # the scan deals eight heads at a time; 65, 128 and 7 tokens: chunks with a rest, whole ones, less than one
    cfg = lm.config([lm.delta(heads, heads, dim, vdim), lm.retention(heads, dim, vdim, 8)], width=66, vocab=50)
    w = lm.random_weights(cfg, seed=heads)
    tokens = [int(t) for t in np.random.default_rng(vdim).integers(0, 50, 200)]
    ref = lo.forward(cfg, w, tokens)
    dec = lm.runner(cfg, w, "float32", max_seq=256)
    state, at = dec.new_state(), 0
    for n in (65, 128, 7):
        assert lm.errors(dec.forward(state, tokens[at:at + n], at), ref[at:at + n]).max() < TOL["float32"], (at, n)
        at += n


# two chunks of up to 64 tokens: 256 workgroups of the output kernel, the most that read their operands without LDS (head buckets of 64 and
# more), and 258; value dimensions that end inside of a step of 16, and an odd number of steps
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("heads", [128, 129])
@pytest.mark.parametrize("dim,vdim", [(24, 20), (40, 44), (70, 100), (130, 140)])
def test_recurrences_on_either_side_of_a_full_chip(dim, vdim, heads, dtype):
    cfg = lm.config([lm.delta(heads, heads, dim, vdim), lm.retention(heads, dim, vdim, 8)], width=66, vocab=50)
    w = lm.random_weights(cfg, seed=heads)
    tokens = [int(t) for t in np.random.default_rng(vdim).integers(0, 50, 165)]
    ref = lo.forward(cfg, w, tokens)
    dec = lm.runner(cfg, w, dtype, max_seq=165)
    state = dec.new_state()
    for at, n in ((0, 70), (70, 30), (100, 65)):
        e = lm.errors(dec.forward(state, tokens[at:at + n], at), ref[at:at + n])
        # at position 0 a head leaves (q . k) v, which its norm scales to size 1: of 258 heads some have a q . k of 1 / 258 of |q| |k| or
        # less, whose relative error in f32 is that much larger (3.5e-5 seen in the logits, 1e-6 at the other positions)
        first = 1 if at == 0 else 0
        assert e[first:].max() < TOL[dtype] and e[0] < max(TOL[dtype], 258 * 1e-6), (at, n)


# ---------------------------------------------------------------------------------------------- attention of long prompts
# (head, 64 queries) tiles in numbers that take the kernel with keys and values in LDS: two sets of blocks, 64 queries of which the
# last are missing, windows inside of a block and across pooled ones, positions off the blocks' borders in the second portion; in f32
# the kernel on matrix instructions in the whole prompt and the second portion, in the first one wavefront per query
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("arch,layer,T", [
    ("suripel", lm.attention(32, 4, 100, 124, 70, 8), 300),
    ("suripel", lm.attention(96, 16, 50, 64, 33, 4), 390),
    ("lesarax", lm.rotary(48, 2, 128, 40), 200),
    ("lesarax", lm.latent(60, 64, 64, 48, 40, 64, 40), 450),
    ("lesarax", lm.latent(44, 120, 16, 128, 40, 100, 50), 230),  # rotated eight dimensions at a time ...
    ("lesarax", lm.latent(36, 100, 28, 90, 40, 64, 10**6), 260),   # ... and one by one
])
def test_attention_of_long_prompts(arch, layer, T, dtype):
    import torch

    cfg = lm.config([layer], width=72) if arch == "suripel" else lm.lesarax([layer], width=72)
    w = (lm.random_weights if arch == "suripel" else lm.lesarax_weights)(cfg, seed=T)
    tokens = np.random.default_rng(T).integers(0, cfg["vocab"], T)
    ref = lo.forward(cfg, w, tokens)
    dec = lm.runner(cfg, w, dtype, T + 70)
    state = dec.new_state()
    whole = dec.forward(state, tokens, 0)
    assert lm.errors(whole, ref).max() < TOL[dtype]
    parts = torch.cat([dec.forward(state, tokens[:37], 0), dec.forward(state, tokens[37:], 37)])
    assert lm.errors(parts, ref).max() < TOL[dtype]
    # what the cache holds past the sequence does not matter: a longer one of values that are not finite lay there
    bad = lm.runner(cfg, w, dtype, T + 70)
    bad._keep[-3][:, :] = float("inf")
    state = bad.new_state()
    bad.forward(state, np.zeros(T + 64, dtype=np.int64), 0, want=[])
    assert torch.equal(dec.forward(state, tokens, 0), whole)


# the same kernel with each size of a head and of the keys' second part; the last 64 queries are 4, 10, 16 and 20; blocks with masks and, without
# a window, ones in which every key is seen; positions off the blocks' borders in the second portion
@pytest.mark.parametrize("layer,T", [
    (lm.latent(40, 128, 64, 128, 40, 64, 100), 260),
    (lm.latent(33, 120, 64, 128, 40, 64, 10**6), 330),
    (lm.latent(64, 64, 16, 64, 40, 64, 100), 400),
    (lm.latent(64, 60, 32, 50, 40, 64, 40), 404),
])
def test_latent_attention_of_long_prompts(pkg, layer, T):
    import ctypes
    import torch

    cfg = lm.lesarax([layer], width=72)
    w = lm.lesarax_weights(cfg, seed=T)
    tokens = np.random.default_rng(T).integers(0, cfg["vocab"], T)
    ref = lo.forward(cfg, w, tokens)
    dec = lm.runner(cfg, w, "bfloat16", T)
    for M, pos0 in ((T, 0), (T - 37, 37)):
        assert pkg.lib().w4a32_layered_attention_kernel(ctypes.byref(dec.cfg), 0, M, pos0) == pkg.ATTENTION_64
    state = dec.new_state()
    assert lm.errors(dec.forward(state, tokens, 0), ref).max() < TOL["bfloat16"]
    parts = torch.cat([dec.forward(state, tokens[:37], 0), dec.forward(state, tokens[37:], 37)])
    assert lm.errors(parts, ref).max() < TOL["bfloat16"]


# f32, few tokens: a wavefront per query up to 80 of them on up to 64 tokens each; matrix instructions where a late portion sees many pooled blocks,
# the last of 32 of them partly or by some queries only
@pytest.mark.parametrize("dim,vdim,heads", [(100, 128, 4), (256, 200, 2), (30, 32, 6)])
def test_f32_attention_of_short_portions(pkg, dim, vdim, heads):
    import ctypes

    cfg = lm.config([lm.attention(heads, 2, dim, vdim, 21, 3)], width=72)
    w = lm.random_weights(cfg, seed=dim)
    portions = [(80, pkg.ATTENTION_QUERY if dim > 64 else pkg.ATTENTION_32), (3, pkg.ATTENTION_QUERY), (250, pkg.ATTENTION_32),
                (2, pkg.ATTENTION_QUERY), (64, pkg.ATTENTION_32), (7, pkg.ATTENTION_32)]
    T = sum(n for n, _ in portions)
    tokens = np.random.default_rng(dim).integers(0, cfg["vocab"], T)
    ref = lo.forward(cfg, w, tokens)
    dec = lm.runner(cfg, w, "float32", T)
    state, at = dec.new_state(), 0
    for n, which in portions:
        assert pkg.lib().w4a32_layered_attention_kernel(ctypes.byref(dec.cfg), 0, n, at) == which, (n, at)
        assert lm.errors(dec.forward(state, tokens[at:at + n], at), ref[at:at + n]).max() < TOL["float32"], (n, at)
        at += n


# A token whose row of the embedding is not finite: its key and value are not, and nobody else's result may meet them but through attention to
# it. In f32 every query in front of it, and behind it every one whose window has left it, keeps its value. (It stands inside of a block of 32
# keys with both kinds; the last row has few tokens on few keys, one wavefront per query.)
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("arch,layer,T,at,left", [
    ("lesarax", lm.rotary(4, 2, 64, 16), 110, 50, None),
    ("lesarax", lm.rotary(3, 1, 24, 8), 100, 70, None),
    ("lesarax", lm.latent(4, 100, 16, 90, 32, 48, 20), 150, 70, 90),
    ("lesarax", lm.latent(2, 140, 40, 130, 32, 48, 33), 130, 40, 73),
    ("suripel", lm.attention(4, 2, 40, 36, 10**6, 8), 90, 77, None),
    ("suripel", lm.attention(4, 2, 40, 36, 24, 8), 130, 77, None),
    ("lesarax", lm.rotary(4, 2, 64, 16), 40, 20, None),
])
def test_f32_attention_keeps_values_apart_that_are_not_finite(arch, layer, T, at, left, bad):
    cfg = lm.config([layer], width=72) if arch == "suripel" else lm.lesarax([layer], width=72)
    w = (lm.random_weights if arch == "suripel" else lm.lesarax_weights)(cfg, seed=T)
    tokens = np.random.default_rng(T).integers(1, cfg["vocab"], T)
    tokens[at] = 0
    ref = lo.forward(cfg, w, tokens)
    dec = lm.runner(cfg, {**w, "embed": np.where(np.arange(cfg["vocab"])[:, None] == 0, bad, w["embed"])}, "float32", T)
    got = dec.forward(dec.new_state(), tokens, 0)
    kept = np.arange(T) < at if left is None else (np.arange(T) < at) | (np.arange(T) >= left)
    # (the first logit of a model that shares its embedding with the head is that row's)
    assert lm.errors(got[:, 1:], ref[:, 1:])[kept].max() < TOL["float32"]
