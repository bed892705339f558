"""W4A32 prefill products whose tile shape and number of k ranges come from the cost of the problem rather than from the
rules for the decoder's shapes: odd row counts, ragged last column tiles, odd numbers of 64-k stages, two to ten ranges,
against the oracle, and the undivided kernel against it as well."""
import numpy as np
import pytest

from conftest import make_acts, make_weights, max_abs_rel

pytestmark = pytest.mark.gpu
EINVAL = -1  # W4A32_EINVAL


@pytest.mark.parametrize("m,k,n,parts", [(14, 2720, 176, 5), (100, 2080, 100, 4), (129, 3584, 307, 6), (190, 4768, 83, 8),
                                         (16, 5600, 64, 10), (256, 5120, 1536, 5), (640, 6176, 1536, 2), (1100, 4992, 400, 3),
                                         (9, 1056, 33, 1), (300, 1024, 3000, 1), (2940, 448, 700, 1)])
def test_products_split_and_tiled_by_cost(pkg, orc, m, k, n, parts):
    import torch
    w, x = make_weights(n, k, seed=n), make_acts(m, k, seed=m, outlier_frac=0.02)
    bias = (np.random.default_rng(2).standard_normal(n) * 0.02).astype(np.float32)
    u4, sc = orc.quant_rhs(w)
    packed = pkg.repack_native(*(torch.from_numpy(a).cuda() for a in (u4, sc.view(np.int16), bias)), n, k)
    need = int(pkg.lib().w4a32_splitk_scratch_bytes(m, k, n))
    assert need == (parts * m * n * 4 if parts > 1 else 0)
    ws = pkg.quant_lhs(torch.from_numpy(x).cuda())
    whole = pkg.matmul_quantized(ws, packed, m, k, n)
    room = torch.full((need // 4 + 64,), 7.0, device="cuda")    # nothing is written behind the partial sums
    split = pkg.matmul_quantized_splitk(ws, packed, m, k, n, scratch=room)
    torch.cuda.synchronize()
    assert bool((room[need // 4:] == 7.0).all())
    rows = np.unique(np.concatenate([np.arange(0, m, 37), [m - 1]]))
    ref = orc.linear(x[rows], u4, sc, bias=bias, threads=8)
    # exact block sums on both sides: what is left is f32 rounding of K / 32 scaled sums, 280 * 2^-24 = 1.7e-5 at the most
    assert max_abs_rel(whole.cpu().numpy()[rows], ref) <= 2e-5
    assert max_abs_rel(split.cpu().numpy()[rows], ref) <= 2e-5


@pytest.mark.parametrize("m,k,n,refused", [(100, 2080, 100, False), (256, 5120, 1536, False), (640, 6112, 96, True)])
def test_results_or_scratch_on_four_bytes(pkg, m, k, n, refused):
    """A product that only its cost splits runs unsplit then; one that a long k splits is refused."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(m)
    packed = pkg.quant_pack_rhs(torch.randn((n, k), generator=g, device="cuda") * 0.02)
    ws = pkg.quant_lhs(torch.randn((m, k), generator=g, device="cuda"))
    need = int(pkg.lib().w4a32_splitk_scratch_bytes(m, k, n))
    assert need > 0
    whole = pkg.matmul_quantized(ws, packed, m, k, n)
    for y_off, scratch_off in ((1, 0), (0, 1), (3, 2)):
        y = torch.full((m * n + 8,), 7.0, device="cuda")
        scratch = torch.empty((need // 4 + 4,), device="cuda")
        rc = pkg.lib().w4a32_matmul_quantized_splitk(y.data_ptr() + 4 * y_off, ws.data_ptr(), packed.data_ptr(), m, k, n,
                                                     scratch.data_ptr() + 4 * scratch_off, need,
                                                     torch.cuda.current_stream().cuda_stream)
        if refused:
            assert rc == EINVAL and bool((y == 7.0).all())
        else:
            assert rc == 0 and torch.equal(y[y_off:y_off + m * n].view(m, n), whole)
            assert bool((y[:y_off] == 7.0).all()) and bool((y[y_off + m * n:] == 7.0).all())
