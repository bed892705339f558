"""Which kernel a portion's attention takes in the layered decoder and which tiles its experts' products, at sizes where all of them
were timed. No GPU: the choice is host code."""
import ctypes

import pytest

QUERY, W32, W64 = 0, 1, 2   # a wavefront per query; 32 queries per workgroup; 64, with keys and values through LDS


def kernel(pkg, dtype, mixer, heads, dim, window, M, pos0, pool=0, rot=0):
    layer = (pkg.LayerConfig * 1)()
    c = layer[0]
    c.mixer, c.heads, c.kv_heads, c.dim, c.vdim, c.scale, c.kv_from = pkg.MIXERS[mixer], heads, heads, dim, dim, dim ** -0.5, -1
    c.window, c.pool, c.rot_dims, c.rot_base = window, pool, rot, 1e4
    if mixer == "latent":
        c.q_rank, c.kv_rank, c.rot_part = 64, 64, rot
    cfg = pkg.LayeredConfig(64, 64, 1, 3 if mixer == "attention" else 0, 1e-5, pkg.LAYERED_BF16 if dtype == "bf16" else pkg.LAYERED_F32, 8192, 8192,
                            layer, pkg.NORM_LAYER if mixer == "attention" else pkg.NORM_RMS, 1.0)
    return pkg.lib().w4a32_layered_attention_kernel(ctypes.byref(cfg), 0, M, pos0)


# us in the kernel of 32 queries / of 64
@pytest.mark.parametrize("mixer,heads,dim,window,pool,rot,M,pos0,which", [
    ("attention", 8, 128, 256, 16, 0, 1024, 0, W32),       # 12.4 / 16.2: 256 workgroups of 32 queries, one per CU
    ("latent", 8, 128, 300, 0, 64, 1024, 0, W32),          # 17.2 / 20.6
    ("latent", 16, 128, 300, 0, 16, 512, 1200, W32),       # 15.9 / 18.6
    ("latent", 28, 128, 300, 0, 64, 260, 0, W32),          # 14.8 / 17.6: 252
    ("attention", 64, 128, 1024, 32, 0, 66, 0, W32),       # 8.0 / 8.8: 192
    ("attention", 28, 128, 256, 16, 0, 300, 1500, W64),    # 22.4 / 16.7: 280
    ("latent", 28, 128, 300, 0, 64, 300, 1500, W64),       # 28.4 / 20.1
    ("latent", 6, 128, 300, 0, 32, 1501, 0, W64),          # 25.8 / 18.4: 282
    ("attention", 8, 128, 1024, 32, 0, 2048, 0, W64),      # 36.3 / 30.5
    ("latent", 12, 128, 0, 0, 64, 1501, 0, W64),           # 53.8 / 45.6
    ("latent", 12, 128, 0, 0, 128, 1501, 0, W32),          # a second part of 128 dimensions has no kernel of 64 queries
    ("rotary", 12, 256, 0, 0, 64, 1501, 0, W32),           # nor have heads of 256
])
def test_bf16_prompts(pkg, mixer, heads, dim, window, pool, rot, M, pos0, which):
    assert kernel(pkg, "bf16", mixer, heads, dim, window, M, pos0, pool, rot) == which


# what tests/test_gpu_layered_kernels.py runs as attention of long prompts is what it says
@pytest.mark.parametrize("mixer,heads,dim,window,pool,rot,M", [("attention", 32, 124, 70, 8, 0, 300), ("attention", 96, 64, 33, 4, 0, 390),
                                                               ("rotary", 48, 128, 0, 0, 40, 200), ("latent", 60, 64, 40, 0, 64, 450),
                                                               ("latent", 44, 128, 50, 0, 16, 230), ("latent", 36, 100, 0, 0, 28, 260)])
def test_long_prompts_of_the_gpu_tests(pkg, mixer, heads, dim, window, pool, rot, M):
    assert kernel(pkg, "bf16", mixer, heads, dim, window, M, 0, pool, rot) == W64
    assert kernel(pkg, "f32", mixer, heads, dim, window, M, 0, pool, rot) == W32


# us of a wavefront per query / in the kernel of 32 queries
@pytest.mark.parametrize("heads,dim,window,pool,M,pos0,which", [
    (8, 128, 0, 0, 64, 0, QUERY), (8, 128, 0, 0, 65, 0, W32), (8, 128, 0, 0, 2, 126, QUERY), (8, 128, 0, 0, 2, 127, W32),
    (8, 128, 128, 10**6, 64, 4000, QUERY), (8, 128, 129, 10**6, 64, 4000, W32),
    (4, 128, 64, 4, 65, 0, QUERY), (4, 128, 64, 4, 80, 0, QUERY), (4, 128, 64, 4, 81, 0, W32),   # 16.5 / 17.8 (65)
    (9, 128, 64, 4, 65, 0, W32), (16, 128, 64, 4, 65, 0, W32),                                   # 19.3 / 18.4 (16 heads)
    (4, 64, 64, 4, 65, 0, W32),
    (8, 128, 64, 4, 2, 318, QUERY), (8, 128, 64, 4, 2, 322, W32),   # 64 tokens and 64, 65 pooled blocks
    (8, 128, 64, 4, 2, 1900, W32), (8, 128, 20, 4, 64, 1000, W32),  # 95 / 37, 61 / 29
])
def test_f32_prompts(pkg, heads, dim, window, pool, M, pos0, which):
    mixer, rot = ("attention", 0) if pool else ("rotary", 64)
    assert kernel(pkg, "f32", mixer, heads, dim, window, M, pos0, pool, rot) == which


def test_what_has_no_attention_or_no_portion(pkg):
    assert kernel(pkg, "bf16", "rotary", 8, 128, 0, 1, 0, rot=64) < 0
    assert kernel(pkg, "bf16", "rotary", 8, 128, 0, 8192, 1, rot=64) < 0
    assert kernel(pkg, "bf16", "retention", 8, 128, 0, 64, 0, rot=64) < 0


# us in tiles of 256 x 256 (an expert's last rows in 128 x 256), 128 x 256 and 128 x 128: the chosen one is at most a seventh slower than the best
TILES = [256 << 16 | 256, 128 << 16 | 256, 128 << 16 | 128]


@pytest.mark.parametrize("M,hidden,experts,top,ff,up,down", [
    (900, 1536, 16, 4, 2240, [86.5, 89.1, 80.7], [54.0, 43.3, 49.7]),
    (1501, 1536, 16, 4, 2240, [103.1, 114.5, 111.5], [57.4, 77.7, 69.3]),
    (2048, 1536, 16, 4, 2240, [136.1, 139.7, 146.4], [62.8, 78.9, 88.3]),
    (512, 3584, 16, 4, 4736, [256.7, 282.5, 293.4], [110.4, 170.3, 165.1]),
    (2048, 3584, 16, 4, 4736, [541.1, 627.7, 674.9], [285.3, 313.6, 360.1]),
    (3646, 512, 64, 4, 400, [33.4, 36.1, 24.7], [22.3, 27.0, 21.8]),
    (3369, 2560, 64, 6, 1408, [434.9, 407.5, 404.1], [258.3, 230.6, 236.5]),
    (1402, 1536, 24, 8, 256, [39.8, 28.4, 30.0], [35.2, 33.0, 27.1]),
    (700, 1536, 16, 4, 2240, [90.1, 85.8, 75.7], [51.8, 41.3, 46.1]),
    (1225, 1024, 64, 6, 1024, [63.6, 76.0, 68.6], [41.6, 53.2, 45.7]),
    (3446, 2560, 8, 4, 1408, [201.1, 210.3, 228.1], [125.3, 130.7, 135.1]),
])
def test_tiles_of_the_experts(pkg, M, hidden, experts, top, ff, up, down):
    for which, us in ((0, up), (1, down)):
        tile = pkg.lib().w4a32_op_experts_tile(pkg.LAYERED_BF16, M, hidden, experts, top, ff, which)
        assert us[TILES.index(tile)] <= 1.15 * min(us), which


def test_tiles_of_few_rows_and_f32(pkg):
    tile = lambda dtype, M: pkg.lib().w4a32_op_experts_tile(dtype, M, 1536, 16, 4, 2240, 0)
    assert tile(pkg.LAYERED_BF16, 383) == tile(pkg.LAYERED_F32, 383) == 64 << 16 | 128
    assert tile(pkg.LAYERED_BF16, 384) in TILES and tile(pkg.LAYERED_F32, 384) == TILES[2]
    assert tile(pkg.LAYERED_F32, 4096) == TILES[2]
    assert pkg.lib().w4a32_op_experts_tile(pkg.LAYERED_BF16, 100, 64, 4, 5, 64, 0) < 0
