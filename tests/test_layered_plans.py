"""Which kernel a portion's attention takes in the layered decoder, at sizes where both were timed. No GPU: the choice is host code."""
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


@pytest.mark.parametrize("window,M,pos0,which", [(0, 64, 0, QUERY), (0, 65, 0, W32), (0, 2, 126, QUERY), (0, 2, 127, W32),
                                                 (128, 64, 4000, QUERY), (129, 64, 4000, W32)])
def test_f32_prompts(pkg, window, M, pos0, which):
    assert kernel(pkg, "f32", "rotary", 8, 128, window, M, pos0, rot=64) == which


def test_what_has_no_attention_or_no_portion(pkg):
    assert kernel(pkg, "bf16", "rotary", 8, 128, 0, 1, 0, rot=64) < 0
    assert kernel(pkg, "bf16", "rotary", 8, 128, 0, 8192, 1, rot=64) < 0
    assert kernel(pkg, "bf16", "retention", 8, 128, 0, 64, 0, rot=64) < 0
