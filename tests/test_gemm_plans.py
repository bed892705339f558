"""How many k ranges the W4A32 prefill products are dealt to (the scratch they ask for), at row counts where both the rule for a
long k and the cost of the problem were timed. No GPU: the plan is host code."""
import pytest


@pytest.mark.parametrize("k,n,plans", [
    # the long k of the decoder's shapes: five ranges are not cut to two
    (8960, 1536, {9: 10, 128: 10, 129: 5, 131: 5, 256: 5, 512: 5, 513: 3, 768: 3, 769: 3, 896: 3, 897: 5, 1024: 5, 1025: 2,
                  1152: 2, 1153: 4, 1281: 3, 1664: 3, 1665: 4, 2049: 2, 2432: 2, 2433: 4, 2688: 4, 2689: 1, 8192: 1}),
    (18944, 3584, {9: 4, 128: 4, 129: 4, 257: 3, 385: 4, 1024: 2, 1025: 4, 1152: 4, 1153: 1}),
    # a middling k, few tiles
    (5120, 1536, {9: 10, 129: 5, 257: 3, 512: 2, 641: 1}),
    (1536, 8960, {9: 1, 512: 1, 8192: 1}),
])
def test_k_ranges(pkg, k, n, plans):
    for m, parts in plans.items():
        assert pkg.lib().w4a32_splitk_scratch_bytes(m, k, n) == (4 * m * n * parts if parts > 1 else 0), m
