"""Host-side check of the share GEMM's dispatch rule."""
import pytest

from gemm_rule import choices


@pytest.mark.parametrize("w_bits", [8, 24, 32])
@pytest.mark.parametrize("x,w", [(0, 0), (8, 0), (0, 1)])
def test_empty_sums_have_a_kernel(w_bits, x, w):
    """K = 0 is a sum of nothing: every size has a choice, and it splits no K."""
    sizes = [(1, 1), (5, 33), (512, 512), (512, 4096), (1 << 14, 1 << 14), ((1 << 31) - 1, 1)]
    for kernel, k_split, splits, _, adds in choices([(x, w, w_bits, m, 0, n) for m, n in sizes]):
        assert (kernel, k_split, splits, adds) == ("zero", 0, 0, False)


@pytest.mark.parametrize("w_bits", [8, 24, 32])
def test_k_splits_cover_k(w_bits):
    """The splits are whole 64-word steps that cover K, each with a part of it."""
    sizes = [(m, k, n) for m in (1, 33, 512, 4000) for k in (1, 63, 64, 65, 1000, 2047, 2048, 4096, 131071)
             for n in (1, 129, 1024, 9000)]
    for (m, k, n), (kernel, k_split, splits, planes, adds) in zip(
            sizes, choices([(0, 0, w_bits, m, k, n) for m, k, n in sizes])):
        if kernel == "few":
            continue
        assert k_split % 64 == 0 and (splits - 1) * k_split < k <= splits * k_split
        assert adds == (splits * planes > 1 and kernel != "fused")
        assert kernel in ("reg", "fused") or k % 64 == 0
