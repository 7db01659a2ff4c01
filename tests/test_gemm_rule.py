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


@pytest.mark.parametrize("wdt,few,tiles", [
    ("i8", [(1, 1024, 4096), (64, 1024, 1024), (64, 63, 1024), (8, 64, 8000), (400, 512, 512), (200, 1024, 1024), (1000, 3072, 64)],
     [(64, 64, 1024), (64, 64, 3072), (400, 64, 1024), (1000, 64, 300), (1000, 100, 300), (4000, 100, 70), (100, 128, 3072),
      (400, 300, 512), (512, 64, 512), (1000, 128, 300), (1000, 3072, 128), (512, 1024, 3072)]),
    ("i32split", [(64, 64, 1024), (16, 3072, 1024), (200, 128, 512), (200, 1024, 512), (4000, 1024, 32), (64, 3072, 1024), (1, 3804, 308), (406, 28, 178)],
     [(200, 64, 1024), (64, 64, 3072), (400, 47, 512), (32, 2048, 3072), (8, 4096, 1024), (77, 3072, 1024)]),
    ("i32", [(13, 3072, 1024), (200, 512, 512), (200, 700, 512), (1024, 800, 100), (4000, 1024, 32)],
     [(400, 64, 300), (400, 1024, 300), (702, 19, 3032), (13, 3072, 4096)])])
def test_few_rows_only_where_they_pay(wdt, few, tiles):
    """The few-row kernel where it was measured faster than the tiles (GPU time
    of one product), the tiles elsewhere: short K in many workgroups above all."""
    W = {"i8": 8, "i32split": 24, "i32": 32}[wdt]
    assert [c[0] == "few" for c in choices([(0, 0, W, *s) for s in few + tiles])] == [True] * len(few) + [False] * len(tiles)
