"""GPU parity of the party-local share GEMM against the oracle and fixtures."""
import os

import numpy as np
import pytest

import oracle
import praghip
from conftest import from_dev, to_dev

pytestmark = pytest.mark.gpu


def _run(x, w, shifts=None, mask_bits=64, split=False):
    """split: int32 weights pre-split on the GPU into three signed-byte planes (w_bits 24)."""
    import torch
    tx = to_dev(x)
    tw = torch.from_numpy(np.ascontiguousarray(w)).cuda()
    if split:
        tw = praghip.split_weights(tw)
    ts = None if shifts is None else torch.from_numpy(np.ascontiguousarray(shifts, dtype=np.int8)).cuda()
    y = praghip.share_gemm(tx, tw, shifts=ts, mask_bits=mask_bits)
    torch.cuda.synchronize()
    return from_dev(y)


def test_gemm_golden(gpu, golden_dir):
    data = np.load(os.path.join(golden_dir, "gemm_small.npz"))
    for name in ("i8_a", "i8_shift59", "i32_a", "i32_shift59"):
        sh = data[name + "_shift"] if name + "_shift" in data.files else None
        got = _run(data[name + "_x"], data[name + "_w"], sh, int(data[name + "_mask"][0]))
        np.testing.assert_array_equal(got, data[name + "_y"], err_msg=name)
    yc = _run(data["probe_client"], data["probe_weight"], None, 59)
    ys = _run(data["probe_server"], data["probe_weight"], None, 59)
    np.testing.assert_array_equal((yc + ys) & np.uint64((1 << 59) - 1), data["probe_plain"])


@pytest.mark.parametrize("m,k,n", [(1, 1, 1), (5, 7, 3), (33, 65, 129), (64, 128, 256), (100, 1000, 300),
                                   (31, 2048, 127), (512, 64, 128)])
@pytest.mark.parametrize("wdt", ["i8", "i32", "i32split"])
def test_gemm_ragged_vs_oracle(gpu, m, k, n, wdt):
    print(f"[gemm] m={m} k={k} n={n} {wdt}", flush=True)
    x = oracle.fill_u64(m * k, 1000 + m).reshape(m, k)
    if wdt == "i8":
        w = oracle.fill_i8(n * k, 2000 + n).reshape(n, k)
    else:
        w = (oracle.fill_u64(n * k, 3000 + n) % np.uint64(1 << 21)).astype(np.int64) - (1 << 20)
        w = w.astype(np.int32).reshape(n, k)
    sh = oracle.fill_shift(n, 4000 + k)
    for shifts, mask in ((None, 64), (sh, 59)):
        want = oracle.share_gemm(x, w, shifts, mask)
        np.testing.assert_array_equal(_run(x, w, shifts, mask, split=wdt == "i32split"), want)


def test_gemm_extreme_values(gpu):
    m, k, n = 40, 256, 160
    x = np.full((m, k), np.uint64((1 << 64) - 1))
    x[1] = 0
    x[2] = np.uint64(1 << 63)
    x[3] = np.uint64(0x8080808080808080)
    w = np.full((n, k), -127, dtype=np.int8)
    w[1] = 127
    w[2] = -128
    w[3] = 0
    np.testing.assert_array_equal(_run(x, w), oracle.share_gemm(x, w))
    w32 = np.full((n, k), -(1 << 20), dtype=np.int32)
    w32[1] = 1 << 20
    w32[2] = 0x7F7F7F  # largest weight with three balanced signed bytes
    w32[3] = -0x808080  # smallest
    np.testing.assert_array_equal(_run(x, w32), oracle.share_gemm(x, w32))
    np.testing.assert_array_equal(_run(x, w32, split=True), oracle.share_gemm(x, w32))


def test_gemm_c4_full_shape(gpu):
    """Qwen3 up/gate shape: activation shares u64 [512 x 1024] times int8 [3072 x 1024] -> [512 x 3072] mod 2^64."""
    m, k, n = 512, 1024, 3072
    x = oracle.fill_u64(m * k, 0x5052414700000004).reshape(m, k)
    w = oracle.fill_i8(n * k, 0x5052414700000104).reshape(n, k)
    np.testing.assert_array_equal(_run(x, w), oracle.share_gemm(x, w))


@pytest.mark.parametrize("m,k,n", [(512, 2048, 1024), (512, 3072, 1024), (96, 4096, 256)])
def test_gemm_split_k_shapes(gpu, m, k, n):
    """Shapes whose tiles leave most workgroup slots empty run split-K (64-bit
    atomic accumulation into a zeroed y, then the 59-bit mask): the Qwen3 o
    and down products; and a long-K thin case, on the few-row kernel."""
    print(f"[gemm] split-K m={m} k={k} n={n}", flush=True)
    x = oracle.fill_u64(m * k, 5000 + k).reshape(m, k)
    w = oracle.fill_i8(n * k, 6000 + k).reshape(n, k)
    sh = oracle.fill_shift(n, 7000 + k)
    for shifts, mask in ((None, 64), (sh, 59)):
        np.testing.assert_array_equal(_run(x, w, shifts, mask), oracle.share_gemm(x, w, shifts, mask))


@pytest.mark.parametrize("m,k,n", [(512, 1024, 3072), (500, 1024, 3000), (481, 640, 2900)])
def test_gemm_wide_tiles(gpu, m, k, n):
    """Shapes whose 128-column grid would load the CUs unevenly run 192-column
    tiles with one workgroup per CU (the pipelined kernel): ragged rows and
    columns, shifts and the 59-bit ring included."""
    print(f"[gemm] wide tiles m={m} k={k} n={n}", flush=True)
    x = oracle.fill_u64(m * k, 9000 + n).reshape(m, k)
    w = oracle.fill_i8(n * k, 9100 + n).reshape(n, k)
    sh = oracle.fill_shift(n, 9200 + n)
    for shifts, mask in ((None, 64), (sh, 59)):
        np.testing.assert_array_equal(_run(x, w, shifts, mask), oracle.share_gemm(x, w, shifts, mask))


def test_gemm_c4_f12_presplit(gpu, tmp_path):
    """C4's shape with the reference's weight domain (int32 f12, |w| <= 2^20,
    quantize_weights.py:91,102) pre-split into three signed-byte planes: once
    on the GPU (split_weights) and once on the host at upload
    (MappedWeights.upload_split), both identical and bit-exact against the
    oracle's int32 product, shifts and the 59-bit ring included."""
    import torch
    m, k, n = 512, 1024, 3072
    x = oracle.fill_u64(m * k, 0x5052414700000014).reshape(m, k)
    w = ((oracle.fill_u64(n * k, 0x5052414700000114) % np.uint64((1 << 21) + 1)).astype(np.int64)
         - (1 << 20)).astype("<i4").reshape(n, k)
    w[0, :4] = [1 << 20, -(1 << 20), 0x7F7F7F, -0x808080]
    sh = oracle.fill_shift(n, 0x5052414700000214)
    planes = praghip.split_weights(torch.from_numpy(w).cuda())
    path = tmp_path / "model.layers.0.mlp.up_proj.weight.npy"
    np.save(path, w)
    host_planes = torch.empty((3, n, k), dtype=torch.int8, device="cuda")
    with praghip.MappedWeights(str(path), n, k) as mw:
        mw.upload_split(host_planes)
    torch.cuda.synchronize()
    assert torch.equal(planes, host_planes)
    tx, ts = to_dev(x), torch.from_numpy(sh).cuda()
    for shifts, mask in ((None, 64), (ts, 59)):
        y = praghip.share_gemm(tx, planes, shifts=shifts, mask_bits=mask)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(from_dev(y), oracle.share_gemm(x, w, None if shifts is None else sh, mask))


@pytest.mark.parametrize("m,k,n", [(512, 1024, 3072), (33, 100, 129), (1, 64, 1)])
def test_gemm_valu_form(gpu, m, k, n):
    """The VALU dot-product form (the measured alternative to the MFMA
    kernels) gives the oracle's results, shifts and the 59-bit ring included."""
    import torch
    print(f"[gemm-valu] m={m} k={k} n={n}", flush=True)
    x = oracle.fill_u64(m * k, 8000 + k).reshape(m, k)
    w = oracle.fill_i8(n * k, 8100 + n).reshape(n, k)
    sh = oracle.fill_shift(n, 8200 + m)
    for shifts, mask in ((None, 64), (sh, 59)):
        ts = None if shifts is None else torch.from_numpy(shifts).cuda()
        y = praghip.share_gemm_valu(to_dev(x), torch.from_numpy(w).cuda(), shifts=ts, mask_bits=mask)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(from_dev(y), oracle.share_gemm(x, w, shifts, mask))


def _batch(descs):
    import ctypes

    import torch
    from praghip import _lib
    arr = (_lib.GemmDesc * len(descs))(*[
        _lib.GemmDesc(x.data_ptr(), w.data_ptr(), 0 if s is None else s.data_ptr(), y.data_ptr(), x.shape[0],
                      x.shape[1], w.shape[0], 8, mask) for x, w, s, y, mask in descs])
    _lib.check(_lib.lib().praghip_share_gemm_batch(0, ctypes.cast(arr, ctypes.c_void_p), len(descs), None))
    torch.cuda.synchronize()


def test_gemm_batch_split_k_outputs_cleared_together(gpu):
    """praghip_share_gemm_batch on outputs that hold stale values: products that
    would split K alone run together (the Qwen3 o and down shapes here, with
    and without the 59-bit mask), and one after the other, each with its own
    clear, when such an output is also an earlier product's input: product 1
    reads buffer B as its shares, then product 2 (split K) writes B."""
    import torch
    specs = [(512, 2048, 1024, None, 64), (512, 3072, 1024, 7001, 59), (64, 1024, 512, None, 64),
             (512, 2048, 1024, 7002, 64)]
    descs, want = [], []
    for i, (m, k, n, shseed, mask) in enumerate(specs):
        x = oracle.fill_u64(m * k, 8000 + i).reshape(m, k)
        w = oracle.fill_i8(n * k, 8100 + i).reshape(n, k)
        sh = None if shseed is None else oracle.fill_shift(n, shseed)
        want.append(oracle.share_gemm(x, w, sh, mask))
        ts = None if sh is None else torch.from_numpy(sh.astype(np.int8)).cuda()
        y = to_dev(np.full((m, n), 0x1234, dtype=np.uint64))  # stale values the clear must remove
        descs.append((to_dev(x), torch.from_numpy(w).cuda(), ts, y, mask))
    print("[gemm] batch, outputs cleared together", flush=True)
    _batch(descs)
    for i, d in enumerate(descs):
        np.testing.assert_array_equal(from_dev(d[3]), want[i], err_msg=f"product {i}")
    # overlap: product 1's shares are B, product 2 (split K, [512 x 1024]) writes B
    m, k, n = 512, 1024, 1024
    xb = oracle.fill_u64(m * k, 8200).reshape(m, k)
    w1 = oracle.fill_i8(512 * k, 8201).reshape(512, k)
    x2 = oracle.fill_u64(m * 2048, 8202).reshape(m, 2048)
    w2 = oracle.fill_i8(n * 2048, 8203).reshape(n, 2048)
    B = to_dev(xb)
    y1 = to_dev(np.zeros((m, 512), dtype=np.uint64))
    y0 = to_dev(np.zeros((m, n), dtype=np.uint64))
    tw1, tw2, tx2 = torch.from_numpy(w1).cuda(), torch.from_numpy(w2).cuda(), to_dev(x2)
    print("[gemm] batch, split-K output overlapping an earlier input", flush=True)
    _batch([(tx2, tw2, None, y0, 64), (B, tw1, None, y1, 64), (tx2, tw2, None, B, 64)])
    np.testing.assert_array_equal(from_dev(y1), oracle.share_gemm(xb, w1))
    np.testing.assert_array_equal(from_dev(B), oracle.share_gemm(x2, w2))
    np.testing.assert_array_equal(from_dev(y0), oracle.share_gemm(x2, w2))


@pytest.mark.parametrize("m,k,n", [(1, 15, 1), (1, 17, 33), (3, 127, 31), (4, 128, 32), (5, 129, 33), (8, 1023, 65),
                                   (9, 1025, 64), (16, 2049, 95), (17, 63, 130), (33, 1000, 129), (40, 4097, 257),
                                   (129, 130, 1)])
@pytest.mark.parametrize("wdt", ["i8", "i32", "i32split"])
def test_gemm_any_k_and_alignment(gpu, m, k, n, wdt):
    """Small products, most of them on the few-row kernel, around its edges: rows
    about the 4-row blocks and the 32-row tile, K about the 128-wide chunks and
    64-wide steps (odd K puts every weight row at another alignment), columns
    about 32 and 128; the operands start 8 bytes (x) and one element (w) off 16
    bytes.  Whole-number arithmetic: exact."""
    import torch
    print(f"[gemm] m={m} k={k} n={n} {wdt}", flush=True)
    x = oracle.fill_u64(m * k, 11000 + m).reshape(m, k)
    if wdt == "i8":
        w = oracle.fill_i8(n * k, 12000 + n).reshape(n, k)
        w.flat[0] = -128
    else:
        w = ((oracle.fill_u64(n * k, 13000 + n) % np.uint64(0x7F7F7F + 0x808080 + 1)).astype(np.int64)
             - 0x808080).astype(np.int32).reshape(n, k)
    sh = oracle.fill_shift(n, 14000 + k)
    tx = torch.zeros(m * k + 1, dtype=torch.int64, device="cuda")[1:].view(m, k)
    tx.copy_(to_dev(x))
    tw = torch.from_numpy(w).cuda()
    if wdt == "i32split":
        tw = praghip.split_weights(tw)
    off = torch.zeros(tw.numel() + 1, dtype=tw.dtype, device="cuda")[1:].view(tw.shape)
    off.copy_(tw)
    for shifts, mask in ((None, 64), (sh, 59)):
        ts = None if shifts is None else torch.from_numpy(shifts).cuda()
        y = praghip.share_gemm(tx, off, shifts=ts, mask_bits=mask)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(from_dev(y), oracle.share_gemm(x, w, shifts, mask))


def test_gemm_batch_forms(gpu):
    """A batch mixing few-row, tiled, ragged-K and pre-split products, once
    with separate operands (run together) and once with an output that a later
    product reads (run in list order)."""
    import ctypes

    import torch
    from praghip._lib import GemmDesc, check, lib
    specs = [(3, 256, 70, 8, 64), (40, 128, 300, 8, 59), (300, 192, 520, 8, 64), (20, 100, 33, 8, 64),
             (5, 1000, 64, 24, 59), (64, 64, 128, 24, 64), (1, 64, 4096, 8, 64), (40, 320, 129, 8, 64)] * 5
    # one batch: product 1 reads product 0's output
    chain = [(40, 128, 320, 8, 64), (40, 320, 129, 8, 64)]
    for chained, rows in ((False, specs), (True, chain)):
        descs, keep, want = [], [], []
        prev = None
        for i, (m, k, n, bits, mask) in enumerate(rows):
            x = oracle.fill_u64(m * k, 15000 + i).reshape(m, k)
            tx = to_dev(x)
            if chained and prev is not None:
                x, tx = want[-1], prev
            if bits == 8:
                w = oracle.fill_i8(n * k, 16000 + i).reshape(n, k)
                tw = torch.from_numpy(w).cuda()
            else:
                w = ((oracle.fill_u64(n * k, 16000 + i) % np.uint64(1 << 21)).astype(np.int64) - (1 << 20)).astype(np.int32).reshape(n, k)
                tw = praghip.split_weights(torch.from_numpy(w).cuda())
            sh = oracle.fill_shift(n, 17000 + i)
            ts = torch.from_numpy(sh).cuda()
            y = torch.full((m, n), -1, dtype=torch.int64, device="cuda")
            prev = y
            want.append(oracle.share_gemm(x, w, sh, mask))
            keep.append((tx, tw, ts, y))
            descs.append(GemmDesc(tx.data_ptr(), tw.data_ptr(), ts.data_ptr(), y.data_ptr(), m, k, n, bits, mask))
        arr = (GemmDesc * len(descs))(*descs)
        check(lib().praghip_share_gemm_batch(0, ctypes.cast(arr, ctypes.c_void_p), len(descs),
                                             torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        for i, (_, _, _, y) in enumerate(keep):
            np.testing.assert_array_equal(from_dev(y), want[i], err_msg=f"product {i} {rows[i]}")


@pytest.mark.parametrize("m,n", [(3, 40), (512, 512), (1024, 2048)])
@pytest.mark.parametrize("bits", [8, 24, 32])
def test_gemm_empty_sum(gpu, m, n, bits):
    """K = 0 through the C ABI: y is zeroed, alone and in a batch beside a
    product with terms, whatever the output's size."""
    import ctypes

    import torch
    from praghip._lib import GemmDesc, check, lib
    print(f"[gemm] k=0 m={m} n={n} bits={bits}", flush=True)
    x = torch.ones(16, dtype=torch.int64, device="cuda")
    w = torch.ones(16, dtype=torch.int32, device="cuda")
    y = torch.full((m, n), -1, dtype=torch.int64, device="cuda")
    check(lib().praghip_share_gemm(0, x.data_ptr(), w.data_ptr(), bits, None, y.data_ptr(), m, 0, n, 59, None))
    torch.cuda.synchronize()
    assert not y.any()
    x1, w1 = oracle.fill_u64(600 * 128, 18000).reshape(600, 128), oracle.fill_i8(1000 * 128, 18001).reshape(1000, 128)
    tx, tw = to_dev(x1), torch.from_numpy(w1).cuda()
    y.fill_(-1)
    y1 = torch.full((600, 1000), -1, dtype=torch.int64, device="cuda")
    arr = (GemmDesc * 2)(GemmDesc(x.data_ptr(), w.data_ptr(), 0, y.data_ptr(), m, 0, n, bits, 64),
                         GemmDesc(tx.data_ptr(), tw.data_ptr(), 0, y1.data_ptr(), 600, 128, 1000, 8, 64))
    check(lib().praghip_share_gemm_batch(0, ctypes.cast(arr, ctypes.c_void_p), 2, None))
    torch.cuda.synchronize()
    assert not y.any()
    np.testing.assert_array_equal(from_dev(y1), oracle.share_gemm(x1, w1))


@pytest.mark.parametrize("wdt,m,k,n,want", [
    ("i32split", 1455, 47, 1057, "fused"), ("i32split", 1024, 1, 1024, "fused"), ("i32split", 1030, 65, 1030, "fused"),
    ("i32split", 1000, 700, 1024, "fused"), ("i32split", 300, 200, 6500, "fused"), ("i32split", 2100, 64, 130, "fused"),
    ("i32", 1455, 47, 1057, "fused"), ("i32", 702, 19, 3032, "fused"), ("i32", 1001, 255, 1023, "fused"),
    ("i32", 1001, 257, 1023, "reg"), ("i32split", 1000, 300, 512, "reg")])
def test_gemm_planes_in_one_workgroup(gpu, wdt, m, k, n, want):
    """Three-plane products of short K keep the outputs' sums in registers over
    the planes: rows and columns off the tile, K about a step, odd and even
    step counts, extreme weights, shifts and the 59-bit ring; the two that the
    rule leaves to planes of their own beside them.  Exact."""
    import gemm_rule
    import torch
    print(f"[gemm] m={m} k={k} n={n} {wdt} {want}", flush=True)
    x = oracle.fill_u64(m * k, 19000 + m).reshape(m, k)
    w = ((oracle.fill_u64(n * k, 19100 + n) % np.uint64(0x7F7F7F + 0x808080 + 1)).astype(np.int64)
         - 0x808080).astype(np.int32).reshape(n, k)
    w.flat[0], w.flat[-1] = 0x7F7F7F, -0x808080
    sh = oracle.fill_shift(n, 19200 + k)
    tx, tw = to_dev(x), torch.from_numpy(w).cuda()
    if wdt == "i32split":  # one byte off 16, so that no K takes the LDS DMA
        off = torch.zeros(3 * n * k + 1, dtype=torch.int8, device="cuda")[1:].view(3, n, k)
        off.copy_(praghip.split_weights(tw))
        tw = off
    assert gemm_rule.kernel(wdt, m, k, n, tx.data_ptr(), tw.data_ptr())[0] == want
    for shifts, mask in ((None, 64), (sh, 59)):
        ts = None if shifts is None else torch.from_numpy(shifts).cuda()
        y = torch.full((m, n), -1, dtype=torch.int64, device="cuda")
        praghip.share_gemm(tx, tw, y=y, shifts=ts, mask_bits=mask)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(from_dev(y), oracle.share_gemm(x, w, shifts, mask))


def _mixed_batch(specs, seed, stale=-1):
    """specs: (m, k, n, wdt, mask); runs them as one batch with operands of
    their own and compares each output exactly."""
    import ctypes

    import gemm_rule
    import torch
    from praghip._lib import GemmDesc, check, lib
    descs, keep, want = [], [], []
    for i, (m, k, n, wdt, mask) in enumerate(specs):
        x = oracle.fill_u64(m * k, seed + 4 * i).reshape(m, k)
        if wdt == "i8":
            w = oracle.fill_i8(n * k, seed + 4 * i + 1).reshape(n, k)
        else:
            w = ((oracle.fill_u64(n * k, seed + 4 * i + 1) % np.uint64(1 << 21)).astype(np.int64)
                 - (1 << 20)).astype(np.int32).reshape(n, k)
        tw = torch.from_numpy(w).cuda()
        if wdt == "i32split":
            tw = praghip.split_weights(tw)
        sh = oracle.fill_shift(n, seed + 4 * i + 2)
        tx, ts = to_dev(x), torch.from_numpy(sh).cuda()
        y = torch.full((m, n), stale, dtype=torch.int64, device="cuda")
        keep.append((tx, tw, ts, y))
        want.append(oracle.share_gemm(x, w, sh, mask))
        descs.append(GemmDesc(tx.data_ptr(), tw.data_ptr(), ts.data_ptr(), y.data_ptr(), m, k, n,
                              gemm_rule.W_BITS[wdt], mask))
    arr = (GemmDesc * len(descs))(*descs)
    check(lib().praghip_share_gemm_batch(0, ctypes.cast(arr, ctypes.c_void_p), len(descs),
                                         torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    for i, (_, _, _, y) in enumerate(keep):
        np.testing.assert_array_equal(from_dev(y), want[i], err_msg=f"product {i} {specs[i]}")


def test_gemm_batch_lone_tile_product_and_grouped_planes(gpu):
    """One tiled product among products of few rows keeps its K split; the
    three-plane and int32 products of few rows run in one launch per form."""
    import gemm_rule
    tiled = (200, 3072, 1024, "i8", 59)
    assert gemm_rule.kernel("i8", *tiled[:3])[:3] == ("dma2", 768, 4)
    few = [(16, 3072, 256, "i32split", 59), (3, 1000, 70, "i32split", 64), (9, 129, 300, "i32split", 59),
           (13, 700, 90, "i32", 59), (4, 64, 33, "i32", 64), (16, 1024, 256, "i32", 59), (5, 100, 40, "i8", 64)]
    assert all(gemm_rule.kernel(wdt, m, k, n)[0] == "few" for m, k, n, wdt, _ in few)
    print("[gemm] batch: one tiled product, few rows of every form", flush=True)
    _mixed_batch(few[:3] + [tiled] + few[3:], 20000)
    print("[gemm] batch: few rows alone, more than one launch holds", flush=True)
    _mixed_batch(few * 6, 21000)


def _off(t, elements=1):
    """The tensor's values in memory that starts `elements` past an aligned address."""
    import torch
    flat = torch.zeros(t.numel() + elements, dtype=t.dtype, device="cuda")[elements:]
    return flat.view(t.shape).copy_(t)


@pytest.mark.parametrize("wdt,m,k,n,x_off,w_off,want", [
    ("i8", 486, 90, 1131, 0, 0, ("reg", 1)), ("i8", 700, 500, 700, 0, 0, ("reg", 1)),
    ("i8", 1001, 31, 1025, 0, 0, ("reg", 1)), ("i8", 512, 1024, 1024, 1, 0, ("reg", 2)),
    ("i8", 512, 1024, 1024, 0, 1, ("reg", 2)), ("i8", 300, 2047, 1025, 0, 0, ("reg", 4)),
    ("i32split", 512, 2047, 1024, 0, 0, ("reg", 2)), ("i32split", 130, 4095, 500, 0, 0, ("reg", 4)),
    ("i32", 512, 2047, 1024, 0, 0, ("reg", 2)), ("i32", 130, 4097, 520, 0, 0, ("reg", 4)),
    ("i32", 1000, 640, 1024, 0, 0, ("reg", 1))])
def test_gemm_register_staged_tiles(gpu, wdt, m, k, n, x_off, w_off, want):
    """The register-staged tile: ragged K with the tail that a split or the row
    cuts, odd and even step counts through its two LDS stages, K splits and planes
    that add into y, operands off 16 bytes; exact."""
    import gemm_rule
    import torch
    print(f"[gemm] m={m} k={k} n={n} {wdt} off {x_off} {w_off}", flush=True)
    x = oracle.fill_u64(m * k, 22000 + m).reshape(m, k)
    if wdt == "i8":
        w = oracle.fill_i8(n * k, 22100 + n).reshape(n, k)
        w.flat[-1] = -128
    else:
        w = ((oracle.fill_u64(n * k, 22200 + n) % np.uint64(0x7F7F7F + 0x808080 + 1)).astype(np.int64)
             - 0x808080).astype(np.int32).reshape(n, k)
        w.flat[0], w.flat[-1] = 0x7F7F7F, -0x808080
    sh = oracle.fill_shift(n, 22300 + k)
    tw = torch.from_numpy(w).cuda()
    if wdt == "i32split":
        tw = praghip.split_weights(tw)
    tx, tw = _off(to_dev(x), x_off), _off(tw, w_off)
    assert gemm_rule.kernel(wdt, m, k, n, tx.data_ptr(), tw.data_ptr())[0:3:2] == want
    for shifts, mask in ((None, 64), (sh, 59)):
        ts = None if shifts is None else torch.from_numpy(shifts).cuda()
        y = torch.full((m, n), -1, dtype=torch.int64, device="cuda")
        praghip.share_gemm(tx, tw, y=y, shifts=ts, mask_bits=mask)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(from_dev(y), oracle.share_gemm(x, w, shifts, mask))


def test_gemm_batch_clears_added_outputs_together(gpu):
    """Products of a batch that add into their outputs (planes and K splits on the
    tiles) have them zeroed in one launch: stale outputs, with and without the
    59-bit mask, beside products that store; exact."""
    import gemm_rule
    specs = [(512, 2047, 1024, "i32split", 59), (300, 2047, 1025, "i8", 59), (512, 1024, 1024, "i32", 64),
             (77, 3072, 1024, "i32split", 64), (5, 100, 40, "i8", 59), (600, 128, 1000, "i8", 59), (600, 128, 900, "i8", 64)]
    rule = [gemm_rule.kernel(wdt, m, k, n) for m, k, n, wdt, _ in specs]
    assert [r[4] for r in rule] == [True, True, True, True, False, False, False]
    print("[gemm] batch: outputs that are added into, cleared together", flush=True)
    _mixed_batch(specs, 23000, stale=0x1234)
