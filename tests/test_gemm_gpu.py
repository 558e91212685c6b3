"""GPU parity of the batched ternary GEMM (vx_gemm_i32_dev, MFMA i8) through the C ABI.

The reference has no multi-token kernel; its prefill calls the GEMV once per token (quintrit-runtime/src/engine.rs:
625-631), so the GEMM must equal M independent GEMVs bit for bit. Small shapes are checked against brute force; the
Falcon3-10B FFN shapes (W 23040 x 3072 and 3072 x 23040, M in {8, 32, 128, 512}) against a float64 brute
force of every output.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def gemm(torch, layer, x, ldx=None):
    from quintrit_amd import _lib
    L = _lib.lib()
    rows, cols = layer.shape()
    m = x.shape[0]
    ldx = ldx or cols
    xd = torch.zeros((m, ldx), dtype=torch.int8, device="cuda")
    xd[:, :cols] = torch.from_numpy(x).cuda()
    y = torch.full((m, rows), -7, dtype=torch.int32, device="cuda")
    n = ctypes.c_size_t()
    _lib.check(L.vx_gemm_workspace_bytes(layer.handle, m, ctypes.byref(n)))
    ws = torch.empty(n.value + 256, dtype=torch.uint8, device="cuda")
    base = (ws.data_ptr() + 255) // 256 * 256
    _lib.check(L.vx_gemm_i32_dev(layer.handle, ctypes.c_void_p(xd.data_ptr()), m, ldx, ctypes.c_void_p(y.data_ptr()),
                                 rows, ctypes.c_void_p(base), n.value,
                                 ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    return y.cpu().numpy()


@pytest.mark.parametrize("rows,cols,m", [(64, 160, 1), (1, 1, 3), (65, 161, 13), (130, 3072, 8), (1100, 321, 17),
                                         (200, 4096, 33), (3, 23040, 5), (1024, 3072, 64), (70, 2560, 100),
                                         (300, 6912, 40), (64, 23040, 64), (129, 1, 63), (65, 3200, 65),
                                         (1100, 6913, 97), (8192, 321, 128), (8193, 320, 128)])
def test_gemm_equals_bruteforce(torch_dev, oracle, rows, cols, m):
    from quintrit_amd import VelurexHipLayer
    print(f"[gemm bruteforce] {rows}x{cols} m={m}", flush=True)
    rng = np.random.default_rng(rows * 7 + cols * 3 + m)
    t = rng.integers(-1, 2, size=(rows, cols), dtype=np.int8)
    x = rng.integers(-128, 128, size=(m, cols), dtype=np.int8)
    layer = VelurexHipLayer(oracle.pack_matrix(t), rows, cols, 1.0)
    got = gemm(torch_dev, layer, x, ldx=cols + (cols % 3))
    want = (x.astype(np.float64) @ t.astype(np.float64).T).astype(np.int64)
    assert np.array_equal(got.astype(np.int64), want)
    layer.close()


def test_gemm_extreme_values(torch_dev, oracle):
    """All +1 / -1 weights times -128 / 127 activations: the largest magnitudes the int32 sums reach."""
    from quintrit_amd import VelurexHipLayer
    rows, cols, m = 64, 23040, 4
    for tv in (1, -1):
        t = np.full((rows, cols), tv, np.int8)
        layer = VelurexHipLayer(oracle.pack_matrix(t), rows, cols, 1.0)
        x = np.stack([np.full(cols, -128, np.int8), np.full(cols, 127, np.int8),
                      np.where(np.arange(cols) % 2 == 0, 127, -128).astype(np.int8), np.zeros(cols, np.int8)])
        got = gemm(torch_dev, layer, x)
        want = (x.astype(np.int64) @ t.astype(np.int64).T)
        assert np.array_equal(got.astype(np.int64), want)
        layer.close()


@pytest.mark.parametrize("rows,cols", [(23040, 3072), (3072, 23040)])
def test_gemm_config2_equals_bruteforce(torch_dev, oracle, rows, cols):
    """The Falcon3-10B FFN shapes: i.i.d. trits (P(-1)=P(+1)=0.35), X quantized per token from N(0,1). Every output of
    every M is compared with a float64 BLAS product of the unpacked trits, which is exact here: the operands are
    integers and every partial sum is at most 128 * 23040 < 2^53 in magnitude."""
    from quintrit_amd import VelurexHipLayer
    torch = torch_dev
    t = oracle.gen_trits(0xC2 + rows, (rows, cols))
    tf = t.astype(np.float64)
    layer = VelurexHipLayer(oracle.pack_matrix(t), rows, cols, 1.0)
    rng = np.random.default_rng(rows)
    for m in (8, 32, 48, 64, 128, 512):
        print(f"[gemm config2] {rows}x{cols} m={m}", flush=True)
        x = np.stack([oracle.quantize_i8(rng.standard_normal(cols).astype(np.float32))[0] for _ in range(m)])
        got = gemm(torch, layer, x)
        want = x.astype(np.float64) @ tf.T
        assert np.array_equal(got.astype(np.float64), want), m
    # one token through the GEMV as well: the two kernels agree
    out = torch.empty(rows, dtype=torch.int32, device="cuda")
    layer.gemv_i32(torch.from_numpy(x[5]).cuda(), out)
    assert np.array_equal(out.cpu().numpy(), got[5])
    layer.close()


@pytest.mark.parametrize("pad", [0, 3])  # rows of x in whole 16-byte pieces (where cols allows), and unaligned ones
@pytest.mark.parametrize("rows,cols,m", [(24000, 640, 480), (24001, 336, 511), (13824, 336, 500), (33000, 336, 64),
                                         (200, 2656, 90), (5000, 2672, 100), (60, 112, 33), (300, 14992, 200),
                                         (1000, 80, 129)])
def test_gemm_tiles(torch_dev, oracle, rows, cols, m, pad):
    """The tiled kernel (more than 32 tokens) on x itself (cols in whole 16-byte pieces) in each of its tiles, with and
    without K slices, at the edges of row blocks and token groups, with packed tails of one and of two chunks, against a
    float64 product (exact)."""
    check_gemm(torch_dev, oracle, rows, cols, m, cols + pad)


def check_gemm(torch, oracle, rows, cols, m, ldx):
    from quintrit_amd import VelurexHipLayer
    print(f"[gemm] {rows}x{cols} m={m} ldx={ldx}", flush=True)
    rng = np.random.default_rng(rows + cols + m)
    t = rng.integers(-1, 2, size=(rows, cols), dtype=np.int8)
    x = rng.integers(-128, 128, size=(m, cols), dtype=np.int8)
    layer = VelurexHipLayer(oracle.pack_matrix(t), rows, cols, 1.0)
    got = gemm(torch, layer, x, ldx=ldx)
    assert np.array_equal(got.astype(np.float64), x.astype(np.float64) @ t.astype(np.float64).T)
    layer.close()


# The plan on 256 CUs: tile (token groups, row blocks), K slices and steps, row groups.
@pytest.mark.parametrize("rows,cols,m", [(24001, 641, 480),     # 4 x 3, 63 row groups
                                         (13825, 337, 500),     # 4 x 1, 109 row groups
                                         (33000, 337, 64),      # 2 x 2, 129 row groups
                                         (12000, 5003, 60),     # 2 x 2, 4 slices of 8 steps, 47 row groups
                                         (5000, 14001, 500),    # 4 x 1, 3 slices of 30 steps, 40 row groups
                                         (3072, 23041, 512),    # 4 x 1, 5 slices of 29 steps, 24 row groups
                                         (300, 4003, 300),      # 2 x 1, 9 slices of 3 steps, 3 row groups
                                         (513, 12001, 200)])    # 2 x 1, 11 slices of 7 steps, 5 row groups
def test_gemm_tiles_staged(torch_dev, oracle, rows, cols, m):
    """The tiled kernel on fragments that the staging kernel has written (cols not a multiple of 16), in each of its tiles,
    with row groups below, in and beside whole eights, against a float64 product (exact)."""
    check_gemm(torch_dev, oracle, rows, cols, m, cols)


@pytest.mark.parametrize("rows,cols,m", [(3072, 20003, 40), (2500, 23043, 64), (6000, 9001, 49), (8192, 6912, 33),
                                         (1024, 3072, 16), (1024, 3072, 17), (300, 1600, 32), (1023, 1601, 31)])
def test_gemm_small_forms(torch_dev, oracle, rows, cols, m):
    """The small kernel with two token groups (long rows, 33 to 64 tokens, K slices of 6 steps or more), and with one on both
    sides of the token count from which a slice's sums are stored with the tokens in the lanes."""
    check_gemm(torch_dev, oracle, rows, cols, m, cols + 3)
