"""W8A8 FP8 GEMM (kc_gemm_fp8_w8a8_*) on the GPU against the oracle.

Y[m, n] = sx[m] sw[n] sum_k e4m3(qx[m, k]) e4m3(qw[n, k]).

The matrix core's accumulation is not IEEE fp32 (measured in-bounds on
MI355X): the products of each block of 8 consecutive k are aligned to the
block's largest product and truncated toward zero 14 bits below its leading
bit before the block sum joins the fp32 accumulator; E4M3 subnormals are
exact.  So:
  * integer-valued codes (|value| <= 16: products <= 2^8, truncation step
    <= 2^-6, every partial sum an integer below 2^24) are exact in any
    order, and the fp32 output must equal (float32(sum) * sx[m]) * sw[n]
    bit for bit -- this pins the operand and result layouts of the tiles;
  * codes over the whole finite E4M3 range: every element within the block
    truncation bound, 8 terms x 2^-13 of the block's largest |product|
    <= 2^-10 sum_k |product|, plus fp32 rounding; rel-L2 against the fp64
    oracle <= 2e-4 for fp32 output (about 5e-5 measured) and <= 1e-2 for
    bf16 output (bf16 rounding alone is ~2e-3).
Shapes cover tile tails in M, N and K (K only needs to be a multiple of 16).
An end-to-end case runs the quantizers' output through the GEMM."""
import ctypes

import numpy as np
import pytest

import kc_abi
from kc_abi import ptr, stream
from kc_data import bf16_bits_to_f32, f32_to_bf16_bits, normal_bf16, rel_l2

pytestmark = pytest.mark.gpu


def _dev(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _finite_codes(rng, shape):
    c = rng.integers(0, 256, shape, dtype=np.uint8)
    c[(c & 0x7F) == 0x7F] = 0x7E        # NaN codes -> 448
    return c.view(np.int8)


def _integer_codes(rng, shape, table):
    vals = np.array([c for c in range(256) if np.isfinite(table[c]) and abs(table[c]) <= 16
                     and table[c] == np.round(table[c])], np.uint8)
    return vals[rng.integers(0, vals.size, shape)].view(np.int8)


def _gemm(torch, qx, sx, qw, sw, bf16):
    M, K = qx.shape
    N = qw.shape[0]
    dqx, dsx, dqw, dsw = _dev(torch, qx), _dev(torch, sx), _dev(torch, qw), _dev(torch, sw)
    if bf16:
        y = torch.full((M, N), -7, dtype=torch.int16, device="cuda")
        fn = kc_abi.lib().kc_gemm_fp8_w8a8_bf16
    else:
        y = torch.full((M, N), float("nan"), dtype=torch.float32, device="cuda")
        fn = kc_abi.lib().kc_gemm_fp8_w8a8_f32
    print(f"kc_gemm_fp8_w8a8 {'bf16' if bf16 else 'f32'} M={M} N={N} K={K}", flush=True)
    st = fn(ptr(dqx), ptr(dsx), ptr(dqw), ptr(dsw), ptr(y), M, N, K, stream())
    kc_abi.check("kc_gemm_fp8_w8a8", st)
    out = y.cpu().numpy()
    return bf16_bits_to_f32(out.view(np.uint16)) if bf16 else out


SHAPES = [(128, 128, 128), (1, 1, 16), (16, 16, 128), (200, 300, 272), (37, 513, 1040),
          (256, 1024, 4096), (1000, 130, 48), (129, 129, 144), (512, 384, 8192), (300, 520, 400)]


def _integer_case(rng, oracle, M, N, K):
    """Integer-valued codes and the output they must give bit for bit in fp32."""
    table = oracle.e4m3_decode_table()
    qx = _integer_codes(rng, (M, K), table)
    qw = _integer_codes(rng, (N, K), table)
    sx = rng.uniform(0.001, 2.0, M).astype(np.float32)
    sw = rng.uniform(0.001, 2.0, N).astype(np.float32)
    acc = table[qx.view(np.uint8)].astype(np.float64) @ table[qw.view(np.uint8)].astype(np.float64).T
    assert np.abs(acc).max() < 2 ** 24
    want = (acc.astype(np.float32) * sx[:, None]) * sw[None, :]
    return qx, sx, qw, sw, want


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("bf16", [False, True])
def test_integer_codes_bit_exact(gpu, oracle, M, N, K, bf16):
    """fp32 Y equals the exact sum scaled as (acc * sx) * sw; bf16 Y is that
    value rounded to nearest even.  M <= 64 and the smallest tiles, with N %
    4 == 0 (four columns per lane), N % 2 == 0 (pairs at M <= 64) and the rest."""
    torch = gpu
    rng = np.random.default_rng(M * 7 + N * 3 + K)
    qx, sx, qw, sw, want = _integer_case(rng, oracle, M, N, K)
    y = _gemm(torch, qx, sx, qw, sw, bf16=bf16)
    if bf16:
        want = bf16_bits_to_f32(f32_to_bf16_bits(want))
    if not np.array_equal(y.view(np.uint32), want.view(np.uint32)):
        bad = np.argwhere(y.view(np.uint32) != want.view(np.uint32))
        m, n = bad[0]
        raise AssertionError(f"{len(bad)} mismatches; first at {(m, n)}: gpu {y[m, n]!r} "
                             f"want {want[m, n]!r}")


def _random_shapes(n, seed=2024):
    """Seeded shapes of M <= 64 and the smallest tiles: N a multiple of 8, of
    4 (four columns per lane) or neither, with M, N and K tails of every
    size."""
    rng = np.random.default_rng(seed)
    out = []
    for i in range(n):
        M = int(rng.integers(1, 700))
        N = int(rng.integers(1, 90)) * (8, 4, 1)[i % 3] + (0, 0, int(rng.integers(0, 8)))[i % 3]
        K = 16 * int(rng.integers(1, 70))
        out.append((M, max(N, 1), K))
    return out


@pytest.mark.parametrize("M,N,K", _random_shapes(12))
def test_random_shapes_bit_exact(gpu, oracle, M, N, K):
    """bf16 and fp32 Y on integer-valued codes, bit for bit, at seeded random
    shapes."""
    torch = gpu
    rng = np.random.default_rng(M * 131 + N * 17 + K)
    qx, sx, qw, sw, want = _integer_case(rng, oracle, M, N, K)
    for bf16 in (True, False):
        y = _gemm(torch, qx, sx, qw, sw, bf16=bf16)
        w = bf16_bits_to_f32(f32_to_bf16_bits(want)) if bf16 else want
        assert np.array_equal(y.view(np.uint32), w.view(np.uint32)), (M, N, K, bf16)


# Few tokens (M <= 64): one to four tiles of X, one / two / four weight tiles per
# workgroup (N up to 4096, 8192 and past it), seven from M 33 at N 16385 to
# 28672 and four again past it, odd N, K below one step, with a partial last
# step, and fewer or more steps than the waves of a workgroup.  Larger M: every
# tile of the small-grid kernel (32 x 64, 64 x 64, 64 x 128, 128 x 128, 256 x
# 128) with ragged M and N, and K of fewer, as many and more steps than its LDS
# buffers.
SMALL_GRIDS = [(1, 1, 16), (8, 15, 128), (9, 17, 144), (16, 33, 1040), (5, 40, 2048), (5, 41, 2064),
               (17, 4097, 272), (64, 4096, 1024), (64, 112, 4112), (1, 8200, 2064), (33, 8193, 144),
               (32, 16400, 400), (48, 16401, 272), (64, 16386, 528),
               (33, 28672, 144), (64, 28671, 272), (48, 28673, 272), (64, 32001, 144),
               # past it, where fp32 rows at short K run the 256 x 256 tiles
               (5, 34001, 128), (17, 34001, 384), (48, 34001, 640), (48, 34001, 656), (64, 32768, 512)]
SMALL_GRIDS += [(m, n, k) for m, n in ((65, 131), (200, 2704), (500, 2701), (1000, 2700), (1500, 3900))
                for k in (16, 272, 640, 1168, 2048)]
# K of two steps: two rounds of 256 x 256 tiles, not three of smaller ones
SMALL_GRIDS += [(1500, 14340, 144)]


@pytest.mark.parametrize("M,N,K", SMALL_GRIDS)
def test_small_grids_bit_exact(gpu, oracle, M, N, K):
    """fp32 and bf16 Y on integer-valued codes, bit for bit, where the 256 x
    256 tiles are not used, and at the edge of their use."""
    torch = gpu
    rng = np.random.default_rng(M * 13 + N * 7 + K)
    qx, sx, qw, sw, want = _integer_case(rng, oracle, M, N, K)
    for bf16 in (True, False):
        y = _gemm(torch, qx, sx, qw, sw, bf16=bf16)
        w = bf16_bits_to_f32(f32_to_bf16_bits(want)) if bf16 else want
        assert np.array_equal(y.view(np.uint32), w.view(np.uint32)), (M, N, K, bf16)


# The 256 x 256 tiles: grids that smaller tiles would take more rounds for.  M
# and N tails and whole tiles, N a multiple of 8 (bf16 rows staged through LDS),
# of 4 (four columns per lane) and odd, and K of a partial step only, one whole
# step, one and a tail, odd and even step counts.
BIG_TILES = [(2945, 2696, 16), (2945, 2700, 272), (3071, 2689, 128), (3072, 2816, 144), (500, 16520, 640),
             (512, 16516, 1040), (449, 16641, 400),
             # 49 to 64 tokens, short K, more columns than 28672
             (64, 40001, 272), (49, 50008, 144), (50, 34000, 1024), (64, 50000, 2064)]


@pytest.mark.parametrize("M,N,K", BIG_TILES)
def test_big_tiles_bit_exact(gpu, oracle, M, N, K):
    """fp32 and bf16 Y on integer-valued codes, bit for bit, on the 256 x 256
    tiles."""
    torch = gpu
    rng = np.random.default_rng(M * 5 + N * 3 + K)
    qx, sx, qw, sw, want = _integer_case(rng, oracle, M, N, K)
    for bf16 in (True, False):
        y = _gemm(torch, qx, sx, qw, sw, bf16=bf16)
        w = bf16_bits_to_f32(f32_to_bf16_bits(want)) if bf16 else want
        assert np.array_equal(y.view(np.uint32), w.view(np.uint32)), (M, N, K, bf16)


@pytest.mark.parametrize("M,N,K,kernel", [(m, n, k, "gemm_fp8_kernel<") for m, n, k in BIG_TILES + [(1500, 14340, 144)]] + [
    (64, 4096, 1024, "gemm_fp8_skinny_kernel<4, 1,"), (33, 8193, 144, "gemm_fp8_skinny_kernel<3, 4,"),
    (64, 28671, 272, "gemm_fp8_skinny_kernel<4, 7,"), (48, 28673, 272, "gemm_fp8_skinny_kernel<3, 4,"),
    (64, 33000, 1040, "gemm_fp8_skinny_kernel<4, 4,"), (48, 34001, 656, "gemm_fp8_skinny_kernel<3, 4,"),
    (64, 50000, 2176, "gemm_fp8_skinny_kernel<4, 4,"),
    (65, 131, 2048, "gemm_fp8_tile_kernel<2, 2, 1, 2,"), (200, 2704, 16, "gemm_fp8_tile_kernel<4, 2, 1, 2,"),
    (500, 2701, 16, "gemm_fp8_tile_kernel<4, 2, 1, 4,"), (1000, 2700, 2048, "gemm_fp8_tile_kernel<4, 2, 2, 4,"),
    (1500, 3900, 2048, "gemm_fp8_tile_kernel<4, 4, 4, 2,")])
def test_kernel_of_shape(gpu, M, N, K, kernel):
    """The shapes above run the kernel that they are there for."""
    torch = gpu
    q = torch.zeros(max(M, N) * K, dtype=torch.int8, device="cuda")
    s = torch.ones(max(M, N), device="cuda")
    y = torch.empty(M * N, dtype=torch.float32, device="cuda")
    for fn in (kc_abi.lib().kc_gemm_fp8_w8a8_bf16, kc_abi.lib().kc_gemm_fp8_w8a8_f32):
        names = kc_abi.kernels_of(lambda: kc_abi.check("kc_gemm_fp8_w8a8", fn(
            ptr(q), ptr(s), ptr(q), ptr(s), ptr(y), M, N, K, stream())))
        assert len(names) == 1 and kernel in names[0], names


@pytest.mark.parametrize("bf16,offset", [(True, 0), (True, 1), (True, 4), (False, 1), (False, 2),
                                          (False, 4)])
@pytest.mark.parametrize("M,N,K", [(200, 256, 272), (2945, 2696, 272), (9, 256, 272)])
def test_output_alignment(gpu, oracle, bf16, offset, M, N, K):
    """Y at an element offset inside a larger buffer (N % 8 == 0): the
    16-byte row stores of the 256 x 256 tiles need 16-byte alignment, the
    four-column stores (also those of the smaller tiles, 200 x 256) 8 (bf16) or
    16 (fp32) bytes, the column pairs of M <= 64 4 bytes; other offsets take
    the one-column path.  Bit-exact on integer codes, and nothing outside Y is
    written."""
    torch = gpu
    rng = np.random.default_rng(offset * 13 + bf16)
    qx, sx, qw, sw, want = _integer_case(rng, oracle, M, N, K)
    dqx, dsx, dqw, dsw = _dev(torch, qx), _dev(torch, sx), _dev(torch, qw), _dev(torch, sw)
    if bf16:
        buf = torch.full((M * N + 16,), -7, dtype=torch.int16, device="cuda")
        fn = kc_abi.lib().kc_gemm_fp8_w8a8_bf16
        want = f32_to_bf16_bits(want).view(np.int16)
    else:
        buf = torch.full((M * N + 16,), -7.0, dtype=torch.float32, device="cuda")
        fn = kc_abi.lib().kc_gemm_fp8_w8a8_f32
    print(f"kc_gemm_fp8_w8a8 {'bf16' if bf16 else 'f32'} M={M} N={N} K={K} y offset {offset}", flush=True)
    st = fn(ptr(dqx), ptr(dsx), ptr(dqw), ptr(dsw), buf.data_ptr() + offset * buf.element_size(), M, N, K,
            stream())
    kc_abi.check("kc_gemm_fp8_w8a8", st)
    out = buf.cpu().numpy()
    assert np.all(out[:offset] == -7) and np.all(out[offset + M * N:] == -7)
    got = out[offset:offset + M * N].reshape(M, N)
    assert np.array_equal(got.view(np.uint16 if bf16 else np.uint32), want.view(np.uint16 if bf16 else np.uint32))


@pytest.mark.parametrize("M,N,K", SHAPES + [(2945, 2696, 400)])
@pytest.mark.parametrize("bf16", [False, True])
def test_full_range_codes_vs_oracle(gpu, oracle, M, N, K, bf16):
    torch = gpu
    rng = np.random.default_rng(M + N * 5 + K * 11 + bf16)
    qx = _finite_codes(rng, (M, K))
    qw = _finite_codes(rng, (N, K))
    sx = rng.uniform(1e-4, 1e-2, M).astype(np.float32)
    sw = rng.uniform(1e-4, 1e-2, N).astype(np.float32)
    y = _gemm(torch, qx, sx, qw, sw, bf16)
    truth = oracle.gemm_fp8_w8a8_f64(qx, sx, qw, sw)
    assert np.all(np.isfinite(y))
    err = rel_l2(y, truth)
    assert err <= (1e-2 if bf16 else 2e-4), err
    if not bf16:
        table = np.abs(oracle.e4m3_decode_table().astype(np.float64))
        mag = (table[qx.view(np.uint8)] @ table[qw.view(np.uint8)].T) * sx[:, None] * sw[None, :]
        bound = 2.0 ** -10 * mag + 2.0 ** -22 * np.abs(truth) + 1e-30
        worst = np.max(np.abs(y - truth) / bound)
        assert worst <= 1.0, worst


def test_quantized_linear_end_to_end(gpu, oracle):
    """bf16 X [64, 4096] per token and W [1024, 4096] per channel through the
    GPU quantizer, then the GEMM: equal to the oracle on the same codes, and
    within FP8's error of the unquantized product."""
    torch = gpu
    M, N, K = 64, 1024, 4096
    xb = normal_bf16((M, K), seed=31)
    wb = normal_bf16((N, K), seed=32, std=0.02)
    L = kc_abi.lib()

    def quant(bits):
        rows, cols = bits.shape
        d = _dev(torch, bits.view(np.int16))
        q = torch.empty(rows, cols, dtype=torch.int8, device="cuda")
        s = torch.empty(rows, dtype=torch.float32, device="cuda")
        print(f"kc_quantize_fp8_per_token_bf16 rows={rows} cols={cols}", flush=True)
        st = L.kc_quantize_fp8_per_token_bf16(ptr(d), ptr(q), ptr(s), rows, cols, stream())
        kc_abi.check("kc_quantize_fp8_per_token_bf16", st)
        return q.cpu().numpy(), s.cpu().numpy()

    qx, sx = quant(xb)
    qw, sw = quant(wb)
    eqx, esx = oracle.quantize_fp8_per_token_bf16(xb)
    np.testing.assert_array_equal(qx, eqx)
    np.testing.assert_array_equal(sx, esx)
    y = _gemm(torch, qx, sx, qw, sw, bf16=True)
    truth = oracle.gemm_fp8_w8a8_f64(qx, sx, qw, sw)
    assert rel_l2(y, truth) < 1e-2
    exact = bf16_bits_to_f32(xb).astype(np.float64) @ bf16_bits_to_f32(wb).astype(np.float64).T
    assert rel_l2(y, exact) < 0.08


def test_argument_errors(gpu):
    L = kc_abi.lib()
    d = ctypes.c_void_p(256)
    for M, N, K, p in [(4, 4, 24, d), (-1, 4, 16, d), (4, 4, 16, None)]:
        st = L.kc_gemm_fp8_w8a8_f32(p, d, d, d, d, M, N, K, None)
        assert st == 1, (M, N, K)
        L.kc_get_last_error()
    st = L.kc_gemm_fp8_w8a8_bf16(ctypes.c_void_p(258), d, d, d, d, 4, 4, 16, None)
    assert st == 1
    L.kc_get_last_error()
    assert L.kc_gemm_fp8_w8a8_bf16(d, d, d, d, d, 0, 4, 16, None) == 0


@pytest.mark.parametrize("bf16", [True, False])
def test_empty_contraction_writes_zeros(gpu, bf16):
    """K == 0: Y is the empty sum, 0, for every (m, n); the GEMM kernel (whose
    prologue always loads a first K step) is not launched."""
    torch = gpu
    L = kc_abi.lib()
    M, N = 37, 301   # M * N odd: the last element is a lone half word in bf16
    dt = torch.bfloat16 if bf16 else torch.float32
    y = torch.full((M, N), 7.0, dtype=dt, device="cuda")
    sx = torch.ones(M, device="cuda")
    sw = torch.ones(N, device="cuda")
    qx = torch.empty(M, 0, dtype=torch.int8, device="cuda")
    qw = torch.empty(N, 0, dtype=torch.int8, device="cuda")
    fn = L.kc_gemm_fp8_w8a8_bf16 if bf16 else L.kc_gemm_fp8_w8a8_f32
    for _ in range(2):
        st = fn(ptr(qx), ptr(sx), ptr(qw), ptr(sw), ptr(y), M, N, 0, stream())
        assert st == 0, L.kc_last_error_string()
        torch.cuda.synchronize()
        assert torch.count_nonzero(y).item() == 0
        y.fill_(-3.0)
