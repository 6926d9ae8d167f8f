// fp8_gemm_small.hip -- the FP8 W8A8 GEMM (see fp8_gemm.hip) where 256 x 256
// tiles leave most of the 256 CUs idle: a decode batch (M <= 64), and grids
// of few tiles.  Y[m, n] = sx[m] sw[n] sum_k e4m3(qx[m,k]) e4m3(qw[n,k]).
//
// M <= 64: gemm_fp8_skinny_kernel, bound by the weight stream.  256 x 256
// tiles ran 16 to 112 workgroups there, each walking all of K alone, for
// whatever M: N 6144, K 4096 53 us, now 7.8 / 9.1 / 10.5 us at M 16 / 32 / 48;
// N 4096, K 14336 161 us, now 13 / 17 / 24 us at M 16 / 32 / 64; N 28672,
// K 8192 105 us, now 37 / 52 us at M 8 / 64 (235 MB: 33 us at 7 TB/s).
// Larger M: gemm_fp8_tile_kernel, with the tile that the table at the bottom
// expects to finish first.
#include <algorithm>
#include <type_traits>

#include "fp8_gemm.hpp"

namespace {

using namespace kc::fp8;

constexpr int kSkinnyM = 64;
constexpr int kGroupM = 4;

// ---------------------------------------------------------------------------
// M <= 64.  A workgroup of KW waves owns RT tiles of 16 weight rows and all
// MT = ceil(M / 16) tiles of X; wave w takes K steps w, w + KW, ... of 128
// bytes, D of them in flight in registers, and the KW partial sums of every
// output meet in LDS in a fixed order.  No barrier stands in the K loop, and
// neither operand goes through LDS: with K split over the waves no two of
// them read the same bytes.
// ---------------------------------------------------------------------------
// One 128-byte K step of 16 rows in registers: load h (0, 1) reads 8 whole
// rows, lane l taking 16-byte chunk 2 (l / 16) + l % 2 of row 8 h + (l % 16) / 2,
// so that each load touches 8 cache lines, all of each.  The operand's own
// layout (64 bytes of each of 16 rows per load) reads 20-25 % slower from HBM
// and holds the load unit about twice as long (N 4096, K 14336, M 16: 19.3 us).
struct Frag {
    u32x4 h0, h1;
};

// The matrix-core operand of a step: lane (i, kb) needs 32 bytes of one row.
// A lane and its neighbour l ^ 1 hold two chunks of two rows; the even lane
// keeps row (l % 16) / 2, the odd lane row 8 + (l % 16) / 2, both chunks in
// order (one select with a quad permutation per dword).  Operand row i is
// then tile row row_of(i) = i / 2 + 8 (i % 2).
__device__ __forceinline__ uint32_t swap_pair(uint32_t v) {  // lane l reads lane l ^ 1
    return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(v), 0xB1, 0xF, 0xF, true));
}

__device__ __forceinline__ i32x8 as_operand(const Frag& f, bool even) {
    const uint32_t a[4] = {f.h0.x, f.h0.y, f.h0.z, f.h0.w}, b[4] = {f.h1.x, f.h1.y, f.h1.z, f.h1.w};
    i32x8 o;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        const uint32_t an = swap_pair(a[d]), bn = swap_pair(b[d]);
        o[d] = static_cast<int32_t>(even ? a[d] : bn);
        o[4 + d] = static_cast<int32_t>(even ? an : b[d]);
    }
    return o;
}

template <int MT, int RT, int KW, int D, bool YBF16>
__global__ __launch_bounds__(KW * 64) void gemm_fp8_skinny_kernel(
    const int8_t* __restrict__ qx, const float* __restrict__ sx, const int8_t* __restrict__ qw,
    const float* __restrict__ sw, void* __restrict__ y, int M, int N, int K, bool vec) {
    __shared__ f32x4 red[KW][RT * MT][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int i = lane & 15, kb = lane >> 4;
    const bool even = (lane & 1) == 0;
    const int n0 = static_cast<int>(blockIdx.x) * 16 * RT;
    const int8_t* wbase = qw + static_cast<int64_t>(n0) * K;
    const int chunk = 2 * kb + (i & 1), r8 = i >> 1;
    uint32_t woff[RT][2], xoff[MT][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int r = 0; r < RT; ++r)
            woff[r][h] = static_cast<uint32_t>(min(n0 + 16 * r + 8 * h + r8, N - 1) - n0) * static_cast<uint32_t>(K) + 16u * chunk;
#pragma unroll
        for (int c = 0; c < MT; ++c)
            xoff[c][h] = static_cast<uint32_t>(min(16 * c + 8 * h + r8, M - 1)) * static_cast<uint32_t>(K) + 16u * chunk;
    }

    f32x4 acc[RT][MT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int c = 0; c < MT; ++c) acc[r][c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const int full = K / kBK;
    const int mine = full > wave ? (full - wave + KW - 1) / KW : 0;  // K steps wave, wave + KW, ...

    Frag wf[D][RT], xf[D][MT];
    auto load = [&](int slot, int j) {
        const int64_t k = static_cast<int64_t>(wave + KW * min(j, mine - 1)) * kBK;
        const int8_t* wp = wbase + k;
        const int8_t* xp = qx + k;
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            wf[slot][r].h0 = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wp + woff[r][0]));
            wf[slot][r].h1 = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wp + woff[r][1]));
        }
#pragma unroll
        for (int c = 0; c < MT; ++c) {
            xf[slot][c].h0 = *reinterpret_cast<const u32x4*>(xp + xoff[c][0]);
            xf[slot][c].h1 = *reinterpret_cast<const u32x4*>(xp + xoff[c][1]);
        }
    };
    auto multiply = [&](const Frag (&w)[RT], const Frag (&x)[MT]) {
        i32x8 b[MT];
#pragma unroll
        for (int c = 0; c < MT; ++c) b[c] = as_operand(x[c], even);
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const i32x8 a = as_operand(w[r], even);
#pragma unroll
            for (int c = 0; c < MT; ++c)
                acc[r][c] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b[c], acc[r][c], 0, 0, 0,
                                                                             kE8M0One, 0, kE8M0One);
        }
    };
    // the scales of the tiles this wave finishes, ahead of the operand loads
    constexpr int kFin = (RT * MT + KW - 1) / KW;
    float fsx[kFin], fsw[kFin][4];
#pragma unroll
    for (int u = 0; u < kFin; ++u) {
        const int t = min(wave + u * KW, RT * MT - 1);
        fsx[u] = sx[min(16 * (t % MT) + (i >> 1) + 8 * (i & 1), M - 1)];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            fsw[u][e] = sw[min(n0 + 16 * (t / MT) + 2 * kb + (e & 1) + 8 * (e >> 1), N - 1)];
    }
    if (mine > 0) {
#pragma unroll
        for (int d = 0; d < D; ++d) load(d, d);
        __builtin_amdgcn_sched_barrier(0);
        int j = 0;
        for (; j + D < mine; j += D) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                multiply(wf[d], xf[d]);
                load(d, j + D + d);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int d = 0; d < D; ++d)
            if (j + d < mine) multiply(wf[d], xf[d]);
    }
    if (K % kBK != 0 && wave == full % KW) {  // the partial last step
        const int kvalid = K - full * kBK;
        auto tail = [&](const int8_t* base, const uint32_t (&off)[2]) {
            const u32x4 z{0u, 0u, 0u, 0u};
            Frag f{z, z};
            if (16 * chunk < kvalid) {
                f.h0 = *reinterpret_cast<const u32x4*>(base + static_cast<int64_t>(full) * kBK + off[0]);
                f.h1 = *reinterpret_cast<const u32x4*>(base + static_cast<int64_t>(full) * kBK + off[1]);
            }
            return f;
        };
        Frag w[RT], x[MT];
#pragma unroll
        for (int r = 0; r < RT; ++r) w[r] = tail(wbase, woff[r]);
#pragma unroll
        for (int c = 0; c < MT; ++c) x[c] = tail(qx, xoff[c]);
        multiply(w, x);
    }
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int c = 0; c < MT; ++c) red[wave][r * MT + c][lane] = acc[r][c];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kFin; ++u) {
        const int t = wave + u * KW;
        if (t >= RT * MT) break;
        f32x4 v = red[0][t][lane];
#pragma unroll
        for (int w = 1; w < KW; ++w) {
            const f32x4 o = red[w][t][lane];
            v = f32x4{v.x + o.x, v.y + o.y, v.z + o.z, v.w + o.w};
        }
        // D: lane (i, g) holds operand rows 4 g + v of W, column i of X, that is
        // outputs n = 2 g, 2 g + 8, 2 g + 1, 2 g + 9 (v = 0 .. 3) of row row_of(i)
        const int m = 16 * (t % MT) + (i >> 1) + 8 * (i & 1);
        if (m >= M) continue;
        const float sxm = fsx[u];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int n = n0 + 16 * (t / MT) + 2 * kb + 8 * h;
            if (n >= N) break;
            const float v0 = ((h ? v.y : v.x) * sxm) * fsw[u][2 * h];
            const int64_t at = static_cast<int64_t>(m) * N + n;
            if (vec || n + 1 < N) {
                const float v1 = ((h ? v.w : v.z) * sxm) * fsw[u][2 * h + 1];
                if constexpr (YBF16) {
                    const uint32_t lo = kc::f32_to_bf16(v0), hi = kc::f32_to_bf16(v1);
                    if (vec) *reinterpret_cast<uint32_t*>(static_cast<uint16_t*>(y) + at) = lo | hi << 16;
                    else static_cast<uint16_t*>(y)[at] = lo, static_cast<uint16_t*>(y)[at + 1] = hi;
                } else {
                    static_cast<float*>(y)[at] = v0;
                    static_cast<float*>(y)[at + 1] = v1;
                }
            } else {
                if constexpr (YBF16) static_cast<uint16_t*>(y)[at] = kc::f32_to_bf16(v0);
                else static_cast<float*>(y)[at] = v0;
            }
        }
    }
}

template <int MT, int RT, int KW, int D, bool YBF16>
int launch_skinny(const char* fn, const int8_t* qx, const float* sx, const int8_t* qw, const float* sw, void* y, int M,
                  int N, int K, hipStream_t stream) {
    gemm_fp8_skinny_kernel<MT, RT, KW, D, YBF16><<<static_cast<unsigned>((N + 16 * RT - 1) / (16 * RT)), KW * 64, 0, stream>>>(
        qx, sx, qw, sw, y, M, N, K, N % 2 == 0 && kc::aligned(y, 4));
    return kc::check_launch(fn);
}

// Row tiles per workgroup: one, two or four, the fewest that leave at most one
// workgroup per CU, since every workgroup reads all of X (M 32, K 4096: N 6144
// 11.5 us at one tile, 9.1 at two; N 28672 37.5 at one, 27.8 at two, 24.5 at
// four); four beyond, two of them on a CU.  Seven with three or four tiles of X
// to share, while they fill one round of the CUs (N 16385 to 28672): M 64,
// K 8192 54.0 -> 44.0 us at N 17000, 55.5 -> 44.4 at 20480, 61.5 -> 49.0 at 28672,
// M 48, K 4096 26.3 -> 24.0, 27.3 -> 24.7, 29.8 -> 29.2 (only where four leave a
// 257th workgroup or so they gain nothing: N 16400 22.0 -> 23.6, M 64 27.9 -> 26.6);
// with a second round they lose (M 64, K 8192 62.0 us at four against 80.4 at seven at N 28800, 65.2 against
// 86.0 at 32768), and with two tiles of X too (M 32, N 28672, K 4096 24.5 against
// 29.4).  At one tile, eight waves with one tile of X and four with more (M 16,
// N 4096, K 4096 5.9 against 6.8 us; M 32, K 14336 18.1 against 16.9); two steps
// in flight instead of four where a wave has no more (N 1024, K 1024 5.5 -> 4.4).
template <int MT, bool YBF16>
int skinny(const char* fn, const int8_t* qx, const float* sx, const int8_t* qw, const float* sw, void* y, int M, int N,
           int K, hipStream_t stream) {
    constexpr int kRowsPerTile = 16 * 256;
    constexpr int kw = MT == 1 ? 8 : 4;
    if (N <= kRowsPerTile) {
        if (K <= 2 * kw * kBK) return launch_skinny<MT, 1, kw, 2, YBF16>(fn, qx, sx, qw, sw, y, M, N, K, stream);
        return launch_skinny<MT, 1, kw, 4, YBF16>(fn, qx, sx, qw, sw, y, M, N, K, stream);
    }
    if (N <= 2 * kRowsPerTile) return launch_skinny<MT, 2, 8, 2, YBF16>(fn, qx, sx, qw, sw, y, M, N, K, stream);
    if constexpr (MT >= 3) {
        if (N > 4 * kRowsPerTile && N <= 7 * kRowsPerTile)
            return launch_skinny<MT, 7, 4, 1, YBF16>(fn, qx, sx, qw, sw, y, M, N, K, stream);
    }
    return launch_skinny<MT, 4, 4, 2, YBF16>(fn, qx, sx, qw, sw, y, M, N, K, stream);
}

// Past N 28672 a short K leaves each of the many workgroups above little but its
// start and its sum through LDS, and 256 x 256 tiles are faster again, the more so
// the fuller their rounds of 256 tiles (65536 columns) are; K that is no multiple
// of 128 costs the kernel above, whose loads then straddle cache lines, about 20 %
// more than the large tiles.  M 49 to 64, bf16: N 40000 16.0 -> 12.9 us at K 256 and
// level from 1024, N 64000 32.7 -> 27.5 at K 1024, 3 % at 2048, and with K 2064 to
// 6160 15 to 20 %; N 90000 level from 1024.  Fewer tokens only where fp32 rows are
// stored (M 48, N 64000, K 512 bf16 8 % faster here, fp32 7 % slower; M 33, N 40000, K 624
// 22 % slower, M 16, N 64000, K 128 12 %).  N 28673 to 32768 at K 256 fp32, M 64 21 %.
template <bool YBF16>
bool large_tiles_at_short_k(int mt, int N, int K) {
    constexpr int64_t kRound = 256 * 256;  // columns of a round of large tiles
    if (N <= 28672) return false;
    const bool whole = K % kBK == 0;
    const int64_t fill = 100 * int64_t{N} / ((N + kRound - 1) / kRound * kRound);  // per cent
    if (mt == 4) {
        if (fill <= 50) return !YBF16 && K <= 512;
        if (fill <= 70) return K <= (whole ? 1024 : 1600);
        return !whole || K <= 2048;
    }
    if (YBF16 || fill <= 50) return false;
    if (mt == 1) return K <= 128;
    return K <= (whole ? 256 * mt - 128 : fill <= 70 ? 640 : 1600);
}

// ---------------------------------------------------------------------------
// M > 64.  A workgroup computes a tile of 16 TM WGM x 16 TN WGN outputs with
// KG groups of WGM x WGN waves; group g takes K steps g, g + KG, ... and the
// groups' sums meet in LDS at the end (each group finishes 1 / KG of the
// rows).  As in the 256 x 256 kernel the steps go from global memory straight
// into LDS (rows of 128 bytes, chunks XOR-swizzled by row), here through ST
// buffers per group, and one barrier per step publishes them; but the
// operands of step it + 1 are read into registers while step it is
// multiplied, so a buffer is free for step it + ST as soon as its barrier has
// passed, and no MFMA waits for LDS.  The loads and the operand reads are
// spread over the MFMAs.  Bound by how fast the steps arrive from L2: 128 x 128
// tiles of 1000 x 4096 x 14336 read 933 MB there in 65 to 68 us a call (14 TB/s;
// 57 us with the operands already in L2, 38 us without loads and reads), 64 x 64
// of 256 x 4096 x 14336 474 MB in 36.5 (13 TB/s); the matrix cores are 34 and 14 %
// busy.  The first calls after an idle GPU take 73 to 82 us.
// ---------------------------------------------------------------------------
template <int TM, int TN, int WGM, int WGN, int KG, int ST>
struct TileShape {
    static constexpr int kRowsM = 16 * TM * WGM, kRowsN = 16 * TN * WGN;
    static constexpr int kWavesG = WGM * WGN;          // waves of one K group
    static constexpr int kThreadsT = 64 * kWavesG * KG;
    static constexpr int kStage = (kRowsM + kRowsN) * kBK;
    static constexpr int kLoads = (kRowsM + kRowsN) / 8 / kWavesG;  // per wave and stage
    static constexpr int kScales = KG * ST * kStage;
    static constexpr int kLds = kScales + (kRowsM + kRowsN) * 4;
};

// lds_dma16 from a scalar base and a 32-bit lane offset.
__device__ __forceinline__ void lds_dma16s(uint32_t voff, const void* sbase, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "s"(lds_base)
                 : "memory", "m0");
}

// Lane offsets of one wave's loads of a step (ROWS rows of 128 bytes, WAVES
// waves): load i carries rows 8 (kPer wave + i) .. + 7 of the tile, lane l row
// l / 8 of them, chunk (l % 8) ^ swizzle(row); rows past `rows` read the last
// one, chunks past `valid` bytes of the step the last valid chunk.
template <int ROWS, int WAVES>
__device__ __forceinline__ void row_offsets(uint32_t (&off)[ROWS / 8 / WAVES], int rows, uint32_t K, int wave, int lane,
                                            int valid) {
    constexpr int kPer = ROWS / 8 / WAVES;
    static_assert(kPer * 8 * WAVES == ROWS, "whole loads per wave");
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const int row = 8 * (kPer * wave + i) + (lane >> 3);
        const int chunk = (lane & 7) ^ swizzle(row);
        off[i] = static_cast<uint32_t>(min(row, rows - 1)) * K + static_cast<uint32_t>(min(16 * chunk, valid - 16));
    }
}

template <int TM, int TN, int WGM, int WGN, int KG, int ST, bool YBF16>
__global__ __launch_bounds__(64 * WGM * WGN * KG) void gemm_fp8_tile_kernel(
    const int8_t* __restrict__ qx, const float* __restrict__ sx, const int8_t* __restrict__ qw,
    const float* __restrict__ sw, void* __restrict__ y, int64_t M, int64_t N, int64_t K,
    int tiles_m, int tiles_n, bool vec) {
    using S = TileShape<TM, TN, WGM, WGN, KG, ST>;
    extern __shared__ __align__(16) uint8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int kg = wave / S::kWavesG, wg = wave % S::kWavesG;
    const int wm = wg / WGN, wn = wg % WGN;
    const int b = blockIdx.x, nb = gridDim.x;
    const int x = b % 8, q = nb / 8, r = nb % 8;
    const int lin = x * q + min(x, r) + b / 8;
    const int per_group = kGroupM * tiles_n;
    const int first_m = (lin / per_group) * kGroupM;
    const int group_m = min(tiles_m - first_m, kGroupM);
    const int tm = first_m + (lin % per_group) % group_m;
    const int tn = (lin % per_group) / group_m;
    const int64_t m0 = static_cast<int64_t>(tm) * S::kRowsM, n0 = static_cast<int64_t>(tn) * S::kRowsN;

    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    asm volatile("" ::"s"(y), "s"(sx), "s"(sw));
    const int full = static_cast<int>(K / kBK);
    const int kvalid = static_cast<int>(K - static_cast<int64_t>(full) * kBK);
    const int steps = full + (kvalid != 0);
    const int iters = (steps + KG - 1) / KG;  // K step s = KG it + kg
    float* scl = reinterpret_cast<float*>(lds + S::kScales);
    for (int t = threadIdx.x; t < S::kRowsM + S::kRowsN; t += S::kThreadsT) {
        const int64_t si = t < S::kRowsM ? m0 + t : n0 + (t - S::kRowsM);
        scl[t] = t < S::kRowsM ? (si < M ? sx[si] : 0.0f) : (si < N ? sw[si] : 0.0f);
    }
    // K step s = KG it + kg; steps past the end load the last one (not multiplied)
    constexpr int kPerM = S::kRowsM / 8 / S::kWavesG, kPerN = S::kRowsN / 8 / S::kWavesG;
    uint8_t* buf = lds + kg * ST * S::kStage;
    const uint32_t lds0 = lds_address(buf);
    const int8_t* xbase = qx + m0 * K;
    const int8_t* wbase = qw + n0 * K;
    const int xrows = static_cast<int>(min(M - m0, int64_t{S::kRowsM})), wrows = static_cast<int>(min(N - n0, int64_t{S::kRowsN}));
    uint32_t xo[kPerM], wo[kPerN];
    row_offsets<S::kRowsM, S::kWavesG>(xo, xrows, static_cast<uint32_t>(K), wg, lane, kBK);
    row_offsets<S::kRowsN, S::kWavesG>(wo, wrows, static_cast<uint32_t>(K), wg, lane, kBK);
    auto load = [&](int it) {
        const int s = min(KG * it + kg, steps - 1);
        const int64_t k0 = static_cast<int64_t>(s) * kBK;
        const uint32_t st = __builtin_amdgcn_readfirstlane(lds0 + (it % ST) * S::kStage);
        if (s < full) {
#pragma unroll
            for (int i = 0; i < kPerM; ++i) lds_dma16s(xo[i], xbase + k0, st + 1024 * (kPerM * wg + i));
#pragma unroll
            for (int i = 0; i < kPerN; ++i) lds_dma16s(wo[i], wbase + k0, st + S::kRowsM * kBK + 1024 * (kPerN * wg + i));
        } else {
            uint32_t xt[kPerM], wt[kPerN];
            row_offsets<S::kRowsM, S::kWavesG>(xt, xrows, static_cast<uint32_t>(K), wg, lane, kvalid);
            row_offsets<S::kRowsN, S::kWavesG>(wt, wrows, static_cast<uint32_t>(K), wg, lane, kvalid);
#pragma unroll
            for (int i = 0; i < kPerM; ++i) lds_dma16s(xt[i], xbase + k0, st + 1024 * (kPerM * wg + i));
#pragma unroll
            for (int i = 0; i < kPerN; ++i) lds_dma16s(wt[i], wbase + k0, st + S::kRowsM * kBK + 1024 * (kPerN * wg + i));
        }
    };
    struct Ops {
        i32x8 a[TM], b[TN];
    };
    auto read = [&](Ops& o, int it) {
        const uint8_t* st = buf + (it % ST) * S::kStage;
#pragma unroll
        for (int j = 0; j < TN; ++j) o.b[j] = read_operand<false>(st + S::kRowsM * kBK, 16 * TN * wn + 16 * j, lane, kBK);
#pragma unroll
        for (int i = 0; i < TM; ++i) o.a[i] = read_operand<false>(st, 16 * TM * wm + 16 * i, lane, kBK);
    };
    auto multiply = [&](const Ops& o) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(o.b[j], o.a[i], acc[i][j], 0, 0, 0,
                                                                             kE8M0One, 0, kE8M0One);
    };
#pragma unroll
    for (int p = 0; p < ST; ++p)
        if (p < iters) load(p);
    const int whole = full / KG;  // iterations in which every K group has a full step
    // stage `it` of every wave landed, stage it - 1 read by every wave
    auto publish = [&](int it, int younger) {
        if (younger >= ST - 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(S::kLoads * (ST - 1)) : "memory");
        else if (ST > 2 && younger == ST - 2) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(S::kLoads * (ST - 2)) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };
    Ops o[2];
    if (whole > 0) {
        publish(0, min(iters, ST) - 1);
        read(o[0], 0);
    }
    // iteration it: step it is in registers; step it + 1 is read while it is
    // multiplied, and its buffer then takes step it + ST
    auto step = [&](Ops& cur, Ops& nxt, int it) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(S::kLoads * (ST - 2)) : "memory");
        const int64_t k0 = static_cast<int64_t>(KG * (it + ST) + kg) * kBK;
        const uint32_t st = __builtin_amdgcn_readfirstlane(lds0 + (it % ST) * S::kStage);
        const uint8_t* rd = buf + ((it + 1) % ST) * S::kStage;
        // the loads into LDS and the operand reads spread over the MFMAs: a
        // load holds its wave until the memory pipe takes it
        constexpr int kM = TM * TN, kR = TM + TN, kL = kPerM + kPerN;
#pragma unroll
        for (int q = 0; q < kM; ++q) {
            const int i = q / TN, j = q % TN;
            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(cur.b[j], cur.a[i], acc[i][j], 0, 0, 0,
                                                                         kE8M0One, 0, kE8M0One);
#pragma unroll
            for (int u = q * kR / kM; u < (q + 1) * kR / kM; ++u) {
                if (u < TN) nxt.b[u] = read_operand<false>(rd + S::kRowsM * kBK, 16 * TN * wn + 16 * u, lane, kBK);
                else nxt.a[u - TN] = read_operand<false>(rd, 16 * TM * wm + 16 * (u - TN), lane, kBK);
            }
#pragma unroll
            for (int u = q * kL / kM; u < (q + 1) * kL / kM; ++u) {
                if (u < kPerM) lds_dma16s(xo[u], xbase + k0, st + 1024 * (kPerM * wg + u));
                else lds_dma16s(wo[u - kPerM], wbase + k0, st + S::kRowsM * kBK + 1024 * (kPerN * wg + u - kPerM));
            }
        }
    };
    int it = 0;
    for (; it + ST + 1 < whole; it += 2) {
        step(o[0], o[1], it);
        step(o[1], o[0], it + 1);
    }
    for (; it < whole; ++it) {  // the last steps
        multiply(o[0]);
        if (it + 1 < whole) {
            publish(it + 1, 0);
            if (it + ST < iters) load(it + ST);
            read(o[0], it + 1);
        }
    }
    if (whole < iters) {
        publish(whole, 0);
        const int s = KG * whole + kg;
        const uint8_t* st = buf + (whole % ST) * S::kStage;
        if (s < full) {
            read(o[0], whole);
            multiply(o[0]);
        } else if (s < steps) {
#pragma unroll
            for (int j = 0; j < TN; ++j) o[0].b[j] = read_operand<true>(st + S::kRowsM * kBK, 16 * TN * wn + 16 * j, lane, kvalid);
#pragma unroll
            for (int i = 0; i < TM; ++i) o[0].a[i] = read_operand<true>(st, 16 * TM * wm + 16 * i, lane, kvalid);
            multiply(o[0]);
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    // K groups: each finishes its share of the A blocks
    constexpr int kOwn = TM / KG;
    static_assert(kOwn * KG == TM, "A blocks split over the K groups");
    if constexpr (KG > 1) {
        f32x4* red = reinterpret_cast<f32x4*>(lds);  // [from][to][wave][kOwn TN][lane]
#pragma unroll
        for (int g = 0; g < KG; ++g) {
            if (g == kg) continue;
#pragma unroll
            for (int i = 0; i < kOwn; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    red[(((kg * KG + g) * S::kWavesG + wg) * kOwn * TN + i * TN + j) * 64 + lane] = acc[g * kOwn + i][j];
        }
        __syncthreads();
    }
    auto store = [&](auto group) {
        constexpr int G = decltype(group)::value;
        const int j16 = lane & 15, g = lane >> 4;
#pragma unroll
        for (int i = 0; i < kOwn; ++i) {
            const int rl = 16 * TM * wm + 16 * (G * kOwn + i) + j16;
            const int64_t m = m0 + rl;
            const float sxm = scl[rl];
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                f32x4 v = acc[G * kOwn + i][j];
                if constexpr (KG > 1) {
                    const f32x4* red = reinterpret_cast<const f32x4*>(lds);
#pragma unroll
                    for (int o = 0; o < KG; ++o) {
                        if (o == G) continue;
                        const f32x4 w = red[(((o * KG + G) * S::kWavesG + wg) * kOwn * TN + i * TN + j) * 64 + lane];
                        v = f32x4{v.x + w.x, v.y + w.y, v.z + w.z, v.w + w.w};
                    }
                }
                const int nl = 16 * TN * wn + 16 * j + 4 * g;
                const int64_t n = n0 + nl;
                if (m >= M) continue;
                const f32x4 s4 = *reinterpret_cast<const f32x4*>(scl + S::kRowsM + nl);
                const float rv[4] = {(v.x * sxm) * s4.x, (v.y * sxm) * s4.y, (v.z * sxm) * s4.z, (v.w * sxm) * s4.w};
                if (vec && n + 3 < N) {
                    if constexpr (YBF16) {
                        const uint32_t lo = kc::f32_to_bf16(rv[0]) | static_cast<uint32_t>(kc::f32_to_bf16(rv[1])) << 16;
                        const uint32_t hi = kc::f32_to_bf16(rv[2]) | static_cast<uint32_t>(kc::f32_to_bf16(rv[3])) << 16;
                        *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(y) + m * N + n) = u32x2{lo, hi};
                    } else {
                        *reinterpret_cast<f32x4*>(static_cast<float*>(y) + m * N + n) = f32x4{rv[0], rv[1], rv[2], rv[3]};
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if (n + e >= N) break;
                        if constexpr (YBF16) static_cast<uint16_t*>(y)[m * N + n + e] = kc::f32_to_bf16(rv[e]);
                        else static_cast<float*>(y)[m * N + n + e] = rv[e];
                    }
                }
            }
        }
    };
    if constexpr (KG == 1) {
        store(std::integral_constant<int, 0>{});
    } else if constexpr (KG == 2) {
        if (kg == 0) store(std::integral_constant<int, 0>{});
        else store(std::integral_constant<int, 1>{});
    } else {
        static_assert(KG == 4, "K groups");
        if (kg == 0) store(std::integral_constant<int, 0>{});
        else if (kg == 1) store(std::integral_constant<int, 1>{});
        else if (kg == 2) store(std::integral_constant<int, 2>{});
        else store(std::integral_constant<int, 3>{});
    }
}

template <int TM, int TN, int WGM, int WGN, int KG, int ST, bool YBF16>
int launch_tile(const char* fn, const int8_t* qx, const float* sx, const int8_t* qw, const float* sw, void* y,
                int64_t M, int64_t N, int64_t K, hipStream_t stream) {
    using S = TileShape<TM, TN, WGM, WGN, KG, ST>;
    static const bool ok = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_fp8_tile_kernel<TM, TN, WGM, WGN, KG, ST, YBF16>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, S::kLds) == hipSuccess;
    if (!ok) return kc::set_error(KC_ERR_HIP, "%s: cannot raise the LDS limit", fn);
    const int64_t tm = (M + S::kRowsM - 1) / S::kRowsM, tn = (N + S::kRowsN - 1) / S::kRowsN;
    gemm_fp8_tile_kernel<TM, TN, WGM, WGN, KG, ST, YBF16><<<static_cast<unsigned>(tm * tn), S::kThreadsT, S::kLds, stream>>>(
        qx, sx, qw, sw, y, M, N, K, static_cast<int>(tm), static_cast<int>(tn), N % 4 == 0 && kc::aligned(y, YBF16 ? 8 : 16));
    return kc::check_launch(fn);
}

// Tiles (the 256 x 256 kernel in front), and what a K step of 128 takes when
// every CU holds one of them, in hundredths of a microsecond (measured).  The
// least expected time wins: ceil(tiles / 256) rounds of K / 128 steps each, and
// what a round takes beside them (start, scales, the last barrier and the
// stores; 3 to 14 us measured, one figure for all tiles, which decides only
// between few large and many small tiles at short K: M 4096, N 6144 44.0 us at
// K 1024 in two rounds of 256 x 256, 53.2 in three of 256 x 128, 68.7 against 70.5
// at K 2048; M 1500, N 14336 43.8 against 48.2 and 70.4 against 65.5).  Against
// 256 x 256 tiles: M 128, N 4096, K 4096 48.2 -> 8.5 us (32 x 64); M 256, N 4096,
// K 14336 193 -> 36.5 (64 x 64); M 512, N 4096, K 4096 49.3 -> 18.3 (64 x 128);
// M 1000, N 4096, K 14336 148 -> 67.5 (128 x 128); M 1000, N 6144, K 4096 55 ->
// 35.5 (256 x 128); M 512, N 28672 and M 4096, N 4096 stay.
struct TileCost {
    int rows_m, rows_n, cost;
};
constexpr int kCus = 256;
constexpr int kRoundCost = 600;
constexpr TileCost kTiles[] = {{256, 256, 165}, {256, 128, 97}, {128, 128, 60}, {64, 128, 40}, {64, 64, 28}, {32, 64, 18}};

int best_tile(int64_t M, int64_t N, int64_t K) {
    const int64_t steps = (K + kBK - 1) / kBK;
    int best = 0;
    int64_t least = INT64_MAX;
    for (int i = 0; i < static_cast<int>(sizeof(kTiles) / sizeof(kTiles[0])); ++i) {
        const TileCost& t = kTiles[i];
        const int64_t tiles = ((M + t.rows_m - 1) / t.rows_m) * ((N + t.rows_n - 1) / t.rows_n);
        const int64_t cost = (tiles + kCus - 1) / kCus * (steps * t.cost + kRoundCost);
        if (cost < least) least = cost, best = i;
    }
    return best;
}

}  // namespace

namespace kc {
namespace fp8 {

template <bool YBF16>
bool gemm_small(const char* fn, const int8_t* qx, const float* sx, const int8_t* qw, const float* sw, void* y,
                int64_t M, int64_t N, int64_t K, hipStream_t stream, int* status) {
    // 32-bit lane offsets: at most 256 rows of a tile times K
    if (K > INT32_MAX / 256 || N > INT32_MAX / 2) return false;
    if (M <= kSkinnyM) {
        const int m = static_cast<int>(M), n = static_cast<int>(N), k = static_cast<int>(K);
        if (large_tiles_at_short_k<YBF16>((m + 15) / 16, n, k)) return false;
        switch ((m + 15) / 16) {
            case 1: *status = skinny<1, YBF16>(fn, qx, sx, qw, sw, y, m, n, k, stream); break;
            case 2: *status = skinny<2, YBF16>(fn, qx, sx, qw, sw, y, m, n, k, stream); break;
            case 3: *status = skinny<3, YBF16>(fn, qx, sx, qw, sw, y, m, n, k, stream); break;
            default: *status = skinny<4, YBF16>(fn, qx, sx, qw, sw, y, m, n, k, stream); break;
        }
        return true;
    }
    switch (best_tile(M, N, K)) {
        case 1: *status = launch_tile<4, 4, 4, 2, 1, 3, YBF16>(fn, qx, sx, qw, sw, y, M, N, K, stream); return true;
        case 2: *status = launch_tile<4, 2, 2, 4, 1, 4, YBF16>(fn, qx, sx, qw, sw, y, M, N, K, stream); return true;
        case 3: *status = launch_tile<4, 2, 1, 4, 2, 3, YBF16>(fn, qx, sx, qw, sw, y, M, N, K, stream); return true;
        case 4: *status = launch_tile<4, 2, 1, 2, 2, 4, YBF16>(fn, qx, sx, qw, sw, y, M, N, K, stream); return true;
        case 5: *status = launch_tile<2, 2, 1, 2, 2, 4, YBF16>(fn, qx, sx, qw, sw, y, M, N, K, stream); return true;
        default: return false;
    }
}

template bool gemm_small<true>(const char*, const int8_t*, const float*, const int8_t*, const float*, void*, int64_t,
                               int64_t, int64_t, hipStream_t, int*);
template bool gemm_small<false>(const char*, const int8_t*, const float*, const int8_t*, const float*, void*, int64_t,
                                int64_t, int64_t, hipStream_t, int*);

}  // namespace fp8
}  // namespace kc
