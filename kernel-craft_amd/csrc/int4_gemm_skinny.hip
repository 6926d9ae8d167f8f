// int4_gemm_skinny.hip -- the small-batch INT4 GEMM (see int4_gemm_mfma.hip
// for the operation and the decode) where the K-split kernel's 112 weight rows
// per workgroup leave most of the 256 CUs idle, and for groups below 128.
//
// gemm_int4_skinny_kernel: a workgroup of KW waves owns RT tiles of 16 weight
// rows (RT 1 or 2) and all MT = ceil(M / 16) tiles of X.  Wave w takes the
// pairs of T-blocks (128 k each) w, w + KW, ....  X runs one pair ahead: each
// tile of the next pair's X is requested as soon as this pair's has been
// multiplied; the weights have one set of registers, requested for the next
// pair once both T-blocks of this one are multiplied (two to four sets were
// slower: registers and occupancy).  No barrier stands in the loop, and the KW
// partial sums of every output meet in LDS in a fixed order.
// The K-split kernel's time hardly depends on N (K 14336: 47 us at M 16, 94 at
// M 64, for 37 workgroups as for 74), this one's follows it:
//   N 4096, K 14336: M 16 47.2 -> 15.0 us, M 32 68 -> 22.3, M 64 94 -> 38.4;
//   N 6144, K 4096:  M 4 12.4 -> 7.3, M 16 12.5 -> 8.0, M 64 23.4 -> 17.6;
//   N 14336, K 4096: M 12 12.5 -> 11.1.
// Bound by the loads from the XCD's L2, every workgroup reading all of X, and
// by bringing X into operand order: M 16, N 4096, K 14336 reads 151 MB there for
// 31 MB of weights and coefficients (10 TB/s), M 64 505 MB (13 TB/s), the matrix
// cores 7 and 14 % busy.
//
// Loads.  One wave-wide load covers 8 whole 128-byte lines.  Weights of the
// reference layout: load h of a pair takes rows 8 h .. 8 h + 7, lane (i, kb)
// (i = l % 16, kb = l / 16) chunk kb + 4 (i % 2) of row 8 h + i / 2; neighbouring
// lanes then exchange chunks (one quad permutation and select per dword), and
// operand row i is tile row i / 2 + 8 (i % 2).  The shuffled layout's 1-KB
// blocks are the operand as they stand.  X: load (j1, j0) of a T-block takes
// bytes 128 j1 + 64 b0 + 32 b1 + 16 (i % 2) .. + 15 (kb = 2 b1 + b0) of row
// (i & ~1) + j0; a permlane32 swap exchanges j1 with b1, the quad permutation
// j0 with i % 2, which leaves the lane the 64 bytes of its row that its
// weights multiply.
//
// Groups of 64 and 32 (NG = 2, 4 groups per T-block): the operand lanes of the
// other groups are zeroed, one product per group.  Two tokens, and some shapes
// of three to six (gemvs_faster below), take one GEMV per row of X, as all did
// before.
#include <algorithm>
#include <type_traits>

#include "int4_decode.hpp"
#include "int4_gemm.hpp"
#include "kc_common.hpp"

namespace {

using kc::kWave;
using namespace kc::int4;

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

constexpr int kTBlock = 128;  // k per T-block: 64 bytes of each W row
constexpr int kCoefRow = 36;  // floats per (group, row tile): 16 s, 16 c2 = -s (136 + z), padded
constexpr int kMaxLds = 160 * 1024;
constexpr int kOneTileRows = 16 * 256;  // one 16-row tile per CU

__device__ __forceinline__ bf16x8_t a_operand(uint32_t d, NibConsts k) {
    const u32x4 p{nib_pair(d, k), nib_pair(d >> 4, k), nib_pair(d >> 8, k), nib_pair(d >> 12, k)};
    return __builtin_bit_cast(bf16x8_t, p);
}

template <int CTRL>
__device__ __forceinline__ uint32_t quad(uint32_t v) {
    return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(v), CTRL, 0xF, 0xF, true));
}
constexpr int kXor1 = 0xB1;  // quad permutation [1,0,3,2]

template <int MT, int RT, int KW, int NG, bool SHUF>
__global__ __launch_bounds__(KW * kWave) void gemm_int4_skinny_kernel(
    const uint8_t* __restrict__ packed, const float* __restrict__ scales,
    const uint8_t* __restrict__ zeros, const uint16_t* __restrict__ X, uint16_t* __restrict__ Y,
    int M, int N, int K, int gshift) {
    static_assert(NG == 1 || !SHUF, "the shuffled layout takes groups of 128 or more");
    extern __shared__ __align__(16) char lds[];
    float* coef = reinterpret_cast<float*>(lds);
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int i = lane & 15, kb = lane >> 4;
    const int nT = K / kTBlock, nP = (nT + 1) >> 1;
    const int G = NG > 1 ? NG * nT : nT >> gshift;  // groups per row
    const int nE = NG * nT;                         // coefficient table entries: NG per T-block
    const int n0 = static_cast<int>(blockIdx.x) * 16 * RT;
    const int mine = nP > wave ? (nP - wave + KW - 1) / KW : 0;  // pairs wave, wave + KW, ...
    const bool even = (lane & 1) == 0;

    // operand row of tile row r
    auto operand_row = [](int r) { return SHUF ? r : 2 * (r & 7) + (r >> 3); };

    uint32_t woff[RT][2], xoff[MT][4];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int h = 0; h < 2; ++h)
            woff[r][h] = SHUF ? static_cast<uint32_t>(min(n0 / 16 + r, (N + 15) / 16 - 1) - n0 / 16) * static_cast<uint32_t>(nT) * 1024u + 1024u * h + 16u * lane
                              : static_cast<uint32_t>(min(n0 + 16 * r + 8 * h + (i >> 1), N - 1) - n0) * static_cast<uint32_t>(K >> 1) + 16u * (kb + 4 * (i & 1));
#pragma unroll
    for (int c = 0; c < MT; ++c)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            xoff[c][j] = static_cast<uint32_t>(min(16 * c + ((i & 14) | (j & 1)), M - 1)) * static_cast<uint32_t>(2 * K) + 128u * (j >> 1) + 64u * (kb & 1) + 32u * (kb >> 1) + 16u * (i & 1);
    const uint8_t* wbase = packed + static_cast<int64_t>(n0) * (K >> 1);  // SHUF: the same byte, n0 a multiple of 16
    const uint8_t* xbase = reinterpret_cast<const uint8_t*>(X);
    const bool odd_last = (nT & 1) != 0;

    // coefficients of the workgroup's rows
    constexpr int kRowsW = (16 * RT + KW - 1) / KW;  // rows per wave
    auto stage_load = [&](int tb, float (&sv)[kRowsW][2], uint32_t (&zv)[kRowsW][2]) {
#pragma unroll
        for (int u = 0; u < kRowsW; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int64_t row = min(n0 + min(wave + u * KW, 16 * RT - 1), N - 1);
                const int g = NG > 1 ? min(tb + 64 * h + lane, nE - 1) : min(tb + 64 * h + lane, nE - 1) >> gshift;
                sv[u][h] = scales[row * G + g];
                zv[u][h] = zeros[row * (G >> 1) + (g >> 1)];
            }
    };
    auto stage_store = [&](int tb, const float (&sv)[kRowsW][2], const uint32_t (&zv)[kRowsW][2]) {
#pragma unroll
        for (int u = 0; u < kRowsW; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int e = tb + 64 * h + lane, r = wave + u * KW;
                if (e < nE && r < 16 * RT) {
                    const uint32_t z = ((NG > 1 ? e : e >> gshift) & 1) ? zv[u][h] >> 4 : zv[u][h] & 0xFu;
                    float* p = coef + (e * RT + (r >> 4)) * kCoefRow + operand_row(r & 15);
                    p[0] = sv[u][h];
                    p[16] = -sv[u][h] * static_cast<float>(136u + z);
                }
            }
    };
    float sv[kRowsW][2];
    uint32_t zv[kRowsW][2];
    stage_load(0, sv, zv);
    __builtin_amdgcn_sched_barrier(0);

    u32x4 w[RT][2], x[2][MT][4];
    auto load_w = [&](int j) {
        const int p = wave + KW * min(j, mine - 1);
        const uint8_t* b = wbase + static_cast<int64_t>(p) * (SHUF ? 2048 : 128);
        const bool half = odd_last && p == nP - 1;  // only one T-block left: its bytes twice
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                uint32_t o = woff[r][h];
                if (SHUF) o -= half && h ? 1024u : 0u;
                else o -= half && (i & 1) ? 64u : 0u;
                w[r][h] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(b + o));
            }
    };
    auto load_x = [&](int c, int t, int j) {  // tile c of X, T-block t of pair j
        const int T = min(2 * (wave + KW * j) + t, nT - 1);
        const uint8_t* b = xbase + 256 * T;
#pragma unroll
        for (int q = 0; q < 4; ++q) x[t][c][q] = *reinterpret_cast<const u32x4*>(b + xoff[c][q]);
    };
    if (mine > 0) {
        load_w(0);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int c = 0; c < MT; ++c) load_x(c, t, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    stage_store(0, sv, zv);
    for (int tb = 128; tb < nE; tb += 128) {
        float s2[kRowsW][2];
        uint32_t z2[kRowsW][2];
        stage_load(tb, s2, z2);
        stage_store(tb, s2, z2);
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

    const NibConsts nk = nib_consts();
    uint32_t sel_lo, sel_hi;  // v_perm_b32 selectors, in VGPRs
    asm volatile("v_mov_b32 %0, 0x05040100" : "=v"(sel_lo));
    asm volatile("v_mov_b32 %0, 0x07060302" : "=v"(sel_hi));
    const bf16x8_t ones = __builtin_bit_cast(bf16x8_t, u32x4{0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u});
    f32x4 acc[RT][MT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int c = 0; c < MT; ++c) acc[r][c] = f32x4{0.f, 0.f, 0.f, 0.f};

    // the lane's 16 weight bytes of T-block t of a pair
    auto weights = [&](const u32x4 (&p)[2], int t) -> u32x4 {
        if constexpr (SHUF) return p[t];
        const uint32_t a[4] = {p[0].x, p[0].y, p[0].z, p[0].w}, b[4] = {p[1].x, p[1].y, p[1].z, p[1].w};
        uint32_t o[4];
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            const uint32_t n = quad<kXor1>(t == 0 ? b[d] : a[d]);
            o[d] = t == 0 ? (even ? a[d] : n) : (even ? n : b[d]);
        }
        return u32x4{o[0], o[1], o[2], o[3]};
    };
    // T-block t of the pair in registers (T-block T of the matrix); each tile
    // of X is requested for pair `next` once it has been multiplied
    auto tblock = [&](int T, int t, int next, auto more) {
        bf16x8_t a[RT][4];
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const u32x4 v = weights(w[r], t);
            const uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int s = 0; s < 4; ++s) a[r][s] = a_operand(d[s], nk);
        }
        f32x4 s4[NG][RT], z4[NG][RT];
#pragma unroll
        for (int q = 0; q < NG; ++q)
#pragma unroll
            for (int r = 0; r < RT; ++r) {
                const float* p = coef + ((T * NG + q) * RT + r) * kCoefRow + 4 * kb;
                s4[q][r] = *reinterpret_cast<const f32x4*>(p);
                z4[q][r] = *reinterpret_cast<const f32x4*>(p + 16);
            }
#pragma unroll
        for (int c = 0; c < MT; ++c) {
            // 4 x 4 transpose over each lane quad: piece s of row i into register s
            uint32_t m[4][4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const u32x4 v = x[t][c][q];
                m[q][0] = v.x, m[q][1] = v.y, m[q][2] = v.z, m[q][3] = v.w;
            }
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                // register (j1, j0), lane (i, b1 b0): j1 with b1, then j0 with bit 0 of i
                const auto p0 = __builtin_amdgcn_permlane32_swap(m[0][d], m[2][d], false, false);
                const auto p1 = __builtin_amdgcn_permlane32_swap(m[1][d], m[3][d], false, false);
                const uint32_t t0 = p0[0], t2 = p0[1], t1 = p1[0], t3 = p1[1];
                const uint32_t n0 = quad<kXor1>(t0), n1 = quad<kXor1>(t1), n2 = quad<kXor1>(t2), n3 = quad<kXor1>(t3);
                m[0][d] = even ? t0 : n1;
                m[1][d] = even ? n0 : t1;
                m[2][d] = even ? t2 : n3;
                m[3][d] = even ? n2 : t3;
            }
            bf16x8_t b[4];
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                u32x4 q;
                q.x = __builtin_amdgcn_perm(m[s][2], m[s][0], sel_lo);  // (x0, x4)
                q.y = __builtin_amdgcn_perm(m[s][2], m[s][0], sel_hi);  // (x1, x5)
                q.z = __builtin_amdgcn_perm(m[s][3], m[s][1], sel_lo);  // (x2, x6)
                q.w = __builtin_amdgcn_perm(m[s][3], m[s][1], sel_hi);  // (x3, x7)
                b[s] = __builtin_bit_cast(bf16x8_t, q);
            }
#pragma unroll
            for (int q = 0; q < NG; ++q) {
                // this group's k: with NG > 1 the lanes kb in [4 q / NG, 4 (q + 1) / NG)
                const bool in = NG == 1 || kb / (4 / NG) == q;
                auto group = [&](const bf16x8_t& v) {
                    if constexpr (NG == 1) return v;
                    const u32x4 d = __builtin_bit_cast(u32x4, v);
                    return __builtin_bit_cast(bf16x8_t, u32x4{in ? d.x : 0u, in ? d.y : 0u, in ? d.z : 0u, in ? d.w : 0u});
                };
                f32x4 sum{0.f, 0.f, 0.f, 0.f};  // every row: sum of x over the group
#pragma unroll
                for (int s = 0; s < 4; ++s) sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(group(ones), b[s], sum, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < RT; ++r) {
                    f32x4 d{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int s = 0; s < 4; ++s) d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(group(a[r][s]), b[s], d, 0, 0, 0);
                    f32x4& v = acc[r][c];
                    v.x = fmaf(s4[q][r].x, d.x, fmaf(z4[q][r].x, sum.x, v.x));
                    v.y = fmaf(s4[q][r].y, d.y, fmaf(z4[q][r].y, sum.x, v.y));
                    v.z = fmaf(s4[q][r].z, d.z, fmaf(z4[q][r].z, sum.x, v.z));
                    v.w = fmaf(s4[q][r].w, d.w, fmaf(z4[q][r].w, sum.x, v.w));
                }
            }
            if constexpr (decltype(more)::value) load_x(c, t, next);
            __builtin_amdgcn_sched_barrier(0);  // one tile of X at a time (register demand)
        }
    };
    int j = 0;
    for (; j + 1 < mine; ++j) {
        const int T = 2 * (wave + KW * j);  // not the last pair: both T-blocks exist
        tblock(T, 0, j + 1, std::true_type{});
        tblock(T + 1, 1, j + 1, std::true_type{});
        load_w(j + 1);
        __builtin_amdgcn_sched_barrier(0);
    }
    if (j < mine) {
        const int T = 2 * (wave + KW * j);
        tblock(T, 0, 0, std::false_type{});
        if (T + 1 < nT) tblock(T + 1, 1, 0, std::false_type{});
    }

    // the waves' partial sums, in a fixed order
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // every wave has read its coefficients
    f32x4* red = reinterpret_cast<f32x4*>(lds);
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int c = 0; c < MT; ++c) red[(wave * RT * MT + r * MT + c) * kWave + lane] = acc[r][c];
    __syncthreads();
    for (int t = wave; t < RT * MT; t += KW) {
        f32x4 v = red[t * kWave + lane];
#pragma unroll
        for (int u = 1; u < KW; ++u) {
            const f32x4 o = red[(u * RT * MT + t) * kWave + lane];
            v = f32x4{v.x + o.x, v.y + o.y, v.z + o.z, v.w + o.w};
        }
        const int m = 16 * (t % MT) + i;
        if (m >= M) continue;
        const float vals[4] = {v.x, v.y, v.z, v.w};
        uint16_t* yp = Y + static_cast<int64_t>(m) * N;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int n = n0 + 16 * (t / MT) + (SHUF ? 4 * kb + e : 2 * kb + (e >> 1) + 8 * (e & 1));
            if (n < N) yp[n] = kc::f32_to_bf16(vals[e]);
        }
    }
}

template <int MT, int RT, int KW, int NG, bool SHUF>
int launch(const char* fn, const uint8_t* packed, const float* scales, const uint8_t* zeros, const uint16_t* X,
           uint16_t* Y, int M, int N, int K, int gshift, hipStream_t stream) {
    const size_t coef = static_cast<size_t>(K / kTBlock) * NG * RT * kCoefRow * 4;
    const size_t red = static_cast<size_t>(KW) * RT * MT * kWave * 16;
    const size_t lds = std::max(coef, red);
    if (lds > kMaxLds) return -1;
    static const bool ok = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_int4_skinny_kernel<MT, RT, KW, NG, SHUF>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds) == hipSuccess;
    if (!ok) return kc::set_error(KC_ERR_HIP, "%s: cannot raise the LDS limit", fn);
    const int rows = 16 * RT;
    gemm_int4_skinny_kernel<MT, RT, KW, NG, SHUF><<<static_cast<unsigned>((N + rows - 1) / rows), KW * kWave, lds, stream>>>(
        packed, scales, zeros, X, Y, M, N, K, gshift);
    return kc::check_launch(fn);
}

// One row tile per workgroup up to one workgroup per CU (N 4096), two beyond.
// Eight waves share K (M 64, N 4096, K 4096 15.0 us against 17.6 with four),
// but four where eight do not have the registers: two row tiles with more than
// one tile of X (M 32, N 8192, K 14336 28.9 against 26.7), small groups (M 41,
// N 5760, groups of 64 29.8 against 21.6); and past N 8192, where two
// workgroups share a CU (M 4, N 14336, K 4096: 13.1 against 10.5).
template <int MT, int NG, bool SHUF>
int by_rows(const char* fn, const uint8_t* packed, const float* scales, const uint8_t* zeros, const uint16_t* X,
            uint16_t* Y, int M, int N, int K, int gshift, hipStream_t stream) {
    if (N <= kOneTileRows) {
        constexpr int kw = NG == 1 || MT == 1 ? 8 : 4;
        return launch<MT, 1, kw, NG, SHUF>(fn, packed, scales, zeros, X, Y, M, N, K, gshift, stream);
    }
    if constexpr (MT == 1) {
        if (N <= 2 * kOneTileRows)
            return launch<MT, 2, 8, NG, SHUF>(fn, packed, scales, zeros, X, Y, M, N, K, gshift, stream);
    }
    return launch<MT, 2, 4, NG, SHUF>(fn, packed, scales, zeros, X, Y, M, N, K, gshift, stream);
}

template <int NG, bool SHUF>
int by_tokens(const char* fn, const uint8_t* packed, const float* scales, const uint8_t* zeros, const uint16_t* X,
              uint16_t* Y, int M, int N, int K, int gshift, hipStream_t stream) {
    switch ((M + 15) / 16) {
        case 1: return by_rows<1, NG, SHUF>(fn, packed, scales, zeros, X, Y, M, N, K, gshift, stream);
        case 2: return by_rows<2, NG, SHUF>(fn, packed, scales, zeros, X, Y, M, N, K, gshift, stream);
        case 3: return by_rows<3, NG, SHUF>(fn, packed, scales, zeros, X, Y, M, N, K, gshift, stream);
        default: return by_rows<4, NG, SHUF>(fn, packed, scales, zeros, X, Y, M, N, K, gshift, stream);
    }
}

// Groups of 64 and 32 at few tokens: whether one GEMV per token is expected to
// be faster, in ns.  A GEMV takes 2 us and its weights at 5.5 bytes per ns
// (half a byte each; short rows count as 1650 k); the kernel here 2.9 us and, whatever M, a time per k that
// follows the rows past 8192 (few rows: every workgroup walks all of K alone) and
// is longer for groups of 32, above all where their coefficients (9 bytes per k)
// leave one workgroup per CU.  Measured, GEMVs against this kernel: M 3, K 14336,
// groups of 32: N 1024 10.4 against 21.4 us, N 4096 23.0 / 23.1, N 28672 121 / 173;
// groups of 64: N 1024 10.1 / 15.9, N 4096 22.1 / 17.0; M 5, N 512, K 14336, groups of
// 32 15.7 / 21.2, K 4096 11.1 / 7.7.  Of 720 shapes (M 3 to 12, N 256 to 28672, K 512 to
// 14336) the choice costs more than 3 % on 7, 13 % at most; from M 7 on the GEMVs
// are never clearly faster.
bool gemvs_faster(int M, int N, int K, int group_size) {
    if (M > 6) return false;
    const bool half = group_size == 32;
    const int64_t gemv = 2000 + static_cast<int64_t>(N) * std::max(K, 1650) / 11000;
    int64_t k = K, ps;  // ps per k
    if (N <= kOneTileRows) {
        ps = half ? 1260 : 900;
    } else if (N <= 2 * kOneTileRows) {
        ps = half ? 2150 : 1550;
    } else {
        k = (k + 1023) / 1024 * 1024;  // whole pairs for each of four waves
        ps = static_cast<int64_t>(N) * (!half ? 205 : 9 * K <= 80 * 1024 ? 290 : 400) / 1000;
    }
    return M * gemv < 2900 + k * ps / 1000;
}

}  // namespace

namespace kc {
namespace int4 {

template <bool SHUF>
int gemm_skinny(const char* fn, const uint8_t* packed, const float* scales, const uint8_t* zeros, const uint16_t* X,
                uint16_t* Y, int M, int N, int K, int group_size, hipStream_t stream) {
    if (K > INT32_MAX / 128) return -1;  // 32-bit offsets of 64 rows of X
    if constexpr (!SHUF) {
        if (group_size < kTBlock && gemvs_faster(M, N, K, group_size)) return -1;
        if (group_size == 64) return by_tokens<2, false>(fn, packed, scales, zeros, X, Y, M, N, K, 0, stream);
        if (group_size == 32) return by_tokens<4, false>(fn, packed, scales, zeros, X, Y, M, N, K, 0, stream);
    }
    // Past these N the K-split kernel fills the chip (M 16, N 28672, K 4096:
    // 16.1 us there, 26.6 here; M 32, N 10240, K 4096 16.5 against 16.4; M 48
    // 20.4 against 28.3).  Up to them this kernel is the faster one at K 4096,
    // 5120, 8192, 14336 and 20480, M 2 to 64, on both layouts: 4 to 8 % at the lines
    // (M 16, N 16384, K 8192 22.4 -> 21.5 us; M 64, N 8192, K 8192 39.1 -> 29.7).
    if (N > (M <= 16 ? 4 : 2) * kOneTileRows) return -1;
    // Up to 8 tokens on the reference layout at K below 1024 the waves have a
    // pair of T-blocks at most, and one wave per row tile over all of K
    // (gemm_int4_mfma_kernel) is faster from two row tiles on: M 4, K 512, N 8192
    // 4.0 against 4.2 us, N 12000 4.1 against 5.0; K 640 and 896 3 to 6 % slower up
    // to N 8192, 3 to 17 % faster past it; K 1152 10 to 32 % slower.
    if (!SHUF && M <= 8 && K < 1024 && N > (K <= 512 ? 1 : 2) * kOneTileRows) return -1;
    return by_tokens<1, SHUF>(fn, packed, scales, zeros, X, Y, M, N, K, kc::ilog2(group_size) - 7, stream);
}

template int gemm_skinny<true>(const char*, const uint8_t*, const float*, const uint8_t*, const uint16_t*, uint16_t*, int,
                               int, int, int, hipStream_t);
template int gemm_skinny<false>(const char*, const uint8_t*, const float*, const uint8_t*, const uint16_t*, uint16_t*,
                                int, int, int, int, hipStream_t);

}  // namespace int4
}  // namespace kc
