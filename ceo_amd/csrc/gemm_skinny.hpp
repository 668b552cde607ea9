// Products with few rows (token-by-token generation): D[m, n] = epilogue(
// sum_k A[m, k] opB(k, n) ) for M <= 16 MT, bf16 / fp16, fp32 accumulation.
// Included by gemm.hip.
//
// Bound by the weight matrix, which is read once: the 256 x 256 tiles of
// gemm_fast.hpp leave most CUs without a tile and split along k to fill them,
// a second launch and fp32 partials through memory.  Here a workgroup owns 32
// output columns and all of k, its eight waves taking 32-row steps of k in
// turn, so an (N / 32)-workgroup grid streams the weights with no LDS staging:
//   * a lane holds, for its k group of 8 rows, two neighbouring columns of the
//     weights (4-byte loads, 16 lanes to a 64-byte row piece, 32 or more of
//     them in flight per lane) and pairs the rows up in registers with one
//     byte permute per operand dword, so the column pair becomes two MFMA
//     operands; a k-contiguous B (a weight used transposed) is read as 16-byte
//     operand pieces directly;
//   * the weights are the MFMA's A operand (16 x 16 x 32): lane (r, g) ends up
//     with columns n0 + 2 (4 g + e) + j of row r, eight consecutive columns;
//   * the eight waves' sums meet in LDS, added in wave order (the result does
//     not depend on scheduling), and the epilogue runs on 16-byte row pieces.
// A long k over few columns (the MLP's down product) is split over the idle
// CUs into fp32 partials that gemm_splitk_reduce adds in order.
// 16 rows, weights from memory (large tile with its split-K / this, us):
// 1024 x 3088 15.1 / 5.3, 1024 x 1024 13.1 / 5.0, 1024 x 4096 15.8 / 5.8,
// 4096 x 1024 18.3 / 9.3; 2048 x 8192 21.5 / 12.3 (2.7 TB/s).
#pragma once
#include "gemm_fast.hpp"

namespace efla {
namespace gs {

using gf::EpiArgs;
using mf::bf16;
using mf::bf16x8;
using mf::floatx4;

constexpr int NW = 8, NTH = 64 * NW;
constexpr int BN = 32;  // columns per workgroup

template <typename T>
__device__ __forceinline__ floatx4 mma16(bf16x8 a, bf16x8 b, floatx4 c) {
    if constexpr (__is_same(T, gf::f16))
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(gf::f16x8, a),
                                                       __builtin_bit_cast(gf::f16x8, b), c, 0, 0, 0);
    else
        return mf::mma(a, b, c);
}

// M in 1 .. 16 MT; K % 8 == 0; A rows of 16-byte aligned pieces (lda % 8 ==
// 0); B as BKC [n][k] the same, else [k][n] with N and ldb even, 4-byte
// aligned.  U steps of k are in flight per wave.
template <typename T, bool BKC, int EPI, int MT>
__global__ void __launch_bounds__(NTH) gemm_skinny_kernel(const T* __restrict__ A, long lda,
                                                          const T* __restrict__ B, long ldb,
                                                          int M, int N, int Kall, int kper,
                                                          EpiArgs<T> ea) {
    constexpr int U = MT <= 2 ? 4 : 2;
    __shared__ floatx4 part[NW][MT][2][64];
    const int w = mf::wave(), l = mf::lane(), g = l >> 4, r = l & 15;
    const int n0 = blockIdx.x * BN;
    // this workgroup's range of k (blockIdx.y > 0 only with EPI_PARTIAL)
    const int kbeg = (int)blockIdx.y * kper, K = min(kper, Kall - kbeg);
    A += kbeg;
    B += BKC ? (long)kbeg : (long)kbeg * ldb;
    floatx4 acc[MT][2];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t][0] = acc[t][1] = floatx4{0.f, 0.f, 0.f, 0.f};
    const T* ap[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) ap[t] = A + (long)min(16 * t + r, M - 1) * lda + 8 * g;
    const T* b0 = BKC ? B + (long)min(n0 + 2 * r, N - 1) * ldb + 8 * g
                      : B + (long)(8 * g) * ldb + min(n0 + 2 * r, N - 2);
    const T* b1 = BKC ? B + (long)min(n0 + 2 * r + 1, N - 1) * ldb + 8 * g : nullptr;
    // NU steps of k, s, s + NW, ...: all of their loads, then their products.
    // In the step that k ends in, the lanes of the k groups past the end read
    // group 0 of step 0 and count as zero.
    auto run = [&](int s, auto nu, bool in) {
        constexpr int NU = decltype(nu)::value;
        bf16x8 a[NU][MT], b[NU][2];
        unsigned x[NU][8];
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            const long k0 = in ? 32L * (s + NW * u) : -8L * g;
            if constexpr (BKC) {
                b[u][0] = *reinterpret_cast<const bf16x8*>(b0 + k0);
                b[u][1] = *reinterpret_cast<const bf16x8*>(b1 + k0);
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    x[u][j] = *reinterpret_cast<const unsigned*>(b0 + (k0 + j) * ldb);
            }
#pragma unroll
            for (int t = 0; t < MT; ++t) a[u][t] = *reinterpret_cast<const bf16x8*>(ap[t] + k0);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            if constexpr (!BKC) {
                // rows 2i, 2i + 1 of the column pair -> the pair's two operands
                mf::int4v lo, hi;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    lo[i] = (int)__builtin_amdgcn_perm(x[u][2 * i + 1], x[u][2 * i], 0x05040100u);
                    hi[i] = (int)__builtin_amdgcn_perm(x[u][2 * i + 1], x[u][2 * i], 0x07060302u);
                }
                b[u][0] = __builtin_bit_cast(bf16x8, lo);
                b[u][1] = __builtin_bit_cast(bf16x8, hi);
            }
            if constexpr (NU == 1) {
                if (!in) {
                    b[u][0] = b[u][1] = bf16x8{};
#pragma unroll
                    for (int t = 0; t < MT; ++t) a[u][t] = bf16x8{};
                }
            }
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                acc[t][0] = mma16<T>(b[u][0], a[u][t], acc[t][0]);
                acc[t][1] = mma16<T>(b[u][1], a[u][t], acc[t][1]);
            }
        }
    };
    const int steps = K / 32;
    int s = w;
    for (; s + NW * (U - 1) < steps; s += NW * U) run(s, std::integral_constant<int, U>{}, true);
    for (; 32L * s < K; s += NW) run(s, std::integral_constant<int, 1>{}, 32L * s + 8 * g < K);
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        part[w][t][0][l] = acc[t][0];
        part[w][t][1][l] = acc[t][1];
    }
    __syncthreads();
    // thread -> (row tile, lane): row m, columns n .. n + 7
    typedef gf::Piece<8, T> P8;
    typedef typename P8::vec t8;
    for (int i = threadIdx.x; i < 64 * MT; i += NTH) {
        const int t = i >> 6, li = i & 63;
        const long m = 16 * t + (li & 15), n = n0 + 8 * (li >> 4);
        if (m >= M || n >= N) continue;
        floatx4 s0 = part[0][t][0][li], s1 = part[0][t][1][li];
#pragma unroll
        for (int v = 1; v < NW; ++v) {
            s0 += part[v][t][0][li];
            s1 += part[v][t][1][li];
        }
        if constexpr (EPI == gf::EPI_PARTIAL) {
            float* dst = ea.part + ((long)blockIdx.y * M + m) * ((N + 7) & ~7) + n;
            *reinterpret_cast<floatx4*>(dst) = floatx4{s0[0], s1[0], s0[1], s1[1]};
            *reinterpret_cast<floatx4*>(dst + 4) = floatx4{s0[2], s1[2], s0[3], s1[3]};
            continue;
        }
        float v[8];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[2 * e] = ea.alpha * s0[e];
            v[2 * e + 1] = ea.alpha * s1[e];
        }
        if (ea.bias) {
            const t8 bb = P8::load(ea.bias + n, N - n);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] += (float)bb[e];
        }
        t8 y;
        if constexpr (EPI == gf::EPI_GELU_AUX) {
            t8 pre;
#pragma unroll
            for (int e = 0; e < 8; ++e) pre[e] = (T)v[e];
            P8::store(ea.aux + m * ea.ldaux + n, pre, N - n);
#pragma unroll
            for (int e = 0; e < 8; ++e) y[e] = (T)gelu::gelu_f<true>((float)pre[e]);
        } else {
            if (EPI == gf::EPI_RESID && ea.beta != 0.f) {
                const t8 c = P8::load(ea.c + m * ea.ldc + n, N - n);
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] += ea.beta * (float)c[e];
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) y[e] = (T)v[e];
        }
        P8::store(ea.d + m * ea.ldd + n, y, N - n);
    }
}

}  // namespace gs
}  // namespace efla
