// Chunk-free EFLA steps: a few tokens per sequence continued from a carried
// fp32 state (token-by-token generation, a drafted continuation).  Included by
// efla_q.hip.
//
// Bound by the state: K x V fp32 per (sequence, head) is read once and written
// once, everything else is a few hundred bytes.  A workgroup owns one 64-wide
// value slice of one (sequence, head) state and keeps it in registers through
// all its tokens:
//   u = S^T k,  r = c (v - u),  S <- S + k r^T,  o = S^T q
// with o formed from the old state, o = S_old^T q + (k . q) r, so one reduction
// per token carries both sums.  All of it in fp32, the recurrence as written:
// no 64-token chunk is padded, and the state meets no bf16 rounding (the
// chunked form rounds it as an MFMA operand).
//
// A row of the slice is 16 lanes x 16 bytes; a wave covers 4 rows per load, the
// four waves 16, and a thread holds K / 16 pieces, all in flight at once.
// 64 sequences x 16 heads, K = V = 128, one token (134 MB of states read and
// written): 22.1 us, 6.1 TB/s, against 59.5 us for prep + scan of a padded
// chunk; two tokens 28.5, four 36.8 us (the per-token chain of two barriers
// and two reductions starts to show).  One sequence x 4 heads x 64 x 64: 3.3
// against 9.8 us.
#pragma once
#include "common.hpp"
#include "efla_coeff.hpp"
#include "efla_q_seq.hpp"

namespace efla {
namespace q {
namespace step {

constexpr int NT = 256;
constexpr int VS = 64;
typedef floatx4 floatx4u __attribute__((aligned(4)));  // state rows of any float alignment

// Piece i of a thread is row 16 i + row0, columns v0 + 4 cq .. + 3.  S0 may be
// ST: every element is read and written by one thread.
template <typename T, int K, int V>
__global__ void __launch_bounds__(NT) step_kernel(const T* __restrict__ q,
                                                  const T* __restrict__ k,
                                                  const T* __restrict__ v,
                                                  const T* __restrict__ beta, long tokens, int H,
                                                  const float* S0, float* ST, T* __restrict__ o,
                                                  TokLd ld) {
    constexpr int R = K / 16;
    __shared__ float sk[2][K], sq[2][K], sv[2][VS];
    __shared__ floatx4 part[2][4][16][2];  // [parity][wave][column quad][u | S^T q]
    constexpr int NVS = V / VS;
    const int vs = blockIdx.x % NVS;
    const long bh = blockIdx.x / NVS;
    const int h = (int)(bh % H), v0 = vs * VS;
    const long bos = bh / H * tokens;
    const int w = wave_id(), l = lane_id(), cq = l & 15, row0 = 4 * w + (l >> 4);
    const long sbase = bh * K * V + v0 + 4 * cq;

    // a token's k, q and value slice, and its beta, one token ahead
    constexpr int NL = (2 * K + VS + NT - 1) / NT;
    float nx[NL], nbeta;
    auto fetch = [&](long t) {
        const long tok = bos + t;
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int id = (int)threadIdx.x + NT * i;
            nx[i] = id < K             ? to_f(k[tok * ld.k + (long)h * K + id])
                    : id < 2 * K       ? to_f(q[tok * ld.q + (long)h * K + id - K])
                    : id < 2 * K + VS  ? to_f(v[tok * ld.v + (long)h * V + v0 + id - 2 * K])
                                       : 0.f;
        }
        nbeta = to_f(beta[tok * H + h]);
    };
    fetch(0);
    floatx4 S[R];
#pragma unroll
    for (int i = 0; i < R; ++i)
        S[i] = *reinterpret_cast<const floatx4u*>(S0 + sbase + (long)(16 * i + row0) * V);

    for (long t = 0; t < tokens; ++t) {
        const int p = (int)(t & 1);
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int id = (int)threadIdx.x + NT * i;
            if (id < K) sk[p][id] = nx[i];
            else if (id < 2 * K) sq[p][id - K] = nx[i];
            else if (id < 2 * K + VS) sv[p][id - 2 * K] = nx[i];
        }
        const float bet = nbeta;
        if (t + 1 < tokens) fetch(t + 1);
        __syncthreads();
        // lambda and k . q, by every wave for itself
        float lam = 0.f, kq = 0.f;
#pragma unroll
        for (int i = 0; i < K / 64; ++i) {
            const float a = sk[p][64 * i + l];
            lam += a * a;
            kq += a * sq[p][64 * i + l];
        }
#pragma unroll
        for (int m = 32; m; m >>= 1) {
            lam += __shfl_xor(lam, m);
            kq += __shfl_xor(kq, m);
        }
        float c, dcl, dcb;
        efla_coeff(lam, bet, c, dcl, dcb);
        float kr[R];
        floatx4 u{0.f, 0.f, 0.f, 0.f}, s{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < R; ++i) {
            kr[i] = sk[p][16 * i + row0];
            const float qr = sq[p][16 * i + row0];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                u[e] += kr[i] * S[i][e];
                s[e] += qr * S[i][e];
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
            for (int m = 16; m < 64; m <<= 1) {
                u[e] += __shfl_xor(u[e], m);
                s[e] += __shfl_xor(s[e], m);
            }
        }
        if (l < 16) {
            part[p][w][cq][0] = u;
            part[p][w][cq][1] = s;
        }
        __syncthreads();
        // (the other parity's buffers are rewritten only after the next
        // token's first barrier, which every wave reaches past these reads)
        floatx4 r;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float ut = part[p][0][cq][0][e] + part[p][1][cq][0][e] +
                             part[p][2][cq][0][e] + part[p][3][cq][0][e];
            r[e] = c * (sv[p][4 * cq + e] - ut);
        }
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) S[i][e] += kr[i] * r[e];
        if (w == 0 && l < 16) {
            T* dst = o + ((bos + t) * H + h) * V + v0 + 4 * cq;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float st = part[p][0][cq][1][e] + part[p][1][cq][1][e] +
                                 part[p][2][cq][1][e] + part[p][3][cq][1][e];
                dst[e] = from_f<T>(st + kq * r[e]);
            }
        }
    }
    if (ST) {
#pragma unroll
        for (int i = 0; i < R; ++i)
            *reinterpret_cast<floatx4u*>(ST + sbase + (long)(16 * i + row0) * V) = S[i];
    }
}

}  // namespace step
}  // namespace q
}  // namespace efla
