// Add-RMSNorm of a few rows inside the kernel that consumes them (decode sizes).
//
// A separate add-RMSNorm launch between two projections costs 2.5 - 3 us of
// which the row's own work is a fraction.  For a few rows every workgroup of
// the consumer can afford to do it again: it sums the producer's split-K
// planes, adds the residual, normalises and keeps the bf16 rows in LDS (20 KB
// of L2 reads a row of 2048 with two planes).  The arithmetic and its order
// are add_rmsnorm_kernel's, so the rows' bits are too.  One workgroup stores
// the new residual, into another buffer than the one all of them read.
#pragma once

#include "nq_common.h"
#include "nq_internal.h"

namespace nq {

constexpr int kNormRowsPlanes = 4;  // planes whose loads are in flight together (the most a source has)

struct NormRowsSrc {
    const float *planes;  // [S][M][K]
    int S;
    const uint16_t *residual_in;  // [M][K]
    uint16_t *residual_out;       // [M][K], not residual_in
    const uint16_t *weight;       // [K]
    float eps;
    uint16_t *x_out;  // [M][K] or null
};

// Rows of K, T threads, at most P * T * 8 / K rows: thread t holds the 8 columns t % (K / 8) of rows
// t / (K / 8) + p T / (K / 8).  load() issues every load (before the caller's weight loads, which the
// wait for these then leaves in flight); finish() hands out row, column and the normalised bf16 values.
template <int K, int T, int P>
struct NormRows {
    static constexpr int kVec = K / 8;             // threads a row
    static constexpr int kParts = kVec / kWave;    // waves a row
    static constexpr int kRows = P * T / kVec;     // the most rows
    static_assert(kVec % kWave == 0 && T % kVec == 0, "whole waves a row, one column a thread");
    float4 pl[P][kNormRowsPlanes][2];
    uint4 rb[P], wt;

    __device__ __forceinline__ void load(const NormRowsSrc &n, int M) {
        const int col = static_cast<int>(threadIdx.x) % kVec * 8;
        const int64_t plane = static_cast<int64_t>(M) * K;
#pragma unroll
        for (int p = 0; p < P; ++p) {
            const int row = static_cast<int>(threadIdx.x) / kVec + p * (T / kVec);
            if (row >= M) break;
            const int64_t at = static_cast<int64_t>(row) * K + col;
            rb[p] = *reinterpret_cast<const uint4 *>(n.residual_in + at);
#pragma unroll
            for (int s = 0; s < kNormRowsPlanes; ++s) {
                if (s >= n.S) break;
                pl[p][s][0] = *reinterpret_cast<const float4 *>(n.planes + s * plane + at);
                pl[p][s][1] = *reinterpret_cast<const float4 *>(n.planes + s * plane + at + 4);
            }
        }
        wt = *reinterpret_cast<const uint4 *>(n.weight + col);
    }

    // red: kRows * kParts floats of LDS.  Holds one barrier; the caller's next one covers what emit wrote.
    template <typename Emit>
    __device__ __forceinline__ void finish(const NormRowsSrc &n, int M, bool writer, float *red, Emit emit) {
        const int col = static_cast<int>(threadIdx.x) % kVec * 8;
        const int row0 = static_cast<int>(threadIdx.x) / kVec;
        const int lane = threadIdx.x & (kWave - 1);
        const int part = static_cast<int>(threadIdx.x) % kVec / kWave;
        uint4 h[P];
#pragma unroll
        for (int p = 0; p < P; ++p) {
            const int row = row0 + p * (T / kVec);
            if (row >= M) break;
            float x[8], b[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = 0.f;
#pragma unroll
            for (int s = 0; s < kNormRowsPlanes; ++s) {
                if (s >= n.S) break;
                const float4 u = pl[p][s][0], v = pl[p][s][1];
                x[0] += u.x; x[1] += u.y; x[2] += u.z; x[3] += u.w;
                x[4] += v.x; x[5] += v.y; x[6] += v.z; x[7] += v.w;
            }
            unpack8(rb[p], b);
            uint32_t *ph = reinterpret_cast<uint32_t *>(&h[p]);
#pragma unroll
            for (int e = 0; e < 8; e += 2)
                ph[e / 2] = pack2_bf16(bf16_to_f32(f32_to_bf16(x[e])) + b[e], bf16_to_f32(f32_to_bf16(x[e + 1])) + b[e + 1]);
            unpack8(h[p], x);
            float ss = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) ss += x[e] * x[e];
            ss = group_sum<kWave>(ss);
            if (lane == 0) red[row * kParts + part] = ss;
        }
        __syncthreads();
        float w[8];
        unpack8(wt, w);
#pragma unroll
        for (int p = 0; p < P; ++p) {
            const int row = row0 + p * (T / kVec);
            if (row >= M) break;
            float ss = 0.f;
#pragma unroll
            for (int i = 0; i < kParts; ++i) ss += red[row * kParts + i];
            const float inv = rsqrtf(ss / static_cast<float>(K) + n.eps);
            float x[8];
            unpack8(h[p], x);
            uint4 y;
            uint32_t *py = reinterpret_cast<uint32_t *>(&y);
#pragma unroll
            for (int e = 0; e < 8; e += 2) py[e / 2] = pack2_bf16(x[e] * inv * w[e], x[e + 1] * inv * w[e + 1]);
            emit(row, col, y);
            if (writer) {
                const int64_t at = static_cast<int64_t>(row) * K + col;
                *reinterpret_cast<uint4 *>(n.residual_out + at) = h[p];
                if (n.x_out) *reinterpret_cast<uint4 *>(n.x_out + at) = y;
            }
        }
    }
};

}  // namespace nq
