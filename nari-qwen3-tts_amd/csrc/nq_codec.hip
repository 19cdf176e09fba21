// Incremental codec-decoder step: the stateful kernels of a batch of streams
// decoded together (model/incremental_codec.py:58-466), fp32 like the
// reference codec (no autocast, executor/build.py:91-95).
//
// Layout.  Activations are channels-last [T, C] with the fresh rows of all
// streams concatenated: stream b owns rows [off[b] * u, off[b + 1] * u) of a
// stage whose time axis is u samples per codec frame (u = 1 at the frame rate,
// then x2, x4, x20 ... x2000 after the upsampling layers).  `off` is the
// frame-level exclusive prefix of the streams' fresh frame counts, so ragged
// chunks (12-48 frames) share every launch.  Each stream's state lives in slot
// slots[b] of per-layer device arrays:
//   - causal Conv1d history  [slots, pad, Cin]  (post-activation inputs)
//   - ConvTranspose1d overlap [slots, s, Cout]  (bias-free expansion tail)
//   - transformer K/V          [slots, R, H, D]  (rotated keys, R = window - 1)
//   - frame position / valid context count [slots]
// A conv or transconv reads the old state, then a second small kernel writes
// the new state in place (a workgroup per stream reads every element it needs
// before it writes the first).

#include "nq_common.h"

namespace nq {
namespace {

constexpr int kCodecThreads = 256;
constexpr int kCus = 256;  // compute units of the chip
// history_update_kernel covers pad * C <= 1024 * 4
constexpr int kHistoryThreads = 1024;
constexpr int kHistoryPerThread = 4;

// stream of stage row t: the largest b with off[b] * u <= t
__device__ __forceinline__ int stream_of(const int32_t *__restrict__ off, int B, int64_t t, int u) {
    int lo = 0, hi = B - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (static_cast<int64_t>(off[mid]) * u <= t) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// Tile `tile` of the streams' rows cut into tiles of at most `rows` rows that never cross a stream (tiles
// counted through the streams in order): every row before the tile's first one that a causal tap can
// read is then a row of the same stream or of its history.  The lanes of a wave count 64 streams at a
// time.  Like stream_of, the last stream reaches to row T.  False past the last tile; uniform over the
// workgroup.  At most T / rows + B tiles exist.
struct StreamTile {
    int b;          // stream
    int64_t first;  // its first row
    int64_t n;      // its rows
    int64_t l0;     // the tile's first row within it
};
__device__ __forceinline__ bool stream_tile(const int32_t *__restrict__ off, int B, int u, int64_t T, int rows,
                                            int tile, StreamTile &s) {
    const int lane = threadIdx.x & (kWave - 1);
    int before = 0;
    for (int b0 = 0; b0 < B; b0 += kWave) {
        const int b = b0 + lane;
        const int lo = off[b < B ? b : B], hi = off[b < B ? b + 1 : B];
        const int64_t end = b + 1 < B && static_cast<int64_t>(hi) * u < T ? static_cast<int64_t>(hi) * u : T;
        const int64_t n = end - static_cast<int64_t>(lo) * u;
        const int count = b < B && n > 0 ? static_cast<int>((n + rows - 1) / rows) : 0;
        int upto = count;
#pragma unroll
        for (int d = 1; d < kWave; d *= 2) {
            const int other = __shfl_up(upto, d, kWave);
            if (lane >= d) upto += other;
        }
        const uint64_t past = __ballot(before + upto > tile);
        if (past) {
            const int at = __builtin_ctzll(past);
            s.b = b0 + at;
            s.first = static_cast<int64_t>(__builtin_amdgcn_readlane(lo, at)) * u;
            const int64_t next = static_cast<int64_t>(__builtin_amdgcn_readlane(hi, at)) * u;
            s.n = (s.b + 1 < B && next < T ? next : T) - s.first;
            const int skipped = before + __builtin_amdgcn_readlane(upto - count, at);
            s.l0 = static_cast<int64_t>(tile - skipped) * rows;
            return true;
        }
        before += __builtin_amdgcn_readlane(upto, kWave - 1);
    }
    return false;
}

int stream_tiles_bound(int64_t T, int B, int rows) { return static_cast<int>(T / rows + (B < T ? B : T)); }

// SnakeBeta x + sin(a x)^2 / b with a = exp(alpha), b = exp(beta) (per channel)
__device__ __forceinline__ float snake(float x, float a, float inv_b) {
    const float s = __sinf(a * x);
    return x + inv_b * s * s;
}

struct Act {
    const float *alpha;  // log-scale, [C] or null (identity)
    const float *beta;
    __device__ __forceinline__ float a_of(int c) const { return expf(alpha[c]); }
    __device__ __forceinline__ float inv_b_of(int c) const { return 1.0f / (expf(beta[c]) + 1e-9f); }
    __device__ __forceinline__ float apply(float x, int c) const {
        if (!alpha) return x;
        return snake(x, a_of(c), inv_b_of(c));
    }
};

// ---------------------------------------------------------------------------
// codebook sum: out[t, c] = sum_q book[q, codes[t, q], c]

__global__ void __launch_bounds__(kCodecThreads)
embed_sum_kernel(const int32_t *__restrict__ codes, int T, int Q, const float *__restrict__ books, int V, int C,
                 float *__restrict__ out, int32_t *status) {
    const int64_t n = static_cast<int64_t>(T) * C;
    for (int64_t i = blockIdx.x * static_cast<int64_t>(kCodecThreads) + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * kCodecThreads) {
        const int64_t t = i / C;
        const int c = static_cast<int>(i - t * C);
        float s = 0.f;
        for (int q = 0; q < Q; ++q) {
            const int id = codes[t * Q + q];
            if (static_cast<unsigned>(id) >= static_cast<unsigned>(V)) {
                if (status) atomicExch(status, NQ_ERR_INVALID_ARGUMENT);
                continue;
            }
            s += books[(static_cast<int64_t>(q) * V + id) * C + c];
        }
        out[i] = s;
    }
}

// ---------------------------------------------------------------------------
// causal Conv1d (groups 1), direct form.  A workgroup covers 256 / CG rows and
// CG groups of 16 output channels; weights of 16 input channels x K taps are
// staged in LDS per round.  Row r, tap k reads input time local - (K-1-k)*dil
// of its own stream: from x when >= 0, else from the stream's history.

constexpr int kConvCi = 16;
constexpr int kConvKMax = 7;

template <int CG>
__global__ void __launch_bounds__(kCodecThreads)
conv_kernel(const float *__restrict__ x, int64_t ldx, int64_t T, const int32_t *__restrict__ off, int B, int u,
            const int32_t *__restrict__ slots, const float *__restrict__ hist, const float *__restrict__ w,
            const float *__restrict__ bias, int Cin, int Cout, int K, int dil, Act act,
            const float *__restrict__ res, int64_t ldres, float *__restrict__ out, int64_t ldo) {
    constexpr int kRows = kCodecThreads / CG;
    __shared__ float ws[CG * 16][kConvCi][kConvKMax];
    __shared__ float sa[kConvCi], sb[kConvCi];
    const int r = threadIdx.x % kRows;
    const int cg = threadIdx.x / kRows;
    const int64_t row = static_cast<int64_t>(blockIdx.x) * kRows + r;
    const int co0 = blockIdx.y * CG * 16;
    const int pad = (K - 1) * dil;
    const bool live = row < T;
    int b = 0;
    int64_t local = 0, base = 0;
    if (live) {
        b = stream_of(off, B, row, u);
        base = static_cast<int64_t>(off[b]) * u;
        local = row - base;
    }
    const float *hrow = hist + static_cast<int64_t>(live ? slots[b] : 0) * pad * Cin;
    float acc[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[j] = 0.f;

    for (int ci0 = 0; ci0 < Cin; ci0 += kConvCi) {
        const int nci = min(kConvCi, Cin - ci0);
        __syncthreads();
        for (int e = threadIdx.x; e < CG * 16 * kConvCi * K; e += kCodecThreads) {
            const int co = e / (kConvCi * K);
            const int rem = e - co * kConvCi * K;
            const int ci = rem / K, k = rem - ci * K;
            float v = 0.f;
            if (co0 + co < Cout && ci < nci) v = w[(static_cast<int64_t>(co0 + co) * Cin + ci0 + ci) * K + k];
            ws[co][ci][k] = v;
        }
        if (act.alpha && threadIdx.x < nci) {
            sa[threadIdx.x] = act.a_of(ci0 + threadIdx.x);
            sb[threadIdx.x] = act.inv_b_of(ci0 + threadIdx.x);
        }
        __syncthreads();
        if (!live) continue;
        for (int k = 0; k < K; ++k) {
            const int64_t src = local - static_cast<int64_t>(K - 1 - k) * dil;
            const float *p = src >= 0 ? x + (base + src) * ldx + ci0 : hrow + (pad + src) * Cin + ci0;
            const bool activate = src >= 0 && act.alpha;
            for (int ci = 0; ci < nci; ++ci) {
                float xv = p[ci];
                if (activate) xv = snake(xv, sa[ci], sb[ci]);
#pragma unroll
                for (int j = 0; j < 16; ++j) acc[j] += xv * ws[cg * 16 + j][ci][k];
            }
        }
    }
    if (!live) return;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const int co = co0 + cg * 16 + j;
        if (co >= Cout) break;
        float y = acc[j] + (bias ? bias[co] : 0.f);
        if (res) y += res[row * ldres + co];
        out[row * ldo + co] = y;
    }
}

// Narrow causal Conv1d (Cin, Cout <= 64): a workgroup owns 256 R rows of one stream, each thread every
// output channel of R of them (rows t, t + 256, ...), so each weight read from LDS feeds R rows.  The
// rows, and the `pad` rows before them (from the stream's history where they lie before its first
// fresh row), are staged in LDS, the fresh ones activated once (row pitch Cin + 1, so the 64 rows a wave
// reads at one channel hit distinct banks), with the weights as [ci][k][co]; every tap then reads LDS.
// Outputs (and the residual) move as float4 when the row strides allow it.
//
// kUnit: the decoder's whole residual unit in one launch (Cin == Cout == CO, seven taps):
// out = res + conv1x1(snake2(conv(snake1(x)) + bias)) + bias2, with res the
// input x itself.  The 1x1 convolution runs in registers on the thread's
// conv outputs (its weights [ci][co] in LDS), in the order of the separate
// 1x1 launch, so the bits are those of the two launches; the intermediate
// tensor never reaches memory.
//
// With tiles cut from the concatenated rows of all streams, a wave near a stream's start read every tap
// through generic pointers: one stream's 8000 rows of 8 channels took 14.7 us and take 10.1, 38 and
// 1.8 M rows 16 and 52 us (10.5 and 51), where the multiply-adds and the activation bound it.  A single
// output channel (the decoder's last convolution) computes one, not eight: 1.8 M rows 36 -> 24 us.
template <int CO, int R, bool kUnit = false>
__global__ void __launch_bounds__(kCodecThreads)
conv_small_kernel(const float *__restrict__ x, int64_t ldx, int64_t T, const int32_t *__restrict__ off, int B, int u,
                  const int32_t *__restrict__ slots, const float *__restrict__ hist, const float *__restrict__ w,
                  const float *__restrict__ bias, int cin, int Cout, int taps, int dil, Act act,
                  const float *__restrict__ res, int64_t ldres, float *__restrict__ out, int64_t ldo,
                  const float *__restrict__ w2 = nullptr, const float *__restrict__ bias2 = nullptr,
                  Act act2 = Act{nullptr, nullptr}) {
    constexpr int ROWS = kCodecThreads * R;
    extern __shared__ float lds[];
    const int Cin = kUnit ? CO : cin, K = kUnit ? kConvKMax : taps;
    const int pad = (K - 1) * dil;
    const int pitch = Cin + 1;
    float *xs = lds;                                            // [(ROWS + pad) * pitch]
    float *wsm = xs + ((ROWS + pad) * pitch + 3) / 4 * 4;       // [Cin * K * CO], 16-byte aligned
    float *sa = wsm + Cin * K * CO;                             // [Cin]
    float *sb = sa + Cin;                                       // [Cin]
    float *w2s = sb + Cin + (kUnit ? (4 - (Cin * K * CO + 2 * Cin) % 4) % 4 : 0);  // [Cin][CO], 16-byte aligned
    float *sa2 = w2s + Cin * CO;                                // [Cin]
    float *sb2 = sa2 + Cin;                                     // [Cin]
    StreamTile st;
    if (!stream_tile(off, B, u, T, ROWS, static_cast<int>(blockIdx.x), st)) return;
    x += st.first * ldx;
    if (res) res += st.first * ldres;
    out += st.first * ldo;
    // row -1 lies before h
    const float *h = pad ? hist + (static_cast<int64_t>(slots[st.b]) * pad + pad) * Cin : nullptr;
    for (int e = threadIdx.x; e < Cin * K * CO; e += kCodecThreads) {
        const int co = e % CO;
        const int ck = e / CO;
        const int ci = ck / K, k = ck - ci * K;
        wsm[e] = co < Cout ? w[(static_cast<int64_t>(co) * Cin + ci) * K + k] : 0.f;
    }
    if (act.alpha && threadIdx.x < Cin) {
        sa[threadIdx.x] = act.a_of(threadIdx.x);
        sb[threadIdx.x] = act.inv_b_of(threadIdx.x);
    }
    if constexpr (kUnit) {
        for (int e = threadIdx.x; e < Cin * CO; e += kCodecThreads) {
            const int co = e % CO, ci = e / CO;
            w2s[e] = w2[static_cast<int64_t>(co) * Cin + ci];
        }
        if (act2.alpha && threadIdx.x < Cin) {
            sa2[threadIdx.x] = act2.a_of(threadIdx.x);
            sb2[threadIdx.x] = act2.inv_b_of(threadIdx.x);
        }
    }
    __syncthreads();
    // staged row rr is row l0 - pad + rr of the stream (the last one again past its end: those feed no
    // stored output)
    auto source = [&](int rr, int64_t &l) {
        l = st.l0 - pad + rr;
        if (l >= st.n) l = st.n - 1;
        return l < 0 ? h + l * Cin : x + l * ldx;
    };
    if ((Cin & 3) == 0 && (ldx & 3) == 0 &&
        ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(h)) & 15) == 0) {
        // 128-bit loads, kBatch per thread in flight before any is activated and stored
        constexpr int kBatch = R == 1 ? 4 : 8;
        const int vpr = Cin / 4;
        const int nvec = (ROWS + pad) * vpr;
        for (int e0 = threadIdx.x; e0 < nvec; e0 += kBatch * kCodecThreads) {
            float4 v[kBatch];
#pragma unroll
            for (int i = 0; i < kBatch; ++i) {
                const int e = e0 + i * kCodecThreads < nvec ? e0 + i * kCodecThreads : nvec - 1;
                const int rr = e / vpr;
                int64_t l;
                v[i] = *reinterpret_cast<const float4 *>(source(rr, l) + (e - rr * vpr) * 4);
            }
#pragma unroll
            for (int i = 0; i < kBatch; ++i) {
                const int e = e0 + i * kCodecThreads;
                if (e >= nvec) break;
                const int rr = e / vpr, c = (e - rr * vpr) * 4;
                float f[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
                if (act.alpha && st.l0 - pad + rr >= 0) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) f[q] = snake(f[q], sa[c + q], sb[c + q]);
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) xs[rr * pitch + c + q] = f[q];
            }
        }
    } else {
        for (int e = threadIdx.x; e < (ROWS + pad) * Cin; e += kCodecThreads) {
            const int rr = e / Cin, c = e - rr * Cin;
            int64_t l;
            float v = source(rr, l)[c];
            if (act.alpha && l >= 0) v = snake(v, sa[c], sb[c]);
            xs[rr * pitch + c] = v;
        }
    }
    __syncthreads();
    float acc[R][CO];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int j = 0; j < CO; ++j) acc[r][j] = 0.f;
    // one tap's multiply-adds over the input channels: the rows' inputs xr[r][ci], the weights at wk
    // ([ci][k][co] with row pitch kw floats)
    auto channel_loop = [&](const float *const (&xr)[R], const float *wk, int kw) {
        for (int ci = 0; ci < Cin; ++ci) {
            float xv[R];
#pragma unroll
            for (int r = 0; r < R; ++r) xv[r] = xr[r][ci];
            if constexpr (CO % 4 == 0) {
                const float4 *w4 = reinterpret_cast<const float4 *>(wk + ci * kw);
#pragma unroll
                for (int j = 0; j < CO / 4; ++j) {
                    const float4 ww = w4[j];
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        acc[r][4 * j] += xv[r] * ww.x;
                        acc[r][4 * j + 1] += xv[r] * ww.y;
                        acc[r][4 * j + 2] += xv[r] * ww.z;
                        acc[r][4 * j + 3] += xv[r] * ww.w;
                    }
                }
            } else {
#pragma unroll
                for (int j = 0; j < CO; ++j) {
                    const float ww = wk[ci * kw + j];
#pragma unroll
                    for (int r = 0; r < R; ++r) acc[r][j] += xv[r] * ww;
                }
            }
        }
    };
    for (int k = 0; k < K; ++k) {
        const float *xr[R];
#pragma unroll
        for (int r = 0; r < R; ++r) xr[r] = xs + (threadIdx.x + r * kCodecThreads + k * dil) * pitch;
        channel_loop(xr, wsm + k * CO, K * CO);
    }
    if constexpr (kUnit) {
        // the 1x1 convolution of snake2(conv + bias): each thread parks its rows' activated conv
        // outputs in its own rows of the (now free) staging area and reads them back per channel
        __syncthreads();
        const float *yr[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            float *yw = xs + (threadIdx.x + r * kCodecThreads) * pitch;
#pragma unroll
            for (int j = 0; j < CO; ++j) {
                const float y = acc[r][j] + (bias ? bias[j] : 0.f);
                yw[j] = act2.alpha ? snake(y, sa2[j], sb2[j]) : y;
                acc[r][j] = 0.f;
            }
            yr[r] = yw;
        }
        channel_loop(yr, w2s, CO);
        bias = bias2;
    }
    const bool vec = CO % 4 == 0 && Cout == CO && (ldo & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0 &&
                     (!res || ((ldres & 3) == 0 && (reinterpret_cast<uintptr_t>(res) & 15) == 0));
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int64_t row = st.l0 + threadIdx.x + r * kCodecThreads;
        if (row >= st.n) break;
        if (vec) {
#pragma unroll
            for (int j = 0; j < CO / 4; ++j) {
                float4 y = make_float4(acc[r][4 * j], acc[r][4 * j + 1], acc[r][4 * j + 2], acc[r][4 * j + 3]);
                if (bias) {
                    y.x += bias[4 * j];
                    y.y += bias[4 * j + 1];
                    y.z += bias[4 * j + 2];
                    y.w += bias[4 * j + 3];
                }
                if (res) {
                    const float4 q = *reinterpret_cast<const float4 *>(res + row * ldres + 4 * j);
                    y.x += q.x;
                    y.y += q.y;
                    y.z += q.z;
                    y.w += q.w;
                }
                *reinterpret_cast<float4 *>(out + row * ldo + 4 * j) = y;
            }
        } else {
#pragma unroll
            for (int j = 0; j < CO; ++j) {
                if (j >= Cout) break;
                float y = acc[r][j] + (bias ? bias[j] : 0.f);
                if (res) y += res[row * ldres + j];
                out[row * ldo + j] = y;
            }
        }
    }
}

size_t conv_small_lds(int Cin, int K, int dil, int CO, int R, bool unit = false) {
    const size_t rows = static_cast<size_t>(kCodecThreads) * R;
    const size_t unit_floats = unit ? 3 + static_cast<size_t>(Cin) * CO + 2 * Cin : 0;
    return ((rows + (K - 1) * dil) * (Cin + 1) + 3 + static_cast<size_t>(Cin) * K * CO + 2 * Cin + unit_floats) *
           sizeof(float);
}

constexpr size_t kConvLds = 150 * 1024;

// Rows per thread of the narrow convolution: two while the tiles then still fill the chip, one below a
// 256-row tile per CU, where the time is one tile's chain (8000 rows of 8 channels 10.1 us against 12.5;
// 192,000 rows 25.1 against 15.0).  More than 16 channels take one (their sums fill the registers).
int conv_small_rows(int CO, int64_t T, int B) {
    return CO <= 16 && stream_tiles_bound(T, B, kCodecThreads) > kCus ? 2 : 1;
}

// depthwise causal Conv1d (groups == C): one thread per (row, channel)
__global__ void __launch_bounds__(kCodecThreads)
dwconv_kernel(const float *__restrict__ x, int64_t ldx, int64_t T, const int32_t *__restrict__ off, int B, int u,
              const int32_t *__restrict__ slots, const float *__restrict__ hist, const float *__restrict__ w,
              const float *__restrict__ bias, int C, int K, int dil, float *__restrict__ out, int64_t ldo) {
    const int64_t n = T * C;
    const int pad = (K - 1) * dil;
    for (int64_t i = blockIdx.x * static_cast<int64_t>(kCodecThreads) + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * kCodecThreads) {
        const int64_t row = i / C;
        const int c = static_cast<int>(i - row * C);
        const int b = stream_of(off, B, row, u);
        const int64_t base = static_cast<int64_t>(off[b]) * u;
        const int64_t local = row - base;
        const float *hrow = hist + static_cast<int64_t>(slots[b]) * pad * C;
        float y = bias ? bias[c] : 0.f;
        for (int k = 0; k < K; ++k) {
            const int64_t src = local - static_cast<int64_t>(K - 1 - k) * dil;
            const float xv = src >= 0 ? x[(base + src) * ldx + c] : hrow[(pad + src) * C + c];
            y += xv * w[c * K + k];
        }
        out[row * ldo + c] = y;
    }
}

// ---------------------------------------------------------------------------
// Staging of per-stream state tensors (the reference's state objects) into a
// state pool's rows and back, every tensor of up to kStateRows streams in one
// launch.  A state tensor is [A][B][inner], its pool row [B][A][inner]; its
// address travels in the kernel's arguments.  A stream has 39 such tensors of
// 0.2 to 51 KB, so the cost is launches: stacking, transposing and copying
// them one kind at a time took 116 launches and 273 us of a captured
// one-stream step (1324 -> 1053 us with two).

constexpr int kStateKinds = 40;
constexpr int kStateRows = 9;
constexpr int kStateThreads = 1024;

struct StateKind {
    float *pool;
    int row_stride, a, b, inner;
};
struct StateArgs {
    StateKind kind[kStateKinds];
    float *state[kStateRows][kStateKinds];
    const int64_t *position;  // fills frame_pos when given
    int64_t position_stride;
    int64_t *frame_pos;
    const int64_t *context;  // fills ctx_len when given
    int32_t *ctx_len;
};
static_assert(sizeof(StateArgs) <= 4096, "kernel arguments hold 4 KB");

template <bool kToPool>
__global__ void __launch_bounds__(kStateThreads) state_copy_kernel(const StateArgs args) {
    const int row = blockIdx.y;
    const StateKind k = args.kind[blockIdx.x];
    float *state = args.state[row][blockIdx.x];
    float *pool = k.pool + static_cast<int64_t>(row) * k.row_stride;
    if (kToPool && blockIdx.x == 0 && threadIdx.x == 0) {
        if (args.position) args.frame_pos[row] = args.position[row * args.position_stride];
        if (args.context) args.ctx_len[row] = static_cast<int32_t>(args.context[row]);
    }
    const bool vec = k.inner % 4 == 0;  // the host checked that the addresses are 16-byte aligned then
    const int inner = vec ? k.inner / 4 : k.inner;
    const int n = k.a * k.b * inner;
    for (int e = threadIdx.x; e < n; e += kStateThreads) {
        // consecutive threads write consecutive elements
        const int i = e % inner, rest = e / inner;
        const int lo = kToPool ? rest % k.a : rest % k.b, hi = kToPool ? rest / k.a : rest / k.b;
        const int from = (kToPool ? lo * k.b + hi : lo * k.a + hi) * inner + i;
        if (vec) {
            float4 *dst = reinterpret_cast<float4 *>(kToPool ? pool : state);
            const float4 *src = reinterpret_cast<const float4 *>(kToPool ? state : pool);
            dst[e] = src ? src[from] : make_float4(0.f, 0.f, 0.f, 0.f);
        } else {
            float *dst = kToPool ? pool : state;
            const float *src = kToPool ? state : pool;
            dst[e] = src ? src[from] : 0.f;
        }
    }
}

// new history = last pad rows of [history ; act(x)] per stream.  1024 threads of four elements: with 256
// of sixteen the unrolled activations were 11 KB of code, whose fetch a launch of one workgroup waits for.
__global__ void __launch_bounds__(kHistoryThreads)
history_update_kernel(const float *__restrict__ x, int64_t ldx, const int32_t *__restrict__ off, int B, int u,
                      const int32_t *__restrict__ slots, float *__restrict__ hist, int C, int pad, Act act) {
    // one workgroup per stream: every (j, c) of its [pad, C] history is read first (the entries that
    // shift down and the fresh tail rows, activated), then all are written after a barrier, so no
    // entry is overwritten before it is read
    constexpr int kPer = kHistoryPerThread;
    const int b = blockIdx.x;
    const int64_t base = static_cast<int64_t>(off[b]) * u;
    const int64_t F = static_cast<int64_t>(off[b + 1]) * u - base;
    float *h = hist + static_cast<int64_t>(slots[b]) * pad * C;
    const int n = pad * C;
    float v[kPer];
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const int e = threadIdx.x + i * kHistoryThreads;
        v[i] = 0.f;
        if (e < n) {
            const int j = e / C, c = e - j * C;
            v[i] = j + F < pad ? h[(j + F) * C + c] : act.apply(x[(base + F - pad + j) * ldx + c], c);
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const int e = threadIdx.x + i * kHistoryThreads;
        if (e < n) h[e] = v[i];
    }
}

// ---------------------------------------------------------------------------
// causal ConvTranspose1d, kernel 2s, stride s, overlap s.  Output row p of a
// stream (stage u * s): t0 = p / s, j = p % s,
//   y = bias + x[t0] . W[:, :, j] + (t0 > 0 ? x[t0 - 1] . W[:, :, j + s] : overlap[j])

template <int CG>
__global__ void __launch_bounds__(kCodecThreads)
transconv_kernel(const float *__restrict__ x, int64_t ldx, int64_t T_out, const int32_t *__restrict__ off, int B,
                 int u_in, int s, const int32_t *__restrict__ slots, const float *__restrict__ overlap,
                 const float *__restrict__ w, const float *__restrict__ bias, int Cin, int Cout, Act act,
                 float *__restrict__ out, int64_t ldo) {
    constexpr int kRows = kCodecThreads / CG;
    extern __shared__ float tw[];  // [16 ci][CG*16 co][2s]
    __shared__ float sa[kConvCi], sb[kConvCi];
    const int r = threadIdx.x % kRows;
    const int cg = threadIdx.x / kRows;
    const int64_t row = static_cast<int64_t>(blockIdx.x) * kRows + r;
    const int co0 = blockIdx.y * CG * 16;
    const int u_out = u_in * s;
    const bool live = row < T_out;
    int b = 0;
    int64_t local = 0, base_in = 0;
    if (live) {
        b = stream_of(off, B, row, u_out);
        local = row - static_cast<int64_t>(off[b]) * u_out;
        base_in = static_cast<int64_t>(off[b]) * u_in;
    }
    const int64_t t0 = local / s;
    const int j = static_cast<int>(local - t0 * s);
    float acc[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) acc[q] = 0.f;
    const int ks = 2 * s;
    for (int ci0 = 0; ci0 < Cin; ci0 += kConvCi) {
        const int nci = min(kConvCi, Cin - ci0);
        __syncthreads();
        for (int e = threadIdx.x; e < kConvCi * CG * 16 * ks; e += kCodecThreads) {
            const int ci = e / (CG * 16 * ks);
            const int rem = e - ci * CG * 16 * ks;
            const int co = rem / ks, k = rem - co * ks;
            float v = 0.f;
            if (ci < nci && co0 + co < Cout) v = w[(static_cast<int64_t>(ci0 + ci) * Cout + co0 + co) * ks + k];
            tw[e] = v;
        }
        if (act.alpha && threadIdx.x < nci) {
            sa[threadIdx.x] = act.a_of(ci0 + threadIdx.x);
            sb[threadIdx.x] = act.inv_b_of(ci0 + threadIdx.x);
        }
        __syncthreads();
        if (!live) continue;
        const float *x1 = x + (base_in + t0) * ldx + ci0;
        const float *x0 = t0 > 0 ? x + (base_in + t0 - 1) * ldx + ci0 : nullptr;
        for (int ci = 0; ci < nci; ++ci) {
            float a1 = x1[ci], a0 = x0 ? x0[ci] : 0.f;
            if (act.alpha) {
                a1 = snake(a1, sa[ci], sb[ci]);
                if (x0) a0 = snake(a0, sa[ci], sb[ci]);
            }
            const float *wr = tw + (ci * CG * 16 + cg * 16) * ks;
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[q] += a1 * wr[q * ks + j] + a0 * wr[q * ks + j + s];
        }
    }
    if (!live) return;
    const float *ov = overlap + (static_cast<int64_t>(slots[b]) * s + j) * Cout;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        const int co = co0 + cg * 16 + q;
        if (co >= Cout) break;
        float y = acc[q] + (bias ? bias[co] : 0.f);
        if (t0 == 0) y += ov[co];
        out[row * ldo + co] = y;
    }
}

// Narrow causal transposed Conv1d (Cout <= 16, stride s): output row r reads input
// rows r / s and r / s - 1 (the stream's rows are aligned to s at this stage).
// The workgroup stages the (at most 256 / s + 3) input rows its 256 output rows read,
// activated once, in LDS (row pitch Cin + 1) with the weights as [ci][2s][co];
// the first output rows of a stream add its carried overlap instead of an
// earlier input row.  Outputs move as float4 when the row stride allows it.
// With one or a few streams the staging is the time, so its loads are in
// flight together; with many the weights' LDS reads, so they lie with the
// output channels together and are read four at a time: 32 -> 16 channels, s =
// 4: 1600 rows 28 -> 15 us, 363,000 rows 48.7 -> 31.6; 16 -> 8, s = 5: 8000
// rows 10.3 -> 7.5, 1.8 M rows 57 -> 45.
template <int CO>
__global__ void __launch_bounds__(kCodecThreads)
transconv_small_kernel(const float *__restrict__ x, int64_t ldx, int64_t T_out, const int32_t *__restrict__ off,
                       int B, int u_in, int s, const int32_t *__restrict__ slots, const float *__restrict__ overlap,
                       const float *__restrict__ w, const float *__restrict__ bias, int Cin, int Cout, Act act,
                       float *__restrict__ out, int64_t ldo) {
    extern __shared__ float lds[];
    const int ks = 2 * s;
    const int pitch = Cin + 1;
    const int n_max = kCodecThreads / s + 3;  // >= the staged rows for every stride
    float *xs = lds;                                    // [n_max * pitch]
    float *tw = xs + (n_max * pitch + 3) / 4 * 4;       // [Cin][2s][CO], 16-byte aligned
    float *sa = tw + Cin * CO * ks;                     // [Cin]
    float *sb = sa + Cin;                               // [Cin]
    const int64_t T_in = T_out / s;
    const int64_t row0 = static_cast<int64_t>(blockIdx.x) * kCodecThreads;
    const int64_t last = row0 + kCodecThreads - 1 < T_out ? row0 + kCodecThreads - 1 : T_out - 1;
    const int64_t in0 = row0 / s - 1;  // staged input row 0 (may be -1)
    const int n_in = static_cast<int>(last / s - in0 + 1);
    // eight weights, and four 128-bit pieces of the rows, requested before the first is stored
    const int nw = Cin * Cout * ks;
    for (int e0 = threadIdx.x; e0 < nw; e0 += 8 * kCodecThreads) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = w[e0 + i * kCodecThreads < nw ? e0 + i * kCodecThreads : nw - 1];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int e = e0 + i * kCodecThreads;
            if (e >= nw) break;
            const int cc = e / ks, k = e - cc * ks;
            const int ci = Cout == CO ? cc / CO : cc / Cout;
            tw[(ci * ks + k) * CO + cc - ci * Cout] = v[i];
        }
    }
    if (act.alpha && threadIdx.x < Cin) {
        sa[threadIdx.x] = act.a_of(threadIdx.x);
        sb[threadIdx.x] = act.inv_b_of(threadIdx.x);
    }
    __syncthreads();
    if ((Cin & 3) == 0 && (ldx & 3) == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0) {
        const int vpr = Cin / 4, nvec = n_in * vpr;
        for (int e0 = threadIdx.x; e0 < nvec; e0 += 4 * kCodecThreads) {
            float4 v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int e = e0 + i * kCodecThreads < nvec ? e0 + i * kCodecThreads : nvec - 1;
                const int rr = e / vpr;
                const int64_t g = in0 + rr < 0 ? 0 : in0 + rr < T_in ? in0 + rr : T_in - 1;
                v[i] = *reinterpret_cast<const float4 *>(x + g * ldx + (e - rr * vpr) * 4);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int e = e0 + i * kCodecThreads;
                if (e >= nvec) break;
                const int rr = e / vpr, c = (e - rr * vpr) * 4;
                const float f[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    xs[rr * pitch + c + q] = act.alpha ? snake(f[q], sa[c + q], sb[c + q]) : f[q];
            }
        }
    } else {
        for (int e = threadIdx.x; e < n_in * Cin; e += kCodecThreads) {
            const int rr = e / Cin, c = e - rr * Cin;
            const int64_t g = in0 + rr;
            float v = 0.f;
            if (g >= 0 && g < T_in) {
                v = x[g * ldx + c];
                if (act.alpha) v = snake(v, sa[c], sb[c]);
            }
            xs[rr * pitch + c] = v;
        }
    }
    __syncthreads();
    const int64_t row = row0 + threadIdx.x;
    if (row >= T_out) return;
    const int u_out = u_in * s;
    const int b = stream_of(off, B, row, u_out);
    const int64_t gi = row / s;
    const int j = static_cast<int>(row - gi * s);
    const bool first = gi == static_cast<int64_t>(off[b]) * u_in;  // the stream's first input row
    const float *x1 = xs + (gi - in0) * pitch;
    const float *x0 = x1 - pitch;
    float acc[CO];
#pragma unroll
    for (int q = 0; q < CO; ++q) acc[q] = 0.f;
    for (int ci = 0; ci < Cin; ++ci) {
        const float a1 = x1[ci], a0 = first ? 0.f : x0[ci];
        const float4 *w1 = reinterpret_cast<const float4 *>(tw + (ci * ks + j) * CO);
        const float4 *w0 = w1 + s * (CO / 4);
#pragma unroll
        for (int q = 0; q < CO / 4; ++q) {
            const float4 u1 = w1[q], u0 = w0[q];
            acc[4 * q] += a1 * u1.x + a0 * u0.x;
            acc[4 * q + 1] += a1 * u1.y + a0 * u0.y;
            acc[4 * q + 2] += a1 * u1.z + a0 * u0.z;
            acc[4 * q + 3] += a1 * u1.w + a0 * u0.w;
        }
    }
    const float *ov = overlap + (static_cast<int64_t>(slots[b]) * s + j) * Cout;
    float y[CO];
#pragma unroll
    for (int q = 0; q < CO; ++q) {
        y[q] = acc[q] + (bias && q < Cout ? bias[q] : 0.f);
        if (first && q < Cout) y[q] += ov[q];
    }
    if (Cout == CO && (ldo & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0) {
#pragma unroll
        for (int q = 0; q < CO; q += 4)
            *reinterpret_cast<float4 *>(out + row * ldo + q) = make_float4(y[q], y[q + 1], y[q + 2], y[q + 3]);
    } else {
#pragma unroll
        for (int q = 0; q < CO; ++q)
            if (q < Cout) out[row * ldo + q] = y[q];
    }
}

size_t transconv_small_lds(int Cin, int s, int CO) {
    const size_t n_max = kCodecThreads / s + 3;
    return ((n_max * (Cin + 1) + 3) / 4 * 4 + static_cast<size_t>(Cin) * CO * 2 * s + 2 * Cin) * sizeof(float);
}

// new overlap[j, co] = act(x[F - 1]) . W[:, co, s + j]; a workgroup per (stream, 256 outputs), the row
// activated once in LDS and sixteen weights in flight (a thread that did both channel by channel, every
// load waited for, took 7.5 us at one stream and 14.3 at 32; this 4.2
// and 4.6)
__global__ void __launch_bounds__(kCodecThreads)
overlap_update_kernel(const float *__restrict__ x, int64_t ldx, const int32_t *__restrict__ off, int u_in, int s,
                      const int32_t *__restrict__ slots, float *__restrict__ overlap, const float *__restrict__ w,
                      int Cin, int Cout, Act act) {
    __shared__ float xa[kCodecThreads];
    const int b = blockIdx.x;
    const int64_t base = static_cast<int64_t>(off[b]) * u_in;
    const int64_t F = static_cast<int64_t>(off[b + 1]) * u_in - base;
    if (F <= 0) return;  // no fresh input: the stored overlap stays
    const float *xl = x + (base + F - 1) * ldx;
    const int n = s * Cout, e = blockIdx.y * kCodecThreads + threadIdx.x;
    const int co = (e < n ? e : n - 1) / s, j = (e < n ? e : n - 1) - co * s;
    const float *wp = w + static_cast<int64_t>(co) * 2 * s + s + j;
    const int64_t step = static_cast<int64_t>(Cout) * 2 * s;
    float sum = 0.f;
    for (int c0 = 0; c0 < Cin; c0 += kCodecThreads) {
        const int m = Cin - c0 < kCodecThreads ? Cin - c0 : kCodecThreads;
        if (c0) __syncthreads();
        if (static_cast<int>(threadIdx.x) < m) xa[threadIdx.x] = act.apply(xl[c0 + threadIdx.x], c0 + threadIdx.x);
        __syncthreads();
#pragma unroll 16
        for (int i = 0; i < m; ++i) sum += xa[i] * wp[(c0 + i) * step];
    }
    if (e < n) overlap[(static_cast<int64_t>(slots[b]) * s + j) * Cout + co] = sum;
}

// ---------------------------------------------------------------------------
// Gathered operand for running a wide conv or transconv as one GEMM.
//   conv:      A[t, k*Cin + ci] = input of row t at tap k (activated x, or raw history)
//   transconv: A[t, ci] = act(x[t]), A[t, Cin + ci] = act(x[t - 1]) (0 for a stream's
//              first fresh frame; its overlap is added after the GEMM)
// One thread per (row, 4 channels); Cin % 4 == 0.

__global__ void __launch_bounds__(kCodecThreads)
im2col_kernel(const float *__restrict__ x, int64_t ldx, int64_t T, const int32_t *__restrict__ off, int B, int u,
              const int32_t *__restrict__ slots, const float *__restrict__ hist, int Cin, int K, int dil, int transconv,
              Act act, float *__restrict__ a, int64_t lda) {
    const int c4 = Cin / 4;
    const int64_t n = T * K * c4;
    const int pad = transconv ? 0 : (K - 1) * dil;
    for (int64_t i = blockIdx.x * static_cast<int64_t>(kCodecThreads) + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * kCodecThreads) {
        const int64_t row = i / (K * c4);
        const int rem = static_cast<int>(i - row * K * c4);
        const int k = rem / c4, c = (rem - k * c4) * 4;
        const int b = stream_of(off, B, row, u);
        const int64_t base = static_cast<int64_t>(off[b]) * u;
        const int64_t local = row - base;
        const int64_t src = transconv ? local - k : local - static_cast<int64_t>(K - 1 - k) * dil;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (src >= 0) {
            v = *reinterpret_cast<const float4 *>(x + (base + src) * ldx + c);
            if (act.alpha) {
                v.x = act.apply(v.x, c);
                v.y = act.apply(v.y, c + 1);
                v.z = act.apply(v.z, c + 2);
                v.w = act.apply(v.w, c + 3);
            }
        } else if (!transconv) {
            v = *reinterpret_cast<const float4 *>(hist + (static_cast<int64_t>(slots[b]) * pad + pad + src) * Cin + c);
        }
        *reinterpret_cast<float4 *>(a + row * lda + static_cast<int64_t>(k) * Cin + c) = v;
    }
}

// GEMM-path transconv: add the stored overlap to each stream's first `s`
// output rows, then store the new overlap, which the caller computed as
// (last fresh frame) x (kernel tail): new_ov [B, s * Cout].  Thread per
// (stream, j, co) touches one overlap element only.
__global__ void __launch_bounds__(kCodecThreads)
overlap_fixup_kernel(const int32_t *__restrict__ off, int B, int u_in, int s, const int32_t *__restrict__ slots,
                     float *__restrict__ overlap, const float *__restrict__ new_ov, int Cout, float *__restrict__ out,
                     int64_t ldo) {
    const int64_t i = blockIdx.x * static_cast<int64_t>(kCodecThreads) + threadIdx.x;
    if (i >= static_cast<int64_t>(B) * s * Cout) return;
    const int b = static_cast<int>(i / (static_cast<int64_t>(s) * Cout));
    const int rem = static_cast<int>(i - static_cast<int64_t>(b) * s * Cout);
    const int j = rem / Cout, co = rem - j * Cout;
    const int64_t base = static_cast<int64_t>(off[b]) * u_in;
    const int64_t F = static_cast<int64_t>(off[b + 1]) * u_in - base;
    if (F <= 0) return;
    float *ov = overlap + (static_cast<int64_t>(slots[b]) * s + j) * Cout + co;
    out[(base * s + j) * ldo + co] += *ov;
    *ov = new_ov[static_cast<int64_t>(b) * s * Cout + rem];
}

// ---------------------------------------------------------------------------
// transformer attention of one (stream, head): per-head RMSNorm + RoPE of q
// and of the fresh k (positions = frame_position[slot] + fresh index), the
// sliding-window attention over [retained R frames ; fresh frames], and the
// retained K/V advance, in one workgroup (_pre_transformer, :193-381).
//
// Query i of the stream (position P0 + i) sees the positions P0 + i - R ..
// P0 + i: retained slot j (position P0 - R + j) when j >= R - ctx and j >= i,
// fresh frame f when i - R <= f <= i.  The fresh queries go in blocks of 64;
// for block i0 the key rows are the positions P0 + i0 - R + kappa, kappa in
// [0, R + nq): a retained slot (already rotated in the state) while
// i0 - R + kappa < 0, else fresh frame f = i0 - R + kappa, rotated here (and
// written back in place, so a later block reads it rotated) unless an earlier
// block already did.  K, V and the rotated q of a block are staged in LDS
// (rows of D + 4 floats).  Thirty-two queries then go at a time, a thread each
// (query j, window step s), which reads key row j + s: 32 lanes read 32
// consecutive rows, and a 16-byte read spreads over the banks.  A query's
// scores lie in half a wave, which finds its softmax with shuffles and takes
// its channels for P V.  What bounds a launch is this chain, and the code it
// is written in: with a query a lane and the window's steps unrolled (25 KB
// of code, four lanes of 64 at work on a four-frame chunk) a launch took
// 17 us at one stream of four frames and 18.5 us at 32 of 12 - 48, and takes
// 5.6 and 11.0.  A CU holds one workgroup, so its threads are 1024: with 256
// the 32 streams took 18.1, with 512 13.2.  After the last block the new
// retained rows (the last R positions) are written from LDS: the state is read
// (staged) before this workgroup overwrites it, and no other workgroup touches
// this (stream, head).

constexpr int kWinThreads = 1024;
constexpr int kWinQ = 64;     // queries per block
constexpr int kWinMax = 32;   // window (R + 1) the kernel takes
constexpr int kWinGroup = kWinThreads / kWinMax;  // queries whose (query, step) pairs are one per thread

template <int D>
__global__ void __launch_bounds__(kWinThreads)
window_block_kernel(const float *__restrict__ q, float *__restrict__ k, const float *__restrict__ v, int64_t ld,
                    int H, const float *__restrict__ qn, const float *__restrict__ kn, float eps, float log_theta,
                    const int32_t *__restrict__ off, const int32_t *__restrict__ slots,
                    const int64_t *__restrict__ frame_pos, const int32_t *__restrict__ ctx_len, float *state_k,
                    float *state_v, int64_t state_slot_stride, int R, float scale, float *__restrict__ out,
                    int64_t ldo) {
    static_assert(D % 16 == 0 && D <= 64, "rows of 4-channel chunks, whole rows a pass");
    constexpr int P = D + 4;                // LDS row pitch (floats)
    constexpr int LPR = D / 4;              // lanes (4-channel chunks) per row
    constexpr int RPP = kWinThreads / LPR;  // rows staged per pass
    constexpr int HALF = D / 2;             // rotated pairs
    static_assert(kWinThreads % HALF == 0, "a thread makes the angles of one pair");
    __shared__ __attribute__((aligned(16))) float ks[(kWinMax - 1 + kWinQ) * P];
    __shared__ __attribute__((aligned(16))) float vs[(kWinMax - 1 + kWinQ) * P];
    __shared__ __attribute__((aligned(16))) float qs[kWinQ * P];
    __shared__ float ps[kWinThreads];
    __shared__ __attribute__((aligned(16))) float cosines[kWinQ * HALF];
    __shared__ __attribute__((aligned(16))) float sines[kWinQ * HALF];

    const int b = blockIdx.x / H, h = blockIdx.x - (blockIdx.x / H) * H;
    const int64_t t0 = off[b];
    const int F = off[b + 1] - off[b];
    if (F <= 0) return;  // no fresh frames: nothing attends and the state stays as it is
    const int slot = slots[b];
    const int ctx = ctx_len[slot];
    const int64_t P0 = frame_pos[slot];
    const int W = R + 1;
    const int c = threadIdx.x % LPR;  // the thread's 4-channel chunk when staging
    float *sk = state_k + static_cast<int64_t>(slot) * state_slot_stride + h * D;
    float *sv = state_v + static_cast<int64_t>(slot) * state_slot_stride + h * D;
    const int64_t srow = static_cast<int64_t>(H) * D;  // state row stride

    // RMSNorm (weight wn) + rotate-half RoPE of a row held as one 4-channel chunk per lane of its
    // LPR-lane group: the group sums the squares, and chunk c pairs with chunk c ^ (LPR / 2)
    // (channels d and d + D / 2, inv_freq of pair d = theta^(-2d/D)), as the reference rotates them.
    // The block's cosines and sines are made once, in LDS, while its loads are in flight, and serve
    // q and k: with a sincosf in each of the unrolled rows the kernel was a long straight line of
    // code, and fetching it cost as much as its work: 32 streams of 12 - 48
    // frames decode in 1845 us where they took 1871 (20.7 us of each of eight launches).
    const bool first = c < LPR / 2;
    const int pair4 = 4 * (first ? c : c - LPR / 2);  // the chunk's first pair
    const float pair_freq = expf(-log_theta * (2.0f * static_cast<float>(threadIdx.x % HALF) / static_cast<float>(D)));
    auto norm_rope = [&](float4 x, const float4 &w4, int j) {
        float ssq = x.x * x.x + x.y * x.y + x.z * x.z + x.w * x.w;
#pragma unroll
        for (int m = 1; m < LPR; m <<= 1) ssq += __shfl_xor(ssq, m, kWave);
        const float inv = 1.0f / sqrtf(ssq / static_cast<float>(D) + eps);
        const float y[4] = {x.x * inv * w4.x, x.y * inv * w4.y, x.z * inv * w4.z, x.w * inv * w4.w};
        const float4 cs4 = *reinterpret_cast<const float4 *>(cosines + j * HALF + pair4);
        const float4 sn4 = *reinterpret_cast<const float4 *>(sines + j * HALF + pair4);
        const float cs[4] = {cs4.x, cs4.y, cs4.z, cs4.w}, sn[4] = {sn4.x, sn4.y, sn4.z, sn4.w};
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float partner = __shfl_xor(y[e], LPR / 2, kWave);
            o[e] = first ? y[e] * cs[e] - partner * sn[e] : y[e] * cs[e] + partner * sn[e];
        }
        return make_float4(o[0], o[1], o[2], o[3]);
    };
    const float4 qn4 = *reinterpret_cast<const float4 *>(qn + 4 * c), kn4 = *reinterpret_cast<const float4 *>(kn + 4 * c);

    int last_i0 = 0;
    for (int i0 = 0; i0 < F; i0 += kWinQ) {
        last_i0 = i0;
        const int nq = F - i0 < kWinQ ? F - i0 : kWinQ;
        const int rows = R + nq;
        // stage K and V rows kappa (position P0 + i0 - R + kappa) and the block's rotated q; a group
        // of LPR lanes owns one row per pass (every lane of a group takes the same branch).  Every
        // load of the block is issued before the first is used, so the passes share one round trip.
        constexpr int KVP = (kWinMax - 1 + kWinQ + RPP - 1) / RPP;  // K/V passes at most
        constexpr int QP = (kWinQ + RPP - 1) / RPP;                 // q passes at most
        float4 kreg[KVP], vreg[KVP], qreg[QP];
#pragma unroll
        for (int pp = 0; pp < KVP; ++pp) {
            const int kappa = pp * RPP + threadIdx.x / LPR;
            const int fi = i0 - R + kappa;
            kreg[pp] = vreg[pp] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (kappa < rows) {
                if (fi < 0) {  // retained slot i0 + kappa, rotated when it was stored
                    kreg[pp] = *reinterpret_cast<const float4 *>(sk + (i0 + kappa) * srow + 4 * c);
                    vreg[pp] = *reinterpret_cast<const float4 *>(sv + (i0 + kappa) * srow + 4 * c);
                } else {
                    kreg[pp] = *reinterpret_cast<const float4 *>(k + (t0 + fi) * ld + h * D + 4 * c);
                    vreg[pp] = *reinterpret_cast<const float4 *>(v + (t0 + fi) * ld + h * D + 4 * c);
                }
            }
        }
#pragma unroll
        for (int pp = 0; pp < QP; ++pp) {
            const int jq = pp * RPP + threadIdx.x / LPR;
            qreg[pp] = jq < nq ? *reinterpret_cast<const float4 *>(q + (t0 + i0 + jq) * ld + h * D + 4 * c)
                               : make_float4(0.f, 0.f, 0.f, 0.f);
        }
#pragma unroll 1
        for (int i = threadIdx.x; i < nq * HALF; i += kWinThreads)  // query row i / HALF, the thread's pair
            sincosf(static_cast<float>(P0 + i0 + i / HALF) * pair_freq, &sines[i], &cosines[i]);
        __syncthreads();
#pragma unroll
        for (int pp = 0; pp < KVP; ++pp) {
            const int kappa = pp * RPP + threadIdx.x / LPR;
            const int fi = i0 - R + kappa;
            if (kappa < rows) {
                float4 kv = kreg[pp];
                if (fi >= i0) {  // this block's own frame: rotate it, and keep it rotated in place
                    kv = norm_rope(kv, kn4, fi - i0);
                    *reinterpret_cast<float4 *>(k + (t0 + fi) * ld + h * D + 4 * c) = kv;
                }
                *reinterpret_cast<float4 *>(ks + kappa * P + 4 * c) = kv;
                *reinterpret_cast<float4 *>(vs + kappa * P + 4 * c) = vreg[pp];
            }
        }
#pragma unroll
        for (int pp = 0; pp < QP; ++pp) {
            const int jq = pp * RPP + threadIdx.x / LPR;
            if (jq < nq)
                *reinterpret_cast<float4 *>(qs + jq * P + 4 * c) =
                    norm_rope(qreg[pp], qn4, jq);
        }
        __syncthreads();

        // kWinGroup queries at a time, one thread per (query, window step): half a wave holds a query's
        // scores, and its lanes then take the query's channels
        for (int j0 = 0; j0 < nq; j0 += kWinGroup) {
            const int j = j0 + threadIdx.x / kWinMax, s = threadIdx.x % kWinMax;
            const int lowest = max(0, R - i0 - j - ctx);  // the first window step that holds a key
            const bool valid = j < nq && s >= lowest && s < W;
            float score = -INFINITY;
            if (valid) {
                const float *qr = qs + j * P, *kr = ks + (j + s) * P;
                score = 0.f;
#pragma unroll 4
                for (int u = 0; u < D; u += 4) {
                    const float4 qq = *reinterpret_cast<const float4 *>(qr + u);
                    const float4 kk = *reinterpret_cast<const float4 *>(kr + u);
                    score += qq.x * kk.x + qq.y * kk.y + qq.z * kk.z + qq.w * kk.w;
                }
                score *= scale;
            }
            float mx = score;
#pragma unroll
            for (int m = kWinMax / 2; m; m >>= 1) mx = fmaxf(mx, __shfl_xor(mx, m, kWave));
            const float pr = valid ? expf(score - mx) : 0.f;
            float l = pr;
#pragma unroll
            for (int m = kWinMax / 2; m; m >>= 1) l += __shfl_xor(l, m, kWave);
            ps[threadIdx.x] = pr;  // read by the same half wave, whose LDS accesses complete in order
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            constexpr int CPL = D > kWinMax ? D / kWinMax : 1;  // channels per lane
            if (j < nq && s * CPL < D) {
                const float *pj = ps + threadIdx.x - s;
                float acc[CPL] = {};
#pragma unroll 4
                for (int i = lowest; i < W; ++i) {
                    const float *vr = vs + (j + i) * P + s * CPL;
#pragma unroll
                    for (int e = 0; e < CPL; ++e) acc[e] += pj[i] * vr[e];
                }
                float *op = out + (t0 + i0 + j) * ldo + h * D + s * CPL;
                const float il = 1.0f / l;
#pragma unroll
                for (int e = 0; e < CPL; ++e) op[e] = acc[e] * il;
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        if (i0 + kWinQ < F) __syncthreads();  // the block's LDS rows are read before the next block restages them
    }
    // retained rows jr = 0 .. R-1 <- positions P0 + F - R + jr: row kappa = jr + F - last_i0 of the last
    // block's staged K/V (a retained slot or a rotated fresh frame); staged before the first block's
    // barrier, so every read of the old state precedes these stores
    for (int e = threadIdx.x; e < R * LPR; e += kWinThreads) {
        const int jr = e / LPR, cc = e % LPR;
        const int kappa = jr + F - last_i0;
        *reinterpret_cast<float4 *>(sk + jr * srow + 4 * cc) = *reinterpret_cast<const float4 *>(ks + kappa * P + 4 * cc);
        *reinterpret_cast<float4 *>(sv + jr * srow + 4 * cc) = *reinterpret_cast<const float4 *>(vs + kappa * P + 4 * cc);
    }
}

__global__ void advance_kernel(const int32_t *__restrict__ off, int B, const int32_t *__restrict__ slots,
                               int64_t *__restrict__ frame_pos, int32_t *__restrict__ ctx_len, int R) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= B) return;
    const int F = off[b + 1] - off[b];
    const int slot = slots[b];
    frame_pos[slot] += F;
    ctx_len[slot] = min(R, ctx_len[slot] + F);
}

__global__ void __launch_bounds__(kCodecThreads)
pcm16_kernel(const float *__restrict__ x, int64_t n, float *__restrict__ wav, int16_t *__restrict__ pcm) {
    for (int64_t i = blockIdx.x * static_cast<int64_t>(kCodecThreads) + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * kCodecThreads) {
        const float c = fminf(fmaxf(x[i], -1.0f), 1.0f);
        if (wav) wav[i] = c;
        if (pcm) pcm[i] = static_cast<int16_t>(rintf(c * 32767.0f));
    }
}

// ---------------------------------------------------------------------------
// A decoder residual unit of C = 16 or 32 channels on MFMA, for the decoder's
// "high" float32 matmul precision (the reference's convolutions run on cuDNN with
// its TF32 default): out = x + conv1x1(snake2(conv7(snake1(x)) + b1)) + b2 as two
// implicit GEMMs with bf16x3 split products and fp32 sums, each operand v = hi +
// lo + e with hi = bf16(v), lo = bf16(v - hi), |e| <= 2^-16 |v|, a product
// hi*hi + hi*lo + lo*hi.  The 7-tap convolution is D[co][t] = sum_k W[co][k]
// X[k][t] with k = tap * C + ci (zero weights past the seventh tap), X[k][t] =
// snake1(x)[t - (6 - tap) dil][ci]: the weights are the A operand of
// v_mfma_f32_16x16x32_bf16 (split once per workgroup into an LDS fragment table,
// one 16-byte read per lane), the activated input rows the B operand (a lane's 8
// consecutive k are 8 consecutive channels of one input row, staged split in LDS
// as [row][C hi | C lo] with a 16-byte row pad, 8 rows of a lane group then
// cover distinct banks), so a lane ends with 4 consecutive output channels of
// one row.  The activated 7-tap outputs go split, one 16-row tile at a time,
// through the wave's own LDS rows into the B operand of the 1x1 convolution.  A
// workgroup of 4 waves owns 4 x 16 x MT output rows of one stream, and the
// (K-1) dil rows before them come from the stream's history where they lie
// before its first fresh row.
//
// What bounds it is the chain of one workgroup (weights, rows, activation, products), so the weights are
// read as each thread's 28 consecutive floats (as scattered fragment elements every lane of a load met
// its own cache line) and a tile stays within a stream: with tiles over the concatenated rows the rows
// near a stream's start searched their stream and read its history tap by tap, and one such wave held
// its workgroup up.  32 channels at dilation 9: 400 rows of one stream 24.8 -> 11.6 us, 89,600 rows of 32
// streams 50.7 -> 25.4; 16 channels: 1600 rows 14.5 -> 8.6, 358,400 rows 38.9 -> 27.0.

typedef __bf16 cu_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 cu_bf16x2 __attribute__((ext_vector_type(2)));
typedef float cu_floatx2 __attribute__((ext_vector_type(2)));
typedef float cu_floatx4 __attribute__((ext_vector_type(4)));
typedef float cu_weights4 __attribute__((ext_vector_type(4), aligned(4)));  // four floats at any float's address

constexpr int kUnitThreads = 256;
constexpr int kUnitTaps = 7;

constexpr int unit_rows(int MT) { return kUnitThreads / kWave * MT * 16; }  // output rows per workgroup

__device__ __forceinline__ uint32_t cu_pack(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((cu_floatx2){a, b}, cu_bf16x2));
}

// hi / lo bf16 words of the pair (a, b); a - bf16(a) is exact in fp32
__device__ __forceinline__ void cu_split2(float a, float b, uint32_t &hi, uint32_t &lo) {
    hi = cu_pack(a, b);
    lo = cu_pack(a - __uint_as_float(hi << 16), b - __uint_as_float(hi & 0xffff0000u));
}

// hi / lo words of four values
__device__ __forceinline__ void cu_split4(float a, float b, float c, float d, uint2 &hi, uint2 &lo) {
    cu_split2(a, b, hi.x, lo.x);
    cu_split2(c, d, hi.y, lo.y);
}

__device__ __forceinline__ cu_bf16x8 cu_frag(const uint4 &v) { return __builtin_bit_cast(cu_bf16x8, v); }

template <int C>
constexpr int unit_ksteps() {
    return (kUnitTaps * C + 31) / 32;
}

template <int C>
size_t unit_mfma_lds(int pad, int MT) {
    constexpr int NT = C / 16;
    constexpr int RB = 4 * C + 16;
    return static_cast<size_t>(unit_ksteps<C>() * NT * 2 * kWave + NT * 2 * kWave) * 16 +
           static_cast<size_t>(unit_rows(MT) + pad) * RB + static_cast<size_t>(kUnitThreads / kWave) * 16 * RB;
}

template <int C, int MT>
__global__ void __launch_bounds__(kUnitThreads)
unit_mfma_kernel(const float *__restrict__ x, int64_t ldx, int64_t T, const int32_t *__restrict__ off, int B, int u,
                 const int32_t *__restrict__ slots, const float *__restrict__ hist, int dil,
                 const float *__restrict__ w1, const float *__restrict__ b1, Act act1,
                 const float *__restrict__ w2, const float *__restrict__ b2, Act act2,
                 float *__restrict__ out, int64_t ldo) {
    static_assert(C == 16 || C == 32, "16 or 32 channels");
    constexpr int NT = C / 16;               // 16-wide output-channel tiles
    constexpr int KS = unit_ksteps<C>();     // 32-k steps of the 7-tap convolution
    constexpr int RB = 4 * C + 16;           // LDS row bytes
    constexpr int VPR = C / 4;               // float4 per input row
    constexpr int ROWS = unit_rows(MT);      // output rows per workgroup
    constexpr int kBatch = MT == 1 ? 4 : 8;  // 128-bit loads in flight per thread
    extern __shared__ __attribute__((aligned(16))) char ulds[];
    __shared__ float sp[4][32];              // snake1 a, 1/b; snake2 a, 1/b
    uint4 *wf1 = reinterpret_cast<uint4 *>(ulds);      // [KS][NT][hi, lo][64 lanes]
    uint4 *wf2 = wf1 + KS * NT * 2 * kWave;            // [NT][hi, lo][64 lanes]
    char *xs = reinterpret_cast<char *>(wf2 + NT * 2 * kWave);
    const int pad = (kUnitTaps - 1) * dil;
    char *ys = xs + (ROWS + pad) * RB;                 // [wave][16 rows][RB]
    const int tid = threadIdx.x;

    // 1. thread t < C^2 / 4 holds the weights of output channel t / (C / 4) and four consecutive input
    // channels: 28 consecutive floats of w1, four of w2; requested before the tile is known
    const bool has_w = tid < C * C / 4;
    cu_weights4 wr[kUnitTaps], wr2 = {};
#pragma unroll
    for (int i = 0; i < kUnitTaps; ++i)
        wr[i] = *reinterpret_cast<const cu_weights4 *>(w1 + (has_w ? tid : 0) * 4 * kUnitTaps + 4 * i);
    wr2 = *reinterpret_cast<const cu_weights4 *>(w2 + (has_w ? tid : 0) * 4);
    StreamTile st;
    if (!stream_tile(off, B, u, T, ROWS, static_cast<int>(blockIdx.x), st)) return;
    x += st.first * ldx;
    out += st.first * ldo;
    const float *h = hist + (static_cast<int64_t>(slots[st.b]) * pad + pad) * C;  // row -1 lies before it

    // 2. the input rows l0 - pad .. l0 + ROWS - 1 of the stream (the last one again past its end: those
    // feed no stored output); the first batch is in flight while the weights are laid out
    const int nvec = (ROWS + pad) * VPR;
    auto load_batch = [&](int e0, float4 (&v)[kBatch]) {
#pragma unroll
        for (int i = 0; i < kBatch; ++i) {
            const int e = e0 + i * kUnitThreads < nvec ? e0 + i * kUnitThreads : nvec - 1;
            const int rr = e / VPR;
            int64_t l = st.l0 - pad + rr;
            if (l >= st.n) l = st.n - 1;
            const float *row = l < 0 ? h + l * C : x + l * ldx;
            v[i] = *reinterpret_cast<const float4 *>(row + (e - rr * VPR) * 4);
        }
    };
    auto store_batch = [&](int e0, const float4 (&v)[kBatch]) {
#pragma unroll
        for (int i = 0; i < kBatch; ++i) {
            const int e = e0 + i * kUnitThreads;
            if (e >= nvec) break;
            const int rr = e / VPR, c4 = (e - rr * VPR) * 4;
            float f[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
            if (act1.alpha && st.l0 - pad + rr >= 0) {
#pragma unroll
                for (int q = 0; q < 4; ++q) f[q] = snake(f[q], sp[0][c4 + q], sp[1][c4 + q]);
            }
            uint2 hi, lo;
            cu_split4(f[0], f[1], f[2], f[3], hi, lo);
            *reinterpret_cast<uint2 *>(xs + rr * RB + 2 * c4) = hi;
            *reinterpret_cast<uint2 *>(xs + rr * RB + 2 * C + 2 * c4) = lo;
        }
    };
    float4 vb[kBatch];
    load_batch(tid, vb);

    // 3. the weights as split MFMA A fragments: lane (r16, kq) of step j holds W[co = 16 nt + r16][k = 32 j + 8 kq .. + 7]
    if (has_w) {
        const int co = tid / (C / 4), ci = tid % (C / 4) * 4;
        // the half fragment of the four channels at k: hi words, and lo words one fragment on
        auto put = [&](uint4 *frag, int lane, int ci_in, const uint2 &hi, const uint2 &lo) {
            uint2 *at = reinterpret_cast<uint2 *>(frag + lane) + (ci_in >> 2);
            at[0] = hi;
            at[2 * kWave] = lo;
        };
#pragma unroll
        for (int tap = 0; tap < KS * 32 / C; ++tap) {
            uint2 hi = make_uint2(0, 0), lo = make_uint2(0, 0);
            if (tap < kUnitTaps) {
                float f[4];
#pragma unroll
                for (int p = 0; p < 4; ++p) f[p] = wr[(p * kUnitTaps + tap) / 4][(p * kUnitTaps + tap) % 4];
                cu_split4(f[0], f[1], f[2], f[3], hi, lo);
            }
            const int k = (tap * C) % 32 + ci;
            put(wf1 + ((tap * C / 32 * NT + co / 16) * 2) * kWave, (k >> 3) * 16 + (co & 15), k & 7, hi, lo);
        }
        uint2 hi, lo;
        cu_split4(wr2[0], wr2[1], wr2[2], wr2[3], hi, lo);
        put(wf2 + (co / 16 * 2) * kWave, (ci >> 3) * 16 + (co & 15), ci & 7, hi, lo);
        if constexpr (C == 16)  // k 16 .. 31 of the 1x1 convolution
            put(wf2 + (co / 16 * 2) * kWave, ((ci + 16) >> 3) * 16 + (co & 15), ci & 7, make_uint2(0, 0),
                make_uint2(0, 0));
    }
    if (tid < C) {
        sp[0][tid] = act1.alpha ? act1.a_of(tid) : 0.f;
        sp[1][tid] = act1.alpha ? act1.inv_b_of(tid) : 0.f;
        sp[2][tid] = act2.alpha ? act2.a_of(tid) : 0.f;
        sp[3][tid] = act2.alpha ? act2.inv_b_of(tid) : 0.f;
    }

    __syncthreads();  // the snake parameters
    store_batch(tid, vb);
    for (int e0 = tid + kBatch * kUnitThreads; e0 < nvec; e0 += kBatch * kUnitThreads) {
        load_batch(e0, vb);
        store_batch(e0, vb);
    }
    __syncthreads();

    // 4. the 7-tap convolution: wave w owns rows l0 + (MT w + m) 16 + r16, m < MT
    const int lane = tid & (kWave - 1), wave = tid / kWave;
    const int r16 = lane & 15, kq = lane >> 4;
    // the residual rows of the epilogue, loaded now so that their round trip overlaps the MFMAs
    float4 xres[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int64_t l = st.l0 + (wave * MT + m) * 16 + r16;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
            xres[m][nt] = *reinterpret_cast<const float4 *>(x + (l < st.n ? l : st.n - 1) * ldx + nt * 16 + 4 * kq);
    }
    cu_floatx4 acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[m][nt] = cu_floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < KS; ++j) {
        cu_bf16x8 ah[NT], al[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            ah[nt] = cu_frag(wf1[((j * NT + nt) * 2) * kWave + lane]);
            al[nt] = cu_frag(wf1[((j * NT + nt) * 2 + 1) * kWave + lane]);
        }
        const int k0 = 32 * j + 8 * kq, tap = k0 / C, cb = k0 - (k0 / C) * C;
        const int back = tap < kUnitTaps ? (kUnitTaps - 1 - tap) * dil : 0;  // past the 7th tap: zero weights
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const char *rp = xs + ((wave * MT + m) * 16 + r16 + pad - back) * RB + 2 * cb;
            const uint4 bh = *reinterpret_cast<const uint4 *>(rp);
            const uint4 bl = *reinterpret_cast<const uint4 *>(rp + 2 * C);
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                acc[m][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[nt], cu_frag(bh), acc[m][nt], 0, 0, 0);
                acc[m][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[nt], cu_frag(bl), acc[m][nt], 0, 0, 0);
                acc[m][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[nt], cu_frag(bh), acc[m][nt], 0, 0, 0);
            }
        }
    }

    // 5. per tile: y = snake2(conv + b1), split into the wave's own 16 LDS rows (lane (r16, kq) holds
    // y[row r16][co = 16 nt + 4 kq .. + 3]), read back as the B operand of the 1x1 convolution (lane
    // (r16, kq) = y[row r16][ci = 8 kq .. + 7]), then the residual
    char *yw = ys + wave * 16 * RB;
    cu_bf16x8 a2h[NT], a2l[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        a2h[nt] = cu_frag(wf2[(nt * 2) * kWave + lane]);
        a2l[nt] = cu_frag(wf2[(nt * 2 + 1) * kWave + lane]);
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const int co = nt * 16 + 4 * kq;
            float y[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                y[e] = acc[m][nt][e] + (b1 ? b1[co + e] : 0.f);
                if (act2.alpha) y[e] = snake(y[e], sp[2][co + e], sp[3][co + e]);
            }
            uint2 hi, lo;
            cu_split4(y[0], y[1], y[2], y[3], hi, lo);
            char *rp = yw + r16 * RB + 2 * co;
            *reinterpret_cast<uint2 *>(rp) = hi;
            *reinterpret_cast<uint2 *>(rp + 2 * C) = lo;
        }
        __builtin_amdgcn_wave_barrier();  // the wave reads back what its own lanes wrote (LDS keeps its order)
        uint4 bh = make_uint4(0, 0, 0, 0), bl = make_uint4(0, 0, 0, 0);
        if (8 * kq < C) {
            const char *rp = yw + r16 * RB + 16 * kq;
            bh = *reinterpret_cast<const uint4 *>(rp);
            bl = *reinterpret_cast<const uint4 *>(rp + 2 * C);
        }
        __builtin_amdgcn_wave_barrier();  // every lane has read the tile before the next one is written
        const int64_t l = st.l0 + (wave * MT + m) * 16 + r16;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            cu_floatx4 d = cu_floatx4{0.f, 0.f, 0.f, 0.f};
            d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2l[nt], cu_frag(bh), d, 0, 0, 0);
            d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2h[nt], cu_frag(bl), d, 0, 0, 0);
            d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2h[nt], cu_frag(bh), d, 0, 0, 0);
            if (l >= st.n) continue;
            const int co = nt * 16 + 4 * kq;
            const float4 xr = xres[m][nt];
            float4 o;
            o.x = xr.x + d[0] + (b2 ? b2[co] : 0.f);
            o.y = xr.y + d[1] + (b2 ? b2[co + 1] : 0.f);
            o.z = xr.z + d[2] + (b2 ? b2[co + 2] : 0.f);
            o.w = xr.w + d[3] + (b2 ? b2[co + 3] : 0.f);
            *reinterpret_cast<float4 *>(out + l * ldo + co) = o;
        }
    }
}

// 16-row tiles per wave.  One while the 64-row workgroups fit on the chip at once (32 channels: 58 KB of
// LDS, two per CU; 16 channels: 25 KB, where four per CU is the measured line): the shortest chain.  Past
// that the rows before a tile, staged again by the next, and the weights weigh more: 32 channels at
// dilation 9, 89,600 rows: 28.1 / 25.4 / 35.4 us with 1 / 2 / 4 tiles (9600 rows: 12.1 / 14.7 / 20.2);
// 16 channels, 358,400 rows: 30.5 / 27.7 / 27.0 (38,400 rows: 10.4 / 11.4 / 12.7).
int unit_tiles(int C, int64_t T, int B) {
    const int64_t small = stream_tiles_bound(T, B, unit_rows(1));
    if (C == 16) return small <= 4 * kCus ? 1 : 4;
    return small <= 2 * kCus ? 1 : 2;
}

int grid_for(int64_t n) {
    const int64_t g = (n + kCodecThreads - 1) / kCodecThreads;
    return static_cast<int>(g < 1 ? 1 : g > 8192 ? 8192 : g);
}

}  // namespace
}  // namespace nq

using namespace nq;

extern "C" int nq_codec_embed_sum(const int32_t *codes, int T, int Q, const float *books, int V, int C, float *out,
                                  int32_t *status, void *stream) {
    NQ_CHECK_ARG(codes && books && out && T >= 0 && Q > 0 && V > 0 && C > 0);
    if (T == 0) return NQ_OK;
    hipLaunchKernelGGL(embed_sum_kernel, dim3(grid_for(static_cast<int64_t>(T) * C)), dim3(kCodecThreads), 0,
                       static_cast<hipStream_t>(stream), codes, T, Q, books, V, C, out, status);
    return NQ_LAUNCH_STATUS();
}

extern "C" int nq_codec_causal_conv(const float *x, int64_t ldx, int64_t T, const int32_t *offsets, int B, int u,
                                    const int32_t *slots, float *history, const float *w, const float *bias, int Cin,
                                    int Cout, int K, int dilation, int groups, const float *act_alpha,
                                    const float *act_beta, const float *residual, int64_t ldres, float *out,
                                    int64_t ldo, void *stream) {
    NQ_CHECK_ARG(x && offsets && slots && w && out && B > 0 && u > 0 && T >= 0);
    NQ_CHECK_ARG(Cin > 0 && Cout > 0 && K >= 1 && K <= kConvKMax && dilation >= 1);
    NQ_CHECK_ARG(groups == 1 || (groups == Cin && Cin == Cout && !residual && !act_alpha));
    NQ_CHECK_ARG((act_alpha == nullptr) == (act_beta == nullptr));
    NQ_CHECK_ARG(ldx >= Cin && ldo >= Cout && (!residual || ldres >= Cout));
    const int pad = (K - 1) * dilation;
    NQ_CHECK_ARG(pad == 0 || history);
    if (pad * Cin > kHistoryThreads * kHistoryPerThread) return NQ_ERR_UNSUPPORTED;
    if (T == 0) return NQ_OK;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const Act act{act_alpha, act_beta};
    const int co_pad = Cout == 1 ? 1 : Cout <= 8 ? 8 : Cout <= 16 ? 16 : Cout <= 32 ? 32 : 64;
    const int R = conv_small_rows(co_pad, T, B);
    const int most = co_pad <= 16 ? 2 : 1;  // rows per thread the rule may choose
    if (groups == 1 && Cin <= 64 && Cout <= 64 && conv_small_lds(Cin, K, dilation, co_pad, most) <= kConvLds) {
        const size_t lds = conv_small_lds(Cin, K, dilation, co_pad, R);
        const dim3 grid(static_cast<unsigned>(stream_tiles_bound(T, B, kCodecThreads * R)));
#define NQ_SMALL(CO, R)                                                                                              \
        hipLaunchKernelGGL((conv_small_kernel<CO, R>), grid, dim3(kCodecThreads), lds, st, x, ldx, T, offsets, B, u, \
                           slots, history, w, bias, Cin, Cout, K, dilation, act, residual, ldres, out, ldo)
        if (co_pad == 1 && R == 1) NQ_SMALL(1, 1);
        else if (co_pad == 1) NQ_SMALL(1, 2);
        else if (co_pad == 8 && R == 1) NQ_SMALL(8, 1);
        else if (co_pad == 8) NQ_SMALL(8, 2);
        else if (co_pad == 16 && R == 1) NQ_SMALL(16, 1);
        else if (co_pad == 16) NQ_SMALL(16, 2);
        else if (co_pad == 32) NQ_SMALL(32, 1);
        else NQ_SMALL(64, 1);
#undef NQ_SMALL
    } else if (groups == 1) {
        const int cg = Cout <= 16 ? 1 : Cout <= 32 ? 2 : 4;
        const int rows = kCodecThreads / cg;
        dim3 grid(static_cast<unsigned>((T + rows - 1) / rows), static_cast<unsigned>((Cout + cg * 16 - 1) / (cg * 16)));
        if (cg == 1)
            hipLaunchKernelGGL(conv_kernel<1>, grid, dim3(kCodecThreads), 0, st, x, ldx, T, offsets, B, u, slots,
                               history, w, bias, Cin, Cout, K, dilation, act, residual, ldres, out, ldo);
        else if (cg == 2)
            hipLaunchKernelGGL(conv_kernel<2>, grid, dim3(kCodecThreads), 0, st, x, ldx, T, offsets, B, u, slots,
                               history, w, bias, Cin, Cout, K, dilation, act, residual, ldres, out, ldo);
        else
            hipLaunchKernelGGL(conv_kernel<4>, grid, dim3(kCodecThreads), 0, st, x, ldx, T, offsets, B, u, slots,
                               history, w, bias, Cin, Cout, K, dilation, act, residual, ldres, out, ldo);
    } else {
        hipLaunchKernelGGL(dwconv_kernel, dim3(grid_for(T * Cin)), dim3(kCodecThreads), 0, st, x, ldx, T, offsets, B,
                           u, slots, history, w, bias, Cin, K, dilation, out, ldo);
    }
    if (hipGetLastError() != hipSuccess) return NQ_ERR_LAUNCH;
    if (pad > 0) {
        hipLaunchKernelGGL(history_update_kernel, dim3(B), dim3(kHistoryThreads),
                           0, st, x, ldx, offsets, B, u, slots, history, Cin, pad, groups == 1 ? act : Act{nullptr, nullptr});
    }
    return NQ_LAUNCH_STATUS();
}

extern "C" int nq_codec_residual_unit(const float *x, int64_t ldx, int64_t T, const int32_t *offsets, int B, int u,
                                      const int32_t *slots, float *history, int C, int K, int dilation, const float *w1,
                                      const float *b1, const float *a1_alpha, const float *a1_beta, const float *w2,
                                      const float *b2, const float *a2_alpha, const float *a2_beta, float *out,
                                      int64_t ldo, int precision, void *stream) {
    NQ_CHECK_ARG(x && offsets && slots && history && w1 && w2 && out && B > 0 && u > 0 && T >= 0);
    NQ_CHECK_ARG(C > 0 && K >= 2 && K <= kConvKMax && dilation >= 1 && ldx >= C && ldo >= C && out != x);
    NQ_CHECK_ARG(precision == NQ_MATMUL_HIGHEST || precision == NQ_MATMUL_HIGH);
    if (K != kConvKMax) return NQ_ERR_UNSUPPORTED;  // the fused kernels are built for 7 taps
    if ((K - 1) * dilation * C > kHistoryThreads * kHistoryPerThread) return NQ_ERR_UNSUPPORTED;
    NQ_CHECK_ARG((a1_alpha == nullptr) == (a1_beta == nullptr) && (a2_alpha == nullptr) == (a2_beta == nullptr));
    const int co_pad = C <= 8 ? 8 : C <= 16 ? 16 : 32;
    if (C > 32 || C != co_pad) return NQ_ERR_UNSUPPORTED;
    // the split-product MFMA kernel for 16 and 32 channels; 8 channels keep the fp32 direct kernel at
    // either precision (at 1.98 M rows: 58 us against 84 us for the MFMA kernel, whose workgroups are
    // latency-bound at that width)
    const bool split = precision == NQ_MATMUL_HIGH && C >= 16;
    const int pad = (K - 1) * dilation;
    if (split && (ldx % 4 || ldo % 4 || ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out) |
                                          reinterpret_cast<uintptr_t>(history)) & 15)))
        return NQ_ERR_UNSUPPORTED;
    const int R = conv_small_rows(co_pad, T, B), MT = unit_tiles(C, T, B);
    const size_t lds = split ? (C == 16 ? unit_mfma_lds<16>(pad, MT) : unit_mfma_lds<32>(pad, MT))
                             : conv_small_lds(C, K, dilation, co_pad, R, true);
    if (lds > kConvLds) return NQ_ERR_UNSUPPORTED;
    if (T == 0) return NQ_OK;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const Act act1{a1_alpha, a1_beta}, act2{a2_alpha, a2_beta};
    if (split) {
        const dim3 grid(static_cast<unsigned>(stream_tiles_bound(T, B, unit_rows(MT))));
#define NQ_UNIT(CC, MT)                                                                                         \
        hipLaunchKernelGGL((unit_mfma_kernel<CC, MT>), grid, dim3(kUnitThreads), lds, st, x, ldx, T, offsets, B, u, \
                           slots, history, dilation, w1, b1, act1, w2, b2, act2, out, ldo)
        if (C == 16 && MT == 1) NQ_UNIT(16, 1);
        else if (C == 16) NQ_UNIT(16, 4);
        else if (MT == 1) NQ_UNIT(32, 1);
        else NQ_UNIT(32, 2);
#undef NQ_UNIT
    } else {
        const dim3 grid(static_cast<unsigned>(stream_tiles_bound(T, B, kCodecThreads * R)));
#define NQ_UNIT(CO, R)                                                                                               \
        hipLaunchKernelGGL((conv_small_kernel<CO, R, true>), grid, dim3(kCodecThreads), lds, st, x, ldx, T, offsets, \
                           B, u, slots, history, w1, b1, C, C, K, dilation, act1, x, ldx, out, ldo, w2, b2, act2)
        if (co_pad == 8 && R == 1) NQ_UNIT(8, 1);
        else if (co_pad == 8) NQ_UNIT(8, 2);
        else if (co_pad == 16 && R == 1) NQ_UNIT(16, 1);
        else if (co_pad == 16) NQ_UNIT(16, 2);
        else NQ_UNIT(32, 1);
#undef NQ_UNIT
    }
    if (hipGetLastError() != hipSuccess) return NQ_ERR_LAUNCH;
    hipLaunchKernelGGL(history_update_kernel, dim3(B), dim3(kHistoryThreads), 0, st,
                       x, ldx, offsets, B, u, slots, history, C, (K - 1) * dilation, act1);
    return NQ_LAUNCH_STATUS();
}

extern "C" int nq_codec_causal_transconv(const float *x, int64_t ldx, int64_t T_in, const int32_t *offsets, int B,
                                         int u_in, int stride_s, const int32_t *slots, float *overlap, const float *w,
                                         const float *bias, int Cin, int Cout, const float *act_alpha,
                                         const float *act_beta, float *out, int64_t ldo, void *stream) {
    NQ_CHECK_ARG(x && offsets && slots && overlap && w && out && B > 0 && u_in > 0 && stride_s >= 1 && T_in >= 0);
    NQ_CHECK_ARG(Cin > 0 && Cout > 0 && ldx >= Cin && ldo >= Cout);
    NQ_CHECK_ARG((act_alpha == nullptr) == (act_beta == nullptr));
    if (T_in == 0) return NQ_OK;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const Act act{act_alpha, act_beta};
    const int cg = Cout <= 16 ? 1 : Cout <= 32 ? 2 : 4;
    const int rows = kCodecThreads / cg;
    const int64_t T_out = T_in * stride_s;
    const int co_pad = Cout <= 8 ? 8 : 16;
    const dim3 update(static_cast<unsigned>(B), static_cast<unsigned>((stride_s * Cout + kCodecThreads - 1) / kCodecThreads));
    if (Cout <= 16 && transconv_small_lds(Cin, stride_s, co_pad) <= 64 * 1024) {
        const size_t lds = transconv_small_lds(Cin, stride_s, co_pad);
        const dim3 grid(static_cast<unsigned>((T_out + kCodecThreads - 1) / kCodecThreads));
        if (co_pad == 8)
            hipLaunchKernelGGL(transconv_small_kernel<8>, grid, dim3(kCodecThreads), lds, st, x, ldx, T_out, offsets, B,
                               u_in, stride_s, slots, overlap, w, bias, Cin, Cout, act, out, ldo);
        else
            hipLaunchKernelGGL(transconv_small_kernel<16>, grid, dim3(kCodecThreads), lds, st, x, ldx, T_out, offsets,
                               B, u_in, stride_s, slots, overlap, w, bias, Cin, Cout, act, out, ldo);
        if (hipGetLastError() != hipSuccess) return NQ_ERR_LAUNCH;
        hipLaunchKernelGGL(overlap_update_kernel, update, dim3(kCodecThreads), 0, st, x, ldx, offsets, u_in, stride_s,
                           slots, overlap, w, Cin, Cout, act);
        return NQ_LAUNCH_STATUS();
    }
    const size_t lds = static_cast<size_t>(kConvCi) * cg * 16 * 2 * stride_s * sizeof(float);
    if (lds > 64 * 1024) return NQ_ERR_UNSUPPORTED;
    dim3 grid(static_cast<unsigned>((T_out + rows - 1) / rows), static_cast<unsigned>((Cout + cg * 16 - 1) / (cg * 16)));
    if (cg == 1)
        hipLaunchKernelGGL(transconv_kernel<1>, grid, dim3(kCodecThreads), lds, st, x, ldx, T_out, offsets, B, u_in,
                           stride_s, slots, overlap, w, bias, Cin, Cout, act, out, ldo);
    else if (cg == 2)
        hipLaunchKernelGGL(transconv_kernel<2>, grid, dim3(kCodecThreads), lds, st, x, ldx, T_out, offsets, B, u_in,
                           stride_s, slots, overlap, w, bias, Cin, Cout, act, out, ldo);
    else
        hipLaunchKernelGGL(transconv_kernel<4>, grid, dim3(kCodecThreads), lds, st, x, ldx, T_out, offsets, B, u_in,
                           stride_s, slots, overlap, w, bias, Cin, Cout, act, out, ldo);
    if (hipGetLastError() != hipSuccess) return NQ_ERR_LAUNCH;
    hipLaunchKernelGGL(overlap_update_kernel, update, dim3(kCodecThreads), 0, st, x, ldx, offsets, u_in, stride_s, slots,
                       overlap, w, Cin, Cout, act);
    return NQ_LAUNCH_STATUS();
}

extern "C" int nq_codec_window_attention(float *q, float *k, const float *v, int64_t ld, int T, int H, int D,
                                         const float *q_norm, const float *k_norm, float eps, float rope_theta,
                                         const int32_t *offsets, int B, const int32_t *slots, const int64_t *frame_pos,
                                         const int32_t *ctx_len, float *state_k, float *state_v,
                                         int64_t state_slot_stride, int R, int window, float *out, int64_t ldo,
                                         void *stream) {
    NQ_CHECK_ARG(q && k && v && q_norm && k_norm && offsets && slots && frame_pos && ctx_len && out);
    NQ_CHECK_ARG(state_k && state_v && T >= 0 && B > 0 && H > 0 && R >= 0 && window == R + 1);
    NQ_CHECK_ARG(state_slot_stride >= static_cast<int64_t>(R) * H * D);
    NQ_CHECK_ARG(ld >= static_cast<int64_t>(H) * D && ldo >= static_cast<int64_t>(H) * D && rope_theta > 0.f);
    if (D != 16 && D != 32 && D != 64) return NQ_ERR_UNSUPPORTED;
    if (window > nq::kWinMax) return NQ_ERR_UNSUPPORTED;
    if (ld % 4 || ldo % 4 || state_slot_stride % 4 ||
        ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(v) |
          reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(state_k) |
          reinterpret_cast<uintptr_t>(state_v) | reinterpret_cast<uintptr_t>(q_norm) |
          reinterpret_cast<uintptr_t>(k_norm)) & 15))
        return NQ_ERR_UNSUPPORTED;
    if (T == 0) return NQ_OK;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const float lt = logf(rope_theta), scale = 1.0f / sqrtf(static_cast<float>(D));
#define NQ_WIN(DD)                                                                                                \
    hipLaunchKernelGGL(nq::window_block_kernel<DD>, dim3(static_cast<unsigned>(B) * H), dim3(nq::kWinThreads), 0, \
                       st, q, k, v, ld, H, q_norm, k_norm, eps, lt, offsets, slots, frame_pos, ctx_len, state_k,    \
                       state_v, state_slot_stride, R, scale, out, ldo)
    if (D == 64) NQ_WIN(64);
    else if (D == 32) NQ_WIN(32);
    else NQ_WIN(16);
#undef NQ_WIN
    return NQ_LAUNCH_STATUS();
}

extern "C" int nq_codec_advance(const int32_t *offsets, int B, const int32_t *slots, int64_t *frame_pos,
                                int32_t *ctx_len, int R, void *stream) {
    NQ_CHECK_ARG(offsets && slots && frame_pos && ctx_len && B > 0 && R >= 0);
    hipLaunchKernelGGL(advance_kernel, dim3((B + 63) / 64), dim3(64), 0, static_cast<hipStream_t>(stream), offsets, B,
                       slots, frame_pos, ctx_len, R);
    return NQ_LAUNCH_STATUS();
}

extern "C" int nq_codec_state_copy(int rows, int kinds, const int64_t *pool, const int32_t *shapes,
                                   const int64_t *state, int to_pool, const int64_t *position,
                                   int64_t position_stride, int64_t *frame_pos, const int64_t *context,
                                   int32_t *ctx_len, void *stream) {
    using namespace nq;
    NQ_CHECK_ARG(rows >= 1 && kinds >= 1 && pool && shapes && state);
    NQ_CHECK_ARG((!position || (frame_pos && to_pool)) && (!context || (ctx_len && to_pool)));
    for (int k = 0; k < kinds; ++k) {
        const int64_t a = shapes[3 * k], b = shapes[3 * k + 1], inner = shapes[3 * k + 2];
        NQ_CHECK_ARG(pool[k] && a >= 1 && b >= 1 && inner >= 1 && a * b * inner <= (1 << 24));
        const int64_t mask = inner % 4 == 0 ? 15 : 3;
        NQ_CHECK_ARG((pool[k] & mask) == 0);
        for (int r = 0; r < rows; ++r) {
            const int64_t at = state[static_cast<int64_t>(r) * kinds + k];
            NQ_CHECK_ARG((at & mask) == 0 && (at || to_pool));
        }
    }
    for (int r0 = 0; r0 < rows; r0 += kStateRows) {
        const int nr = rows - r0 < kStateRows ? rows - r0 : kStateRows;
        for (int k0 = 0; k0 < kinds; k0 += kStateKinds) {
            const int nk = kinds - k0 < kStateKinds ? kinds - k0 : kStateKinds;
            StateArgs args = {};
            for (int k = 0; k < nk; ++k) {
                const int32_t *sh = shapes + 3 * (k0 + k);
                const int stride = sh[0] * sh[1] * sh[2];
                args.kind[k] = {reinterpret_cast<float *>(pool[k0 + k]) + static_cast<int64_t>(r0) * stride, stride,
                                sh[0], sh[1], sh[2]};
                for (int r = 0; r < nr; ++r)
                    args.state[r][k] = reinterpret_cast<float *>(state[static_cast<int64_t>(r0 + r) * kinds + k0 + k]);
            }
            if (position && k0 == 0) {
                args.position = position + r0 * position_stride;
                args.position_stride = position_stride;
                args.frame_pos = frame_pos + r0;
            }
            if (context && k0 == 0) {
                args.context = context + r0;
                args.ctx_len = ctx_len + r0;
            }
            const dim3 grid(nk, nr), block(kStateThreads);
            if (to_pool)
                hipLaunchKernelGGL(state_copy_kernel<true>, grid, block, 0, static_cast<hipStream_t>(stream), args);
            else
                hipLaunchKernelGGL(state_copy_kernel<false>, grid, block, 0, static_cast<hipStream_t>(stream), args);
        }
    }
    return NQ_LAUNCH_STATUS();
}

extern "C" int nq_codec_pcm16(const float *x, int64_t n, float *wav, int16_t *pcm, void *stream) {
    NQ_CHECK_ARG(x && n >= 0 && (wav || pcm));
    if (n == 0) return NQ_OK;
    hipLaunchKernelGGL(pcm16_kernel, dim3(grid_for(n)), dim3(kCodecThreads), 0, static_cast<hipStream_t>(stream), x, n,
                       wav, pcm);
    return NQ_LAUNCH_STATUS();
}

extern "C" int nq_codec_im2col(const float *x, int64_t ldx, int64_t T, const int32_t *offsets, int B, int u,
                               const int32_t *slots, const float *history, int Cin, int K, int dilation, int transconv,
                               const float *act_alpha, const float *act_beta, float *a, int64_t lda, void *stream) {
    NQ_CHECK_ARG(x && offsets && slots && a && B > 0 && u > 0 && T >= 0 && Cin > 0 && Cin % 4 == 0);
    NQ_CHECK_ARG(ldx % 4 == 0 && lda % 4 == 0 && ldx >= Cin);
    NQ_CHECK_ARG((act_alpha == nullptr) == (act_beta == nullptr));
    if (transconv) {
        NQ_CHECK_ARG(K == 2);
    } else {
        NQ_CHECK_ARG(K >= 1 && dilation >= 1 && (K == 1 || history));
    }
    NQ_CHECK_ARG(lda >= static_cast<int64_t>(K) * Cin);
    if (T == 0) return NQ_OK;
    hipLaunchKernelGGL(im2col_kernel, dim3(grid_for(T * K * (Cin / 4))), dim3(kCodecThreads), 0,
                       static_cast<hipStream_t>(stream), x, ldx, T, offsets, B, u, slots, history, Cin, K, dilation,
                       transconv, Act{act_alpha, act_beta}, a, lda);
    return NQ_LAUNCH_STATUS();
}

extern "C" int nq_codec_history_update(const float *x, int64_t ldx, const int32_t *offsets, int B, int u,
                                       const int32_t *slots, float *history, int C, int pad, const float *act_alpha,
                                       const float *act_beta, void *stream) {
    NQ_CHECK_ARG(x && offsets && slots && history && B > 0 && u > 0 && C > 0 && pad > 0 && ldx >= C);
    NQ_CHECK_ARG((act_alpha == nullptr) == (act_beta == nullptr));
    if (pad * C > nq::kHistoryThreads * nq::kHistoryPerThread) return NQ_ERR_UNSUPPORTED;
    hipLaunchKernelGGL(history_update_kernel, dim3(B), dim3(kHistoryThreads), 0,
                       static_cast<hipStream_t>(stream), x, ldx, offsets, B, u, slots, history, C, pad,
                       Act{act_alpha, act_beta});
    return NQ_LAUNCH_STATUS();
}

extern "C" int nq_codec_transconv_overlap(const int32_t *offsets, int B, int u_in, int stride_s,
                                          const int32_t *slots, float *overlap, const float *new_overlap, int Cout,
                                          float *out, int64_t ldo, void *stream) {
    NQ_CHECK_ARG(offsets && slots && overlap && new_overlap && out && B > 0 && u_in > 0 && stride_s >= 1);
    NQ_CHECK_ARG(Cout > 0 && ldo >= Cout);
    hipLaunchKernelGGL(overlap_fixup_kernel, dim3(grid_for(static_cast<int64_t>(B) * stride_s * Cout)),
                       dim3(kCodecThreads), 0, static_cast<hipStream_t>(stream), offsets, B, u_in, stride_s, slots,
                       overlap, new_overlap, Cout, out, ldo);
    return NQ_LAUNCH_STATUS();
}
