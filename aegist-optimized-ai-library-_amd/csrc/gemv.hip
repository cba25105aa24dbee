// Projections of one or two rows of X (batch-1 decode; the engine's gemv_i8 and
// gemv_bf16, aegist.cu:84-124): Y_s[m, n] (+)= scale_s[n] sum_k X[m, k] W_s[n, k], up to four weights
// sharing X in one launch.
//
// HBM-bound on W and, at these sizes (a 17 MB weight is 3.5 us of HBM), on the launch's one round trip.
// A load instruction is 1 KB of one row (16 bytes per lane), so the stream is contiguous; the products
// run on the VALU in fp32 (x and w exactly, no hi / lo parts), which at one or two rows costs less than
// the MFMA forms' conversion, LDS and barrier steps; the R rows of a wave are summed over the lanes by
// halving exchanges. R, the waves a row is split over and the pieces in flight: see gemv_launch.
// Measured against the MFMA row-tile kernel this replaces (us per launch in a graph, weights from HBM, one row): bf16
// W, fp32 X 32768 x 2048 36.3 -> 22.0 (6.1 TB/s; 20.9 to 21.8 traced), 256 x 2048 6.3 -> 3.4; int8 W, fp32 X
// 2048 x 4096 8.4 -> 4.9, 4096 x 2048 5.6 -> 4.8, 512 x 2048 5.6 -> 3.3, 8192 x 2048 7.1 -> 6.6; bf16 both 9216 x 2048
// 11.3 -> 9.2, 2048 x 4096 7.5 -> 6.0. (A/B figures further down are of other cards: up to 10% off these.)
#include "common.h"

#include <type_traits>

using namespace aegist;

namespace {

typedef uint32_t u4v __attribute__((ext_vector_type(4)));

constexpr int GV_SEG = 4;
struct GemvSeg {
    const void* W;
    const uint16_t* scale;  // per-row scale or null
    float* Y;
    long long ldy;
    int N, b0;              // rows; first workgroup of the launch
};
struct GemvArgs {
    const void* X;
    GemvSeg seg[GV_SEG];
    long long ldx;
    int nseg, M, K, accumulate;
    const uint16_t* nw;  // weight of X's ZNorm (the forms with NV > 0)
    float eps;
};
constexpr int GN_WAVES = 8;  // waves of a workgroup that norms its X

// the 16 bytes of weights a lane holds of a row's 1 KB piece, as floats
template <typename TW> struct GvW;
template <> struct GvW<int8_t> {
    static constexpr int kVals = 16;
    static __device__ __forceinline__ void unpack(u4v q, float (&f)[16]) {
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int b = 0; b < 4; b++) f[4 * i + b] = (float)(int8_t)(q[i] >> (8 * b));
    }
};
template <> struct GvW<uint16_t> {
    static constexpr int kVals = 8;
    static __device__ __forceinline__ void unpack(u4v q, float (&f)[8]) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            f[2 * i] = bf_lo(q[i]);
            f[2 * i + 1] = bf_hi(q[i]);
        }
    }
};

// V consecutive activations
template <int V>
__device__ __forceinline__ void gv_x(const float* p, float (&f)[V]) {
#pragma unroll
    for (int i = 0; i < V / 4; i++) {
        const float4 a = ((const float4*)p)[i];
        f[4 * i] = a.x; f[4 * i + 1] = a.y; f[4 * i + 2] = a.z; f[4 * i + 3] = a.w;
    }
}
template <int V>
__device__ __forceinline__ void gv_x(const uint16_t* p, float (&f)[V]) {
#pragma unroll
    for (int i = 0; i < V / 8; i++) {
        const uint4 a = ((const uint4*)p)[i];
        const uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
        for (int j = 0; j < 4; j++) {
            f[8 * i + 2 * j] = bf_lo(w[j]);
            f[8 * i + 2 * j + 1] = bf_hi(w[j]);
        }
    }
}

// One wave: R consecutive rows of W against MX rows of X. Lane l holds bytes 16 l .. of each row's 1 KB
// pieces, so a load instruction is 1 KB of one row. KS > 1: the rows are KS waves', each with every
// KS-th piece; the sums meet in LDS. Against whole rows per wave (R = 1, more pieces in flight) X is
// read once per R rows instead of once per row, which at one row of X is half of all loads (us, weights
// from HBM): bf16 2048 x 4096 6.8 -> 5.8, 9216 x 2048 9.9 -> 8.8, 32768 x 2048 24.3 -> 23.5,
// 256 x 2048 3.3 -> 3.0; int8 2048 x 4096 6.3 -> 4.9, two rows 7.4 -> 5.4,
// 16384 x 4096 21.0 -> 18.7.
//
// NV > 0: X is the fp32 residual, and the product takes bf16(ZNorm(X)) (K <= 2048 NV). Every workgroup
// norms the rows for itself, into LDS: x and the norm weight are requested ahead of the wave's first
// weights, so the norm runs while those are on their way from HBM. That costs 12 KB of L2 reads per 8
// rows and takes out a launch that only moved 12 KB (4.0 to 4.4 us of a decode layer's chain; a 4-layer
// stack's 16-token generation 2827 -> 2696 us, 2430 to 2470 with KS).
template <typename TW, typename TX, int R, int MX, int PD, int NV = 0, int KS = 1>
__global__ void __launch_bounds__(NV ? WAVE * GN_WAVES : 256) gemv_kernel(const GemvArgs ga) {
    constexpr int V = GvW<TW>::kVals, PIECE = V * WAVE, WAVES = NV ? GN_WAVES : 4;
    static_assert(WAVES % KS == 0, "a row's KS waves are of one workgroup");
    int si = 0;
#pragma unroll
    for (int i = 1; i < GV_SEG; i++)
        if (i < ga.nseg && (int)blockIdx.x >= ga.seg[i].b0) si = i;
    const GemvSeg sg = ga.seg[si];
    const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int n0 = (((int)blockIdx.x - sg.b0) * (WAVES / KS) + wave / KS) * R, N = sg.N, K = ga.K, M = ga.M;
    if (!NV && n0 >= N) return;  // (with KS = 4 all waves of a workgroup or none)
    const TW* W = (const TW*)sg.W;
    const TX* X = (const TX*)ga.X;
    constexpr int NVX = NV ? NV : 1, TPB = WAVE * GN_WAVES;
    __shared__ __attribute__((aligned(16))) uint16_t xs[MX][NV ? NV * 4 * TPB : 1];
    __shared__ float red[MX][GN_WAVES];
    float4 xv[MX][NVX];
    uint2 wv[NVX];
    if constexpr (NV > 0) {
#pragma unroll
        for (int i = 0; i < NV; i++) {
            const int k = 4 * ((int)threadIdx.x + TPB * i), kk = k < K ? k : 0;
#pragma unroll
            for (int m = 0; m < MX; m++)
                xv[m][i] = *(const float4*)((const float*)ga.X + (size_t)min(m, M - 1) * ga.ldx + kk);
            wv[i] = *(const uint2*)(ga.nw + kk);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    // this wave's pieces: every KS-th from k0; pieces past a row's end repeat its first values, taken as zeros
    const bool ragged = K % (KS * PIECE) != 0;
    const int np = ((K + PIECE - 1) / PIECE + KS - 1) / KS, k0 = (wave % KS) * PIECE + V * lane;
    auto off = [&](int p) { return p * (KS * PIECE) + k0 < K ? p * (KS * PIECE) + k0 : 0; };
    const TW* wrow[R];
#pragma unroll
    for (int r = 0; r < R; r++) wrow[r] = W + (size_t)min(n0 + r, N - 1) * K;  // uniform
    u4v q[PD][R];
    auto load = [&](int slot, int p) {
        const int k = off(p);
#pragma unroll
        for (int r = 0; r < R; r++) q[slot][r] = __builtin_nontemporal_load((const u4v*)(wrow[r] + k));
    };
#pragma unroll
    for (int d = 0; d < PD; d++)
        if (d < np) load(d, d);
    // the row of W whose sum this lane ends up with, and what it is added to
    int own = 0;
#pragma unroll
    for (int h = R / 2, b = WAVE / 2; h > 0; h /= 2, b /= 2) own += lane & b ? h : 0;
    const int n = n0 + own;
    float y0[MX];
#pragma unroll
    for (int m = 0; m < MX; m++)
        y0[m] = ga.accumulate ? sg.Y[(size_t)min(m, M - 1) * sg.ldy + min(n, N - 1)] : 0.f;
    if constexpr (NV > 0) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int m = 0; m < MX; m++) {
            float ss = 0.f;
#pragma unroll
            for (int i = 0; i < NV; i++) {
                const float4 v = xv[m][i];
                const float q2 = v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
                ss += 4 * ((int)threadIdx.x + TPB * i) < K ? q2 : 0.f;
            }
            ss = wave_sum_dpp(ss);
            if (lane == 0) red[m][wave] = ss;
        }
        lds_barrier();  // (leaves the weights in flight)
#pragma unroll
        for (int m = 0; m < MX; m++) {
            float ss = 0.f;
#pragma unroll
            for (int i = 0; i < GN_WAVES; i++) ss += red[m][i];
            const float inv = rsqrtf(ss / (float)K + ga.eps);
#pragma unroll
            for (int i = 0; i < NV; i++) {
                const float4 v = xv[m][i];
                *(uint2*)&xs[m][4 * (threadIdx.x + TPB * i)] =
                    uint2{f2bf2((v.x * inv) * (1.f + bf_lo(wv[i].x)), (v.y * inv) * (1.f + bf_hi(wv[i].x))),
                          f2bf2((v.z * inv) * (1.f + bf_lo(wv[i].y)), (v.w * inv) * (1.f + bf_hi(wv[i].y)))};
            }
        }
        lds_barrier();
    }
    float acc[MX][R];
#pragma unroll
    for (int m = 0; m < MX; m++)
#pragma unroll
        for (int r = 0; r < R; r++) acc[m][r] = 0.f;
    for (int p0 = 0; p0 < np; p0 += PD) {
#pragma unroll
        for (int d = 0; d < PD; d++) {
            const int p = p0 + d;
            if (p >= np) break;
            float x[MX][V];
            const bool in = p * (KS * PIECE) + k0 < K;
#pragma unroll
            for (int m = 0; m < MX; m++) {
                if constexpr (NV > 0) gv_x<V>((const TX*)xs[m] + off(p), x[m]);
                else gv_x<V>(X + (size_t)min(m, M - 1) * ga.ldx + off(p), x[m]);
#pragma unroll
                for (int i = 0; i < V; i++) x[m][i] = in ? x[m][i] : 0.f;
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                float f[V];
                u4v w = q[d][r];
                if (ragged) w = in ? w : u4v{0, 0, 0, 0};  // (0 x Inf of the repeated values is no 0)
                GvW<TW>::unpack(w, f);
#pragma unroll
                for (int m = 0; m < MX; m++)
#pragma unroll
                    for (int i = 0; i < V; i++) acc[m][r] = fmaf(f[i], x[m][i], acc[m][r]);
                // one row's weights are unpacked at a time (registers)
#pragma unroll
                for (int m = 0; m < MX; m++) asm volatile("" : "+v"(acc[m][r]));
                __builtin_amdgcn_sched_barrier(0);
            }
            if (p + PD < np) load(d, p + PD);
        }
    }
    // sums over the lanes: halving exchanges leave row `own` of the R in each lane
#pragma unroll
    for (int h = R / 2, b = WAVE / 2; h > 0; h /= 2, b /= 2) {
        const bool up = lane & b;
#pragma unroll
        for (int m = 0; m < MX; m++)
#pragma unroll
            for (int i = 0; i < h; i++) {
                const float keep = up ? acc[m][i + h] : acc[m][i], give = up ? acc[m][i] : acc[m][i + h];
                acc[m][i] = keep + __shfl_xor(give, b, WAVE);
            }
    }
#pragma unroll
    for (int b = WAVE / 2 / R; b > 0; b /= 2)
#pragma unroll
        for (int m = 0; m < MX; m++) acc[m][0] += __shfl_xor(acc[m][0], b, WAVE);
    if constexpr (KS > 1) {
        __shared__ float ksum[WAVES][MX][R];
        if (lane % (WAVE / R) == 0)
#pragma unroll
            for (int m = 0; m < MX; m++) ksum[wave][m][own] = acc[m][0];
        lds_barrier();
        if (wave % KS) return;
#pragma unroll
        for (int m = 0; m < MX; m++) {
#pragma unroll
            for (int i = 1; i < KS; i++) acc[m][0] += ksum[wave + i][m][own];
        }
    }
    if (lane % (WAVE / R) || n >= N) return;
    const float s = sg.scale ? bf2f(sg.scale[n]) : 1.f;
#pragma unroll
    for (int m = 0; m < MX; m++) {
        if (m >= M) break;
        sg.Y[(size_t)m * sg.ldy + n] = y0[m] + acc[m][0] * s;
    }
}

template <typename TW, typename TX, int R, int MX, int PD, int NV = 0, int KS = 1>
int launch_gv(GemvArgs ga, hipStream_t st) {
    constexpr int WAVES = NV ? GN_WAVES : 4, G = WAVES / KS * R;  // rows of W of a workgroup
    int b = 0;
    for (int i = 0; i < ga.nseg; i++) {
        ga.seg[i].b0 = b;
        b += (int)(((long long)ga.seg[i].N + G - 1) / G);
    }
    gemv_kernel<TW, TX, R, MX, PD, NV, KS><<<b, WAVE * WAVES, 0, st>>>(ga);
    return after_launch("gemv");
}

}  // namespace

namespace aegist {

template <typename TW, typename TX, int MX>
static int gemv_launch(const GemvArgs& ga, long long rows, hipStream_t st) {
    // Four waves a row group where K gives each a piece (R = 2 and 8 measured 2 to 15% slower; int8 with
    // K = 2048, two idle waves of four: 4096 rows 5.2 -> 5.8 us).
    // Otherwise whole rows per wave, about 2048 waves where the weights allow it, since a wave's whole
    // stream should be in flight at once; int8 takes 4 rows at most (16 values of x per lane and piece
    // in registers), bf16 2 (4 and 8 measured 5 to 15% slower).
    if constexpr (std::is_same<TW, int8_t>::value) {
        if (ga.K > 3072) return launch_gv<TW, TX, 4, MX, 1, 0, 4>(ga, st);
        if (rows >= 4096) return launch_gv<TW, TX, 4, MX, 2>(ga, st);
        if (rows >= 1024) return launch_gv<TW, TX, 2, MX, 2>(ga, st);
        return launch_gv<TW, TX, 1, MX, 4>(ga, st);
    } else {
        if (ga.K > 1536) return launch_gv<TW, TX, 4, MX, 2, 0, 4>(ga, st);
        if (rows > 2048) return launch_gv<TW, TX, 2, MX, 4>(ga, st);
        return launch_gv<TW, TX, 1, MX, 8>(ga, st);
    }
}

template <typename TW, typename TX>
static int gemv_run(const GemvArgs& ga, long long rows, hipStream_t st) {
    return ga.M == 1 ? gemv_launch<TW, TX, 1>(ga, rows, st) : gemv_launch<TW, TX, 2>(ga, rows, st);
}

// M = 1 or 2 rows of X; the caller has checked K % 16 == 0 and the 16-byte alignment of every row.
int launch_gemv(const void* X, int x_dtype, long long ldx, int w_dtype, int nseg, const void* const* W,
                const uint16_t* const* scale, float* const* Y, const long long* ldy, const int* N, int M, int K,
                int accumulate, hipStream_t st) {
    if (nseg < 1 || nseg > GV_SEG || M < 1 || M > 2) return fail(AEGIST_ERR_SHAPE, "gemv: 1 or 2 rows, 1 to 4 weights");
    GemvArgs ga{};
    ga.X = X;
    ga.ldx = ldx;
    ga.nseg = nseg;
    ga.M = M;
    ga.K = K;
    ga.accumulate = accumulate;
    long long rows = 0;
    for (int i = 0; i < nseg; i++) {
        ga.seg[i] = GemvSeg{W[i], scale[i], Y[i], ldy[i], N[i], 0};
        rows += N[i];
    }
    if (w_dtype == AEGIST_I8)
        return x_dtype == AEGIST_F32 ? gemv_run<int8_t, float>(ga, rows, st) : gemv_run<int8_t, uint16_t>(ga, rows, st);
    return x_dtype == AEGIST_F32 ? gemv_run<uint16_t, float>(ga, rows, st) : gemv_run<uint16_t, uint16_t>(ga, rows, st);
}

// Whether launch_gemv_norm takes these rows.
bool gemv_norm_fits(const float* x, const uint16_t* nw, int M, int K) {
    return M >= 1 && M <= 2 && K >= 16 && K % 16 == 0 && K <= 8192 && (uintptr_t)x % 16 == 0 && (uintptr_t)nw % 8 == 0;
}

template <int MX>
static int gemv_norm_run(const GemvArgs& ga, hipStream_t st) {
    // 8 rows per workgroup (two groups of four waves); measured on one card on a generation of 16 tokens of a
    // 4-layer stack at one / two rows: 2430 / 2655 us, with 16 rows (R = 2 over whole rows) 2515 / 2718, with
    // 4 rows and 4 waves 2436 / 2664, with 4 rows and 8 waves 2504 / 2802, with 16 waves 2585 / 2824
    if (ga.K <= 2048) return launch_gv<uint16_t, uint16_t, 4, MX, 1, 1, 4>(ga, st);
    if (ga.K <= 4096) return launch_gv<uint16_t, uint16_t, 4, MX, 2, 2, 4>(ga, st);
    return launch_gv<uint16_t, uint16_t, 4, MX, 2, 4, 4>(ga, st);
}

// Y_s[m, n] = sum_k bf16(ZNorm(x[m]))[k] W_s[n, k]: the layer stack's norm and input projections at one
// or two rows. x [M, K] fp32, bf16 weights with 16-byte aligned rows; gemv_norm_fits holds.
int launch_gemv_norm(const float* x, const uint16_t* nw, float eps, int nseg, const uint16_t* const* W, float* const* Y,
                     const long long* ldy, const int* N, int M, int K, hipStream_t st) {
    if (nseg < 1 || nseg > GV_SEG || !gemv_norm_fits(x, nw, M, K))
        return fail(AEGIST_ERR_SHAPE, "gemv_norm: 1 or 2 aligned rows of up to 8192, 1 to 4 weights");
    GemvArgs ga{};
    ga.X = x;
    ga.ldx = K;
    ga.nseg = nseg;
    ga.M = M;
    ga.K = K;
    ga.nw = nw;
    ga.eps = eps;
    for (int i = 0; i < nseg; i++) {
        if ((uintptr_t)W[i] % 16) return fail(AEGIST_ERR_SHAPE, "proj: W needs 16-byte aligned rows");
        ga.seg[i] = GemvSeg{W[i], nullptr, Y[i], ldy[i], N[i], 0};
    }
    return M == 1 ? gemv_norm_run<1>(ga, st) : gemv_norm_run<2>(ga, st);
}

}  // namespace aegist
