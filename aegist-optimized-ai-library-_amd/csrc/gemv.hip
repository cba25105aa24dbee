// Projections of one or two rows of X (batch-1 decode; the engine's gemv_i8 and
// gemv_bf16, aegist.cu:84-124): Y_s[m, n] (+)= scale_s[n] sum_k X[m, k] W_s[n, k], up to four weights
// sharing X in one launch.
//
// HBM-bound on W and, at these sizes (a 17 MB weight is 3.5 us of HBM), on the launch's one round trip.
// A load instruction is 1 KB of one row (16 bytes per lane), so the stream is contiguous; the products
// run on the VALU in fp32 (x and w exactly, no hi / lo parts), which at one or two rows costs less than
// the MFMA forms' conversion, LDS and barrier steps; the R rows of a wave are summed over the lanes by
// halving exchanges. R and the pieces in flight by row count: see gemv_launch.
// Measured against the MFMA row-tile kernel this replaces (us, weights from HBM, one row): bf16 W, fp32 X
// 32768 x 2048 36.3 -> 22.9 (5.9 TB/s), 256 x 2048 6.3 -> 3.8; int8 W, fp32 X 2048 x 4096 8.4 -> 6.5,
// 4096 x 2048 5.6 -> 5.3, 512 x 2048 5.6 -> 3.7, 8192 x 2048 7.1 (alike); bf16 both 12352 x 2048
// 12.3 -> 11.6, 2048 x 4096 7.5 -> 6.8.
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
};

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
// pieces, so a load instruction is 1 KB of one row.
template <typename TW, typename TX, int R, int MX, int PD>
__global__ void __launch_bounds__(256) gemv_kernel(const GemvArgs ga) {
    constexpr int V = GvW<TW>::kVals, PIECE = V * WAVE;
    int si = 0;
#pragma unroll
    for (int i = 1; i < GV_SEG; i++)
        if (i < ga.nseg && (int)blockIdx.x >= ga.seg[i].b0) si = i;
    const GemvSeg sg = ga.seg[si];
    const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int n0 = (((int)blockIdx.x - sg.b0) * 4 + wave) * R, N = sg.N, K = ga.K, M = ga.M;
    if (n0 >= N) return;
    const TW* W = (const TW*)sg.W;
    const TX* X = (const TX*)ga.X;
    const int np = (K + PIECE - 1) / PIECE;
    // pieces past a row's end repeat its first values against zeros
    auto off = [&](int p) { return p * PIECE + V * lane < K ? p * PIECE + V * lane : 0; };
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
            const bool in = p * PIECE + V * lane < K;
#pragma unroll
            for (int m = 0; m < MX; m++) {
                gv_x<V>(X + (size_t)min(m, M - 1) * ga.ldx + off(p), x[m]);
#pragma unroll
                for (int i = 0; i < V; i++) x[m][i] = in ? x[m][i] : 0.f;
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                float f[V];
                GvW<TW>::unpack(q[d][r], f);
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
    int own = 0;
#pragma unroll
    for (int h = R / 2, b = WAVE / 2; h > 0; h /= 2, b /= 2) {
        const bool up = lane & b;
        own += up ? h : 0;
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
    const int n = n0 + own;
    if (lane % (WAVE / R) || n >= N) return;
    const float s = sg.scale ? bf2f(sg.scale[n]) : 1.f;
#pragma unroll
    for (int m = 0; m < MX; m++) {
        if (m >= M) break;
        float* y = sg.Y + (size_t)m * sg.ldy + n;
        *y = (ga.accumulate ? *y : 0.f) + acc[m][0] * s;
    }
}

template <typename TW, typename TX, int R, int MX, int PD>
int launch_gv(GemvArgs ga, hipStream_t st) {
    int b = 0;
    for (int i = 0; i < ga.nseg; i++) {
        ga.seg[i].b0 = b;
        b += (ga.seg[i].N + 4 * R - 1) / (4 * R);
    }
    gemv_kernel<TW, TX, R, MX, PD><<<b, 256, 0, st>>>(ga);
    return after_launch("gemv");
}

}  // namespace

namespace aegist {

template <typename TW, typename TX, int MX>
static int gemv_launch(const GemvArgs& ga, long long rows, hipStream_t st) {
    // rows per wave: about 2048 waves where the weights allow it, since a wave's whole stream should
    // be in flight at once; int8 takes 4 rows at most (16 values of x per lane and piece in
    // registers), bf16 2 (4 and 8 measured 5 to 15% slower)
    if constexpr (std::is_same<TW, int8_t>::value) {
        if (rows >= 4096) return launch_gv<TW, TX, 4, MX, 2>(ga, st);
        if (rows >= 1024) return launch_gv<TW, TX, 2, MX, 2>(ga, st);
        return launch_gv<TW, TX, 1, MX, 4>(ga, st);
    } else {
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

}  // namespace aegist
