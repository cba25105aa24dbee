// Projections around the mixer: the weight-streaming matmuls of QLinear
// (aegist/model.py:78-93: int8 weight, per-output-row absmax scale in bf16) and of plain bf16
// weights, as the engine runs them (aegist_rs/kernels/aegist.cu:84-172: gemv_i8, gemv_bf16,
// gemm_i8; called through HybridEngine::mm, aegist_rs/src/hybrid.rs:717-735):
//     Y[m, n] (+)= scale[n] * sum_k X[m, k] W[n, k]
// with fp32 accumulation. accumulate = 1 adds into Y (the residual add of the out-projections).
//
// This file picks the kernel by size and holds the weight stream of decode batches. One or two rows
// run in gemv.hip, the rest up to a few thousand in gemm_mid.hip, the largest in gemm.hip.
//
// int8 and bf16 weights are exact in bf16. From three rows on an fp32 X is split into bf16 hi + lo (hi
// truncated, lo rounded: x = hi + lo to 2^-16 |x|) and both parts go through the MFMA, so the result matches
// an fp32 dot product to ~1e-5 relative; a bf16 X needs only the hi part. One and two rows are fp32
// products on the VALU.
#include "common.h"

#include <algorithm>
#include <cstdlib>

using namespace aegist;

namespace aegist {
bool gemm_bf16_fits(const void* X, long long ldx, const void* W, long long ldw, int M, int N, int K);
bool gemm_i8f32_fits(const void* X, long long ldx, const void* W, long long ldw, int M, int N, int K);
int launch_gemm_i8f32(const float* X, long long ldx, const int8_t* W, long long ldw, const uint16_t* scale, float* Y,
                      long long ldy, int M, int N, int K, int accumulate, hipStream_t st);
int launch_gemm_bf16(const uint16_t* X, long long ldx, const uint16_t* W, long long ldw, float* Y, long long ldy, int M,
                     int N, int K, int accumulate, hipStream_t st);
int launch_gemm_bf16_multi(const uint16_t* X, long long ldx, int nseg, const uint16_t* const* W, const long long* ldw,
                           float* const* Y, const long long* ldy, const int* N, int M, int K, int accumulate,
                           hipStream_t st);
int gemm_mid_form(int x_dtype, int nseg, const int* N, int M, int K, bool tile256, bool stacked);
int launch_gemv(const void* X, int x_dtype, long long ldx, int w_dtype, int nseg, const void* const* W,
                const uint16_t* const* scale, float* const* Y, const long long* ldy, const int* N, int M, int K,
                int accumulate, hipStream_t st);
int launch_gemm_mid(int form, const void* X, int x_dtype, long long ldx, int w_dtype, int nseg, const void* const* W,
                    const uint16_t* const* scale, float* const* Y, const long long* ldy, const int* N, int M, int K,
                    int accumulate, hipStream_t st);
}  // namespace aegist

namespace {

bool stream_enabled() {
    static const bool on = [] {
        const char* e = getenv("AEGIST_PROJ_STREAM");
        return !(e && e[0] == '0');
    }();
    return on;
}

// Up to four weight matrices that share X (a layer's input projections) go in one launch;
// segment i owns workgroups [tile0[i], tile0[i+1]) along grid x.
constexpr int MAX_SEG = 4;
struct ProjSeg {
    const void* W;
    const uint16_t* scale;  // per-row scale or null
    float* Y;
    long long ldy;
    int N;
};
struct ProjSegs {
    ProjSeg s[MAX_SEG];
    int tile0[MAX_SEG + 1];
    int n;
};

// ---------------------------------------------------------------------------------------------
// Decode-size bf16 projections (M <= 16) with W staged through LDS. Lanes that hold (row, run)
// fragments straight from global memory read 16 rows x 64 or 128 bytes per instruction, and the
// DRAM side serves that at ~half the rate of contiguous reads (same card: a read-only kernel
// with that pattern 51% of HBM on 50 MB, 1 KB-contiguous reads 67%). Here every load
// instruction is a direct global -> LDS copy of 1 KB of one pair of W rows (512 bytes each) and
// the MFMA A operands are read back from LDS. Per workgroup: 16 NW rows of W (16 per wave, so
// a wave owns whole output rows and no cross-wave reduction is needed) over all of K, in chunks
// of KC = 256 k through an NS-stage ring (NS = 2 measured best: 3 to 5 stages were 2-50%
// slower); the X rows of each chunk ride in the same stage.
// Slots of 16 bytes in a staged row are XOR-swizzled by the row index (the global address of
// each lane is permuted, the 1 KB it covers is not), so the 16 rows a fragment read touches
// hit 16 different bank groups.
constexpr int SKC = 256;  // k per chunk
template <int NW, int NS>
struct StreamSmem {
    static constexpr int XB = 16 * SKC * 2;  // X bytes per stage (16 rows)
    __attribute__((aligned(16))) unsigned char w[NS][16 * NW][SKC * 2];
    __attribute__((aligned(16))) unsigned char x[NS][XB];
};

// 16 bytes per lane straight from global memory into LDS at lds + 16 lane (lds uniform). Kept
// in a device function: the builtin in a kernel body keeps the host pass from emitting the
// kernel's launch stub.
__device__ __forceinline__ void g2lds16(const void* src, void* lds) {
    __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void*)lds, 16, 0, 0);
}
// The same copy with the nontemporal hint (cache-policy bit 1): the weight stream is read once
// per launch, and kept out of L2 / MALL it runs faster (config 4 decode step 1.637 -> 1.583 ms).
__device__ __forceinline__ void g2lds16_nt(const void* src, void* lds) {
    __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void*)lds, 16, 0, 2);
}

__device__ __forceinline__ void wait_vm(int n) {
    // s_waitcnt vmcnt(n) with the other counters left alone (gfx9 encoding: vmcnt in bits 3:0
    // and 15:14, expcnt 6:4, lgkmcnt 11:8)
    switch (n) {
#define AEG_W(N) case N: __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8)); break;
        AEG_W(0) AEG_W(1) AEG_W(2) AEG_W(3) AEG_W(4) AEG_W(5) AEG_W(6) AEG_W(7) AEG_W(8) AEG_W(9) AEG_W(10)
        AEG_W(11) AEG_W(12) AEG_W(13) AEG_W(14) AEG_W(15) AEG_W(16) AEG_W(20) AEG_W(24) AEG_W(28) AEG_W(32)
        AEG_W(40) AEG_W(48)
#undef AEG_W
        default: __builtin_amdgcn_s_waitcnt(0);
    }
}

template <int NW, int NS>
__global__ __launch_bounds__(64 * NW) void proj_stream_kernel(const uint16_t* __restrict__ X, long long ldx,
                                                               const ProjSegs segs, int M, int K, int accumulate,
                                                               float* __restrict__ part) {
    __shared__ StreamSmem<NW, NS> sm;
    constexpr int RW = 16 * NW;                       // W rows per workgroup
    constexpr int WI = RW / 2 / NW;                   // W load instructions per wave per stage (= 8)
    constexpr int XI = StreamSmem<NW, NS>::XB / 1024 / NW;  // X load instructions per wave per stage
    static_assert(XI * NW * 1024 == StreamSmem<NW, NS>::XB, "X stage must split evenly over the waves");
    constexpr int PER = WI + XI;                      // loads per wave per stage
    const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
    const int r16 = lane % 16, g = lane / 16;
    int si = 0;
#pragma unroll
    for (int i = 1; i < MAX_SEG; i++)
        if (i < segs.n && (int)blockIdx.x >= segs.tile0[i]) si = i;
    const uint16_t* __restrict__ W = (const uint16_t*)segs.s[si].W;
    float* __restrict__ Y = segs.s[si].Y;
    const long long ldy = segs.s[si].ldy;
    const int N = segs.s[si].N;
    const int n0 = ((int)blockIdx.x - segs.tile0[si]) * RW;
    // split K (gridDim.y > 1, one weight matrix): chunks [c0, c1) of this workgroup, partial sums
    // to part[blockIdx.y][m][n] (the caller adds the splits in order)
    const int nall = K / SKC, ks = blockIdx.y, nks = gridDim.y;
    const int c0 = ks * nall / nks, c1 = (ks + 1) * nall / nks, nch = c1 - c0;

    // stage loads of chunk c: this wave's WI pairs of W rows and XI kilobytes of X rows
    auto issue = [&](int cc) {
        const int st = cc % NS, c = c0 + cc;
#pragma unroll
        for (int i = 0; i < WI; i++) {
            const int pr = wave * WI + i;             // row pair
            const int row = 2 * pr + lane / 32, slot = (lane % 32) ^ (row & 15);
            const int n = min(n0 + row, N - 1);
            const uint16_t* src = W + (size_t)n * K + (size_t)c * SKC + slot * 8;
            g2lds16_nt(src, &sm.w[st][2 * pr][0]);
        }
        constexpr int XROWB = SKC * 2;   // bytes of one X row per chunk
#pragma unroll
        for (int i = 0; i < XI; i++) {
            const int off = (wave * XI + i) * 1024 + lane * 16;  // byte offset in the stage's X block
            const int m = off / XROWB, kb = off % XROWB;
            const int mm = min(m, M - 1);
            const unsigned char* src = (const unsigned char*)(X + (size_t)mm * ldx + (size_t)c * SKC) + kb;
            g2lds16(src, &sm.x[st][(wave * XI + i) * 1024]);
        }
    };

    f32x4 acc{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < NS - 1; c++)
        if (c < nch) issue(c);
    const int row = 16 * wave + r16;  // this lane's W row (A operand)
    for (int c = 0; c < nch; c++) {
        // chunk c's loads are done once only the later chunks' (at most NS - 2) are in flight
        const int later = min(NS - 2, nch - 1 - c);
        wait_vm(later * PER);
        lds_barrier();
        if (c + NS - 1 < nch) issue(c + NS - 1);  // into the stage chunk c - 1 used (all waves are past it)
        const int st = c % NS;
#pragma unroll
        for (int i = 0; i < SKC / 32; i++) {
            // k block i of the chunk: lane (row, g) takes slot 4 i + g of its row (swizzled)
            const bf16x8 a = *(const bf16x8*)&sm.w[st][row][((4 * i + g) ^ (row & 15)) * 16];
            const bf16x8 b = *(const bf16x8*)&sm.x[st][(r16 * SKC + 32 * i + 8 * g) * 2];
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
        }
    }
    // lane (m = r16, g) holds Y[m][n0 + 16 wave + 4 g .. +3]
    const int nb = n0 + 16 * wave + 4 * g, m = r16;
    if (m >= M || nb >= N) return;
    if (part) {
        float* pp = part + ((size_t)ks * M + m) * N + nb;
        if (nb + 3 < N && (N % 4) == 0) {
            *(f32x4*)pp = acc;
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (nb + j < N) pp[j] = acc[j];
        }
        return;
    }
    float* yp = Y + (size_t)m * ldy + nb;
    if (nb + 3 < N && ((uintptr_t)yp % 16) == 0) {
        f32x4 v = acc;
        if (accumulate) v += *(const f32x4*)yp;
        *(f32x4*)yp = v;
    } else {
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (nb + j < N) yp[j] = (accumulate ? yp[j] : 0.f) + acc[j];
    }
}

template <int NW, int NS>
int launch_stream(const uint16_t* X, long long ldx, ProjSegs segs, int M, int K, int accumulate, hipStream_t st,
                  float* part = nullptr, int nks = 1) {
    int t = 0;
    for (int i = 0; i < segs.n; i++) {
        segs.tile0[i] = t;
        t += (segs.s[i].N + 16 * NW - 1) / (16 * NW);
    }
    segs.tile0[segs.n] = t;
    proj_stream_kernel<NW, NS><<<dim3(t, nks), 64 * NW, 0, st>>>(X, ldx, segs, M, K, accumulate, part);
    return 0;
}

// The kernel of a product whose operands are all below 2^31 - 16 bytes.
int run_proj(const void* X, int xd, long long ldx, int wd, const ProjSegs& segs, int M, int K, int accumulate,
             hipStream_t st) {
    const bool i8 = wd == AEGIST_I8, f32 = xd == AEGIST_F32;
    const void* W[MAX_SEG];
    const uint16_t* scale[MAX_SEG];
    float* Y[MAX_SEG];
    long long ldw[MAX_SEG], ldy[MAX_SEG], rows = 0, tiles = 0;
    int N[MAX_SEG];
    // past 64 rows the 256 x 256 MFMA tiles take int8 weights with fp32 activations (the engine's
    // gemm_i8, one launch per weight) and unscaled bf16 weights with bf16 activations (all weights
    // in one launch, stacked along N, when each but the last has a multiple of 8 rows)
    bool tile256 = M > 64 && i8 == f32, stack8 = segs.n <= 3, scaled = false;
    for (int i = 0; i < segs.n; i++) {
        const ProjSeg& sg = segs.s[i];
        W[i] = sg.W;
        scale[i] = sg.scale;
        Y[i] = sg.Y;
        ldw[i] = K;
        ldy[i] = sg.ldy;
        N[i] = sg.N;
        rows += sg.N;
        tiles += (sg.N + 31) / 32;
        scaled |= sg.scale != nullptr;
        if (i8) tile256 = tile256 && gemm_i8f32_fits(X, ldx, sg.W, K, M, sg.N, K);
        else tile256 = tile256 && !sg.scale && gemm_bf16_fits(X, ldx, sg.W, K, M, sg.N, K);
        if (i + 1 < segs.n && sg.N % 8) stack8 = false;
    }
    // one or two rows: whole-row loads on the VALU; two rows on int8 weights of 8192 and more rows stay
    // with the MFMA form (131072 x 2048: 63 against 78 us, 8192 x 2048 7.4 against 7.7)
    if (M == 1 || (M == 2 && !(i8 && rows >= 8192)))
        return launch_gemv(X, xd, ldx, wd, segs.n, W, scale, Y, ldy, N, M, K, accumulate, st);
    // bf16 weights and activations at 3 to 16 rows, no row scales, K a multiple of the chunk: the
    // LDS-staged stream when it takes more than one workgroup per CU (9216 x 2048, 16 rows: 11.3
    // against 12.8 us on the MFMA form, 12352 x 2048 13.0 against 14.4; below, the K split over
    // the waves of a workgroup keeps more loads in flight: 8192 x 2048 11.7 against 8.8 us)
    if (M <= 16 && !i8 && !f32 && K % SKC == 0 && !scaled && tiles > 256 && stream_enabled()) {
        launch_stream<2, 2>((const uint16_t*)X, ldx, segs, M, K, accumulate, st);
        return after_launch("proj_stream");
    }
    const int form = gemm_mid_form(xd, segs.n, N, M, K, tile256, !i8 && stack8);
    if (form >= 0)
        return launch_gemm_mid(form, X, xd, ldx, wd, segs.n, W, scale, Y, ldy, N, M, K, accumulate, st);
    if (i8) {
        for (int i = 0; i < segs.n; i++) {
            int rc = launch_gemm_i8f32((const float*)X, ldx, (const int8_t*)W[i], K, scale[i], Y[i], ldy[i], M, N[i], K,
                                       accumulate, st);
            if (rc) return rc;
        }
        return 0;
    }
    if (stack8)
        return launch_gemm_bf16_multi((const uint16_t*)X, ldx, segs.n, (const uint16_t* const*)W, ldw, Y, ldy, N, M, K,
                                      accumulate, st);
    for (int i = 0; i < segs.n; i++) {
        int rc = launch_gemm_bf16((const uint16_t*)X, ldx, (const uint16_t*)W[i], K, Y[i], ldy[i], M, N[i], K, accumulate,
                                  st);
        if (rc) return rc;
    }
    return 0;
}

}  // namespace

namespace aegist {

// Y_i[m, n] (+)= scale_i[n] * sum_k X[m, k] W_i[n, k] for nseg (<= 4) weight matrices sharing X.
int launch_proj_multi(const void* X, int x_dtype, long long ldx, int w_dtype, int nseg, const void* const* W,
                      const uint16_t* const* scale, float* const* Y, const long long* ldy, const int* N, int M, int K,
                      int accumulate, hipStream_t st) {
    if (nseg < 1 || nseg > MAX_SEG) return fail(AEGIST_ERR_SHAPE, "proj: 1 to 4 weight matrices per launch");
    if (M < 0 || K < 0) return fail(AEGIST_ERR_SHAPE, "proj: negative size");
    if (K % 16) return fail(AEGIST_ERR_SHAPE, "proj: K must be a multiple of 16");
    const int xs = x_dtype == AEGIST_F32 ? 4 : 2;
    if (ldx < K || (ldx * xs) % 16 || (uintptr_t)X % 16)
        return fail(AEGIST_ERR_SHAPE, "proj: X needs 16-byte aligned rows (ldx >= K)");
    ProjSegs segs{};
    for (int i = 0; i < nseg; i++) {
        if (N[i] < 0) return fail(AEGIST_ERR_SHAPE, "proj: negative size");
        if (N[i] == 0) continue;
        if (ldy[i] < N[i]) return fail(AEGIST_ERR_SHAPE, "proj: ldy < N");
        if ((uintptr_t)W[i] % 16) return fail(AEGIST_ERR_SHAPE, "proj: W needs 16-byte aligned rows");
        segs.s[segs.n++] = ProjSeg{W[i], scale ? scale[i] : nullptr, Y[i], ldy[i], N[i]};
    }
    if (M == 0 || segs.n == 0) return 0;
    if ((w_dtype != AEGIST_I8 && w_dtype != AEGIST_BF16) || (x_dtype != AEGIST_F32 && x_dtype != AEGIST_BF16))
        return fail(AEGIST_ERR_DTYPE, "proj: W must be AEGIST_I8 or AEGIST_BF16, X AEGIST_F32 or AEGIST_BF16");
    // the kernels address operands through 31-bit byte offsets: larger ones go in blocks of rows
    const long long lim = 0x7ffffff0LL, ws = w_dtype == AEGIST_I8 ? 1 : 2;
    // (rows so long that 8 of W or 3 of X pass the limit: one row of X at a time, whose kernel does not)
    const bool huge = 8LL * K * ws >= lim || 3 * ldx * xs >= lim;
    const long long mb = huge ? 1 : (lim - 1) / std::max(1LL, ldx * xs);
    const long long nb = huge ? 0x7fffffffLL : std::max(8LL, (lim - 1) / std::max(1LL, K * ws) / 256 * 256);
    if (M <= mb) {
        bool whole = true;
        for (int i = 0; i < segs.n; i++) whole &= segs.s[i].N <= nb;
        if (whole) return run_proj(X, x_dtype, ldx, w_dtype, segs, M, K, accumulate, st);
    }
    for (long long m = 0; m < M; m += mb)
        for (int i = 0; i < segs.n; i++)
            for (long long n = 0; n < segs.s[i].N; n += nb) {
                const ProjSeg& sg = segs.s[i];
                ProjSegs one{};
                one.n = 1;
                one.s[0] = ProjSeg{(const char*)sg.W + n * K * ws, sg.scale ? sg.scale + n : nullptr, sg.Y + m * sg.ldy + n,
                                   sg.ldy, (int)std::min<long long>(nb, sg.N - n)};
                int rc = run_proj((const char*)X + m * ldx * xs, x_dtype, ldx, w_dtype, one,
                                  (int)std::min<long long>(mb, M - m), K, accumulate, st);
                if (rc) return rc;
            }
    return 0;
}

// Split-K form for decode sizes: part[ks][m][n] = sum over the ks-th of nks slices of K of
// X[m, k] W[n, k] (bf16 X and W, M <= 16, K a multiple of 256 with at least nks chunks). The
// caller adds the nks slices in order (the layer stack does it inside the next ZNorm).
int launch_proj_splitk(const uint16_t* X, long long ldx, const uint16_t* W, float* part, int nks, int M, int N, int K,
                       hipStream_t st) {
    if (M < 1 || M > 16 || N < 1 || K % SKC || K / SKC < nks || nks < 1 || ldx < K || ldx % 8 || (uintptr_t)X % 16 ||
        (uintptr_t)W % 16)
        return fail(AEGIST_ERR_SHAPE, "proj_splitk: need M <= 16, K % 256 == 0, K / 256 >= splits, aligned rows");
    ProjSegs segs{};
    segs.s[0] = ProjSeg{W, nullptr, part, N, N};
    segs.n = 1;
    launch_stream<2, 2>(X, ldx, segs, M, K, 0, st, part, nks);
    return after_launch("proj_stream_splitk");
}

int launch_proj(const void* X, int x_dtype, long long ldx, const void* W, int w_dtype, const uint16_t* scale, float* Y,
                long long ldy, int M, int N, int K, int accumulate, hipStream_t st) {
    return launch_proj_multi(X, x_dtype, ldx, w_dtype, 1, &W, &scale, &Y, &ldy, &N, M, K, accumulate, st);
}

}  // namespace aegist

extern "C" int aegist_gemv_i8(const float* x, const int8_t* W, const uint16_t* scale, float* y, int N, int K,
                              int accumulate, void* stream) {
    return launch_proj(x, AEGIST_F32, K, W, AEGIST_I8, scale, y, N, 1, N, K, accumulate, AEG_STREAM(stream));
}

extern "C" int aegist_gemv_bf16(const float* x, const uint16_t* W, float* y, int N, int K, void* stream) {
    return launch_proj(x, AEGIST_F32, K, W, AEGIST_BF16, nullptr, y, N, 1, N, K, 0, AEG_STREAM(stream));
}

extern "C" int aegist_gemm_i8(const float* X, const int8_t* W, const uint16_t* scale, float* Y, int M, int N, int K,
                              int accumulate, void* stream) {
    return launch_proj(X, AEGIST_F32, K, W, AEGIST_I8, scale, Y, N, M, N, K, accumulate, AEG_STREAM(stream));
}

extern "C" int aegist_linear(const void* X, int x_dtype, long long ldx, const void* W, int w_dtype,
                             const uint16_t* scale, float* Y, long long ldy, int M, int N, int K, int accumulate,
                             void* stream) {
    return launch_proj(X, x_dtype, ldx, W, w_dtype, scale, Y, ldy, M, N, K, accumulate, AEG_STREAM(stream));
}

extern "C" int aegist_linear_multi(const void* X, int x_dtype, long long ldx, int w_dtype, int n, const void* const* W,
                                   const uint16_t* const* scale, float* const* Y, const long long* ldy, const int* N,
                                   int M, int K, int accumulate, void* stream) {
    if (!W || !Y || !ldy || !N) return fail(AEGIST_ERR_SHAPE, "linear_multi: null argument array");
    return launch_proj_multi(X, x_dtype, ldx, w_dtype, n, W, scale, Y, ldy, N, M, K, accumulate, AEG_STREAM(stream));
}
