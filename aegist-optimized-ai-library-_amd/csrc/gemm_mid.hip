// Projections of middling batches, Y_s[M, N_s] (+)= scale_s[n] X[M, K] W_s[N_s, K]^T for up to four
// weights sharing X: from 3 rows of X to as many as the 256 x 256 tiles of gemm.hip leave part of
// the chip idle for. int8 or bf16 W, fp32 or bf16 X, fp32 Y, on v_mfma_f32_16x16x32_bf16.
//
// What bounds it: at these sizes neither HBM (an 8192 x 2048 int8 weight is 17 MB, 3 us) nor the
// matrix cores, but how much of the chip a tile split fills and what every workgroup pulls through
// L2 (about 16 TB/s in all) and converts. So the tile varies: a workgroup is KG groups of NWN
// waves; wave (kg, wn) owns 16 RT rows of W against 16 MT rows of X over every KG-th 64-k step, and
// the groups' partial tiles are added in LDS in group order (deterministic, no workspace). W goes
// from global memory straight to MFMA operands in registers (each weight byte is read and converted
// once per workgroup, PD steps ahead); X goes through registers into LDS as bf16 hi (and, for fp32 X,
// lo) parts, split once per workgroup instead of once per wave and W row tile, double-buffered with
// one LDS-only barrier per step. 16-byte slots of a staged row are XOR-swizzled by the row.
//
// Measured against the kernels that served these sizes before (one card, us per launch in a graph; other cards
// and placements of the operands up to a quarter more: 300 x 8192 x 2048 int8 34 to 43, 1024 rows 62 to 70):
//   int8 W, fp32 X   300 x 8192 x 2048: 117 -> 34   300 x 2048 x 4096: 221 -> 25   1024 x 8192 x 2048: 119 -> 63
//   bf16 W, bf16 X    64 x 2048 x 4096: 21 -> 9.6    300 x 2048 x 4096: 83 -> 25     300 x 8192 x 2048: 47 -> 33
// Prefetching four steps instead of two, or accumulating in fewer, larger tiles at small M, gained
// nothing: a step costs 0.1 to 0.2 us even in the smallest tile (the barrier, the LDS round trip and
// the dependent products), which is why small tiles with K split over 8 waves win there.
#include "common.h"

#include <type_traits>

using namespace aegist;

namespace {

typedef int int4v __attribute__((ext_vector_type(4)));

constexpr int MKS = 64;                             // k per step
constexpr int kMidBufWord3 = 0x00020000;            // buffer resource word 3 on gfx9: 32-bit data, no swizzle
// past every operand (< 2^31 - 16 bytes): loads return 0. Offsets are unsigned, since a second load lies 16
// bytes past it
constexpr uint32_t kMidOob = 0x7ffffff0u;

constexpr int MID_SEG = 4;
struct MidSeg {
    const void* W;
    const uint16_t* scale;  // per-row scale or null
    float* Y;
    long long ldy;
    int N, t0;              // rows; first N tile of the launch
};
struct MidArgs {
    const void* X;
    MidSeg seg[MID_SEG];
    int nseg, ldx, M, K, accumulate, tiles_m, ntiles, per_xcd;
};

// offset of the 16 bytes that follow those at `off`
__device__ constexpr uint32_t next16(uint32_t off) { return off + 16; }
static_assert(next16(kMidOob) > kMidOob, "the load after an out-of-range one is out of range too");

__device__ __forceinline__ int4v buf16(__amdgpu_buffer_rsrc_t rs, uint32_t off) {
    return __builtin_bit_cast(int4v, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
}

// A lane's 16 weights of one row and step as two bf16x8 fragments; slot(h, g) is the 8-value slot
// of the step that fragment h of lane group g holds. Each load instruction of a wave covers 64
// contiguous bytes of 16 rows: int8 lanes take 16 consecutive values, bf16 lanes 8 of each half.
template <typename TW> struct MidW;
template <> struct MidW<int8_t> {
    int4v r;
    static __device__ __forceinline__ int slot(int h, int g) { return 2 * g + h; }
    // k0: first k of the step; rows end at K (a multiple of 16)
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rs, int row, int k0, int g, int K) {
        r = buf16(rs, k0 + 16 * g < K ? (uint32_t)(row + k0 + 16 * g) : kMidOob);
    }
    __device__ __forceinline__ bf16x8 frag(int h) const {
        // int8 -> fp32 is exact and keeps 8 significant bits, so its top half is the exact bf16
        uint32_t p[4];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint32_t d = (uint32_t)r[2 * h + i];
            const float f0 = (float)(int8_t)d, f1 = (float)(int8_t)(d >> 8);
            const float f2 = (float)(int8_t)(d >> 16), f3 = (float)(int8_t)(d >> 24);
            p[2 * i] = __builtin_amdgcn_perm(__float_as_uint(f1), __float_as_uint(f0), 0x07060302u);
            p[2 * i + 1] = __builtin_amdgcn_perm(__float_as_uint(f3), __float_as_uint(f2), 0x07060302u);
        }
        return __builtin_bit_cast(bf16x8, p);
    }
};
template <> struct MidW<uint16_t> {
    int4v r[2];
    static __device__ __forceinline__ int slot(int h, int g) { return 4 * h + g; }
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rs, int row, int k0, int g, int K) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int k = k0 + 32 * h + 8 * g;
            r[h] = buf16(rs, k < K ? (uint32_t)(row + k) * 2 : kMidOob);
        }
    }
    __device__ __forceinline__ bf16x8 frag(int h) const { return __builtin_bit_cast(bf16x8, r[h]); }
};

// 8 consecutive activations of one row
template <typename TX> struct MidX;
template <> struct MidX<float> {
    static constexpr int kParts = 2;
    int4v r[2];
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rs, uint32_t off) {
        r[0] = buf16(rs, off);
        r[1] = buf16(rs, next16(off));
    }
    // x = hi + lo, hi = x truncated to bf16, lo = the rounded remainder: |x - hi - lo| <= 2^-16 |x|
    __device__ __forceinline__ void store(unsigned char* dst, int part) const {
        uint32_t h[4], l[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t u0 = (uint32_t)r[e / 2][2 * (e % 2)], u1 = (uint32_t)r[e / 2][2 * (e % 2) + 1];
            h[e] = __builtin_amdgcn_perm(u1, u0, 0x07060302u);
            typedef float f2 __attribute__((ext_vector_type(2)));
            typedef __bf16 b2 __attribute__((ext_vector_type(2)));
            const f2 lo = {__uint_as_float(u0) - __uint_as_float(u0 & 0xffff0000u),
                           __uint_as_float(u1) - __uint_as_float(u1 & 0xffff0000u)};
            l[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(lo, b2));
        }
        *(uint4*)dst = uint4{h[0], h[1], h[2], h[3]};
        *(uint4*)(dst + part) = uint4{l[0], l[1], l[2], l[3]};
    }
};
template <> struct MidX<uint16_t> {
    static constexpr int kParts = 1;
    int4v r;
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rs, uint32_t off) { r = buf16(rs, off); }
    __device__ __forceinline__ void store(unsigned char* dst, int) const { *(int4v*)dst = r; }
};

// With exact bf16 X what is left of an output's error is the fp32 sums' and grows with the root of the number
// of products added one after the other. So they are short chains where they were before these tiles (kShort: up
// to 64 rows, and int8 weights): kSets sets of accumulators take the step's 32-k halves (and, of four, the
// steps) in turn, K / (KG kSets) products each; the forms of few K groups that int8 weights take at the largest
// batches add theirs up every kFlush steps. 2-norm error, one set and now: bf16 16 rows of 8192 x 2048 1.31e-7,
// 0.98e-7, of 2048 x 4096 1.37e-7, 1.06e-7, 64 of 12352 x 2048 1.86e-7, 0.98e-7; int8 W, bf16 X, 600 rows of
// 4096 x 8192 2.79e-7, 1.0e-7. It costs 0 to 6% at up to 64 rows, up to 14% at 300 of int8 12352 x 2048. (Past 64 rows
// bf16 W is in the place of full-K chains, except in the form of 4 K groups on 32 rows, whose chains would be
// longer than with the 8 before. fp32 X: its split's 2^-17 is 40 times as much; one set.)
template <typename TW, typename TX, int RT, int MT, int KG, bool kShort>
struct MidSums {
    static constexpr bool kBf16X = MidX<TX>::kParts == 1, kI8 = sizeof(TW) == 1;
    static constexpr int kFlush = kBf16X && kI8 && KG <= 2 ? 4 : 0;
    static constexpr int kSets = !kBf16X || !kShort || kFlush || KG == 1 ? 1 : (KG == 2 && RT * MT <= 4) || (KG == 4 && MT == 2) ? 4 : 2;
};

template <typename TW, typename TX, int RT, int MT, int NWN, int KG, int PD, bool kShort>
__global__ void __launch_bounds__(64 * NWN * KG) gemm_mid_kernel(const MidArgs ga) {
    using Sums = MidSums<TW, TX, RT, MT, KG, kShort>;
    constexpr int kSets = Sums::kSets, kFlush = Sums::kFlush;
    static_assert(kFlush % PD == 0 && kSets <= 2 * PD, "sums are flushed between rounds of PD steps");
    constexpr int BM = 16 * MT, BN = 16 * RT * NWN, TPG = 64 * NWN, SL = BM * 8 / TPG;
    static_assert(SL >= 1 && SL * TPG == BM * 8, "the X stage must split evenly over the group's threads");
    constexpr int kPart = BM * MKS * 2;                       // bytes of one part (hi or lo) of an X stage
    constexpr int kStage = kPart * MidX<TX>::kParts;
    constexpr int kRed = KG > 1 ? (KG - 1) * NWN * RT * MT * 1024 : 0;
    constexpr int kLds = 2 * KG * kStage > kRed ? 2 * KG * kStage : kRed;
    __shared__ __attribute__((aligned(1024))) unsigned char lds[kLds];

    // XCD x runs the logical tiles [x n / 8, (x + 1) n / 8), M tiles fastest: the workgroups that
    // share W rows run on one XCD and read them through its L2
    const int li = (blockIdx.x % 8) * ga.per_xcd + blockIdx.x / 8;
    if (li >= ga.ntiles) return;
    const int m0 = (li % ga.tiles_m) * BM, tn = li / ga.tiles_m;
    int si = 0;
#pragma unroll
    for (int i = 1; i < MID_SEG; i++)
        if (i < ga.nseg && tn >= ga.seg[i].t0) si = i;
    const MidSeg sg = ga.seg[si];
    const int n0 = (tn - sg.t0) * BN;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
    const int kg = wave / NWN, wn = wave % NWN, r16 = lane % 16, g = lane / 16, tg = tid - kg * TPG;
    const int M = ga.M, N = sg.N, K = ga.K;

    const __amdgpu_buffer_rsrc_t wrs =
        __builtin_amdgcn_make_buffer_rsrc((void*)sg.W, (short)0, (int)((long long)N * K * sizeof(TW)), kMidBufWord3);
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)ga.X, (short)0, (int)(((long long)(M - 1) * ga.ldx + K) * sizeof(TX)), kMidBufWord3);
    int wbase[RT];
#pragma unroll
    for (int rt = 0; rt < RT; rt++) wbase[rt] = min(n0 + 16 * (RT * wn + rt) + r16, N - 1) * K;
    int xbase[SL], xdst[SL];
#pragma unroll
    for (int i = 0; i < SL; i++) {
        const int q = tg + TPG * i, row = q / 8, s = q % 8;
        xbase[i] = min(m0 + row, M - 1) * ga.ldx + 8 * s;
        xdst[i] = row * 128 + ((s ^ ((row >> 1) & 7)) * 16);
    }
    unsigned char* const buf = lds + kg * 2 * kStage;
    const int xs8 = 8 * (tg % 8);  // this thread's k offset inside a step

    MidX<TX> xr[PD][SL];
    MidW<TW> wr[PD][RT];
    // steps past K load zeros (both operands), so every K group runs the same number of steps
    auto load_x = [&](int set, int t) {
        const int k0 = (kg + KG * t) * MKS;
        const bool ok = k0 + xs8 < K;
#pragma unroll
        for (int i = 0; i < SL; i++) xr[set][i].load(xrs, ok ? (uint32_t)(xbase[i] + k0) * (uint32_t)sizeof(TX) : kMidOob);
    };
    auto load_w = [&](int slot, int t) {
#pragma unroll
        for (int rt = 0; rt < RT; rt++) wr[slot][rt].load(wrs, wbase[rt], (kg + KG * t) * MKS, g, K);
    };
    auto store_x = [&](int set, int t) {
#pragma unroll
        for (int i = 0; i < SL; i++) xr[set][i].store(buf + (t & 1) * kStage + xdst[i], kPart);
    };

    f32x4 part[kSets][RT][MT], acc[RT][MT];
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
#pragma unroll
            for (int u = 0; u < kSets; u++) part[u][rt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
            acc[rt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
        }

    // the row scales of the lane's 4 RT outputs, requested before the stream
    const bool fin = kg == 0;
    uint16_t sraw[RT][4];
    if (fin && sg.scale) {
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
#pragma unroll
            for (int j = 0; j < 4; j++) sraw[rt][j] = sg.scale[min(n0 + 16 * (RT * wn + rt) + 4 * g + j, N - 1)];
    }

    const int nt = (K + MKS * KG - 1) / (MKS * KG);
    load_x(0, 0);
#pragma unroll
    for (int d = 0; d < PD; d++) load_w(d, d);
    store_x(0, 0);
#pragma unroll
    for (int d = 0; d < PD; d++) load_x(d, 1 + d);
    lds_barrier();
    // step t (slot = t % PD): X of step t + 1 goes from registers to LDS and its registers take
    // step t + 1 + PD; the products of step t; W registers refilled with step t + PD
    auto step = [&](int t, int slot) {
        store_x(slot, t + 1);
        load_x(slot, t + 1 + PD);
        const unsigned char* cur = buf + (slot & 1) * kStage;  // PD is even: slot and t agree
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
            f32x4(&sum)[RT][MT] = part[(2 * slot + ks) % kSets];
            bf16x8 a[RT];
#pragma unroll
            for (int rt = 0; rt < RT; rt++) a[rt] = wr[slot][rt].frag(ks);
            if (ks == 1) load_w(slot, t + PD);
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                const int row = 16 * mt + r16;
                const unsigned char* p = cur + row * 128 + ((MidW<TW>::slot(ks, g) ^ ((row >> 1) & 7)) * 16);
                const bf16x8 bh = *(const bf16x8*)p;
#pragma unroll
                for (int rt = 0; rt < RT; rt++)
                    sum[rt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[rt], bh, sum[rt][mt], 0, 0, 0);
                if constexpr (MidX<TX>::kParts == 2) {
                    const bf16x8 bl = *(const bf16x8*)(p + kPart);
#pragma unroll
                    for (int rt = 0; rt < RT; rt++)
                        sum[rt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[rt], bl, sum[rt][mt], 0, 0, 0);
                }
            }
        }
        lds_barrier();
    };
    // Rounds of PD steps; steps past K are products of zeros. A step of 4 and 8 K groups is 256 and 512 k, so there
    // an odd one out has its own code (1536 = 3 steps of 8 groups: 33 rows of 5120 x 1536 int8 12.4 -> 10.7 us);
    // in the forms of fewer groups that copy costs more than the step (555 x 4096 x 2048 bf16 32.5, 33.3 with it)
    constexpr bool kTail = KG >= 4;
    static_assert(PD == 2, "the step left over is slot 0's");
    int t = 0;
    for (; t + (kTail ? PD : 1) <= nt; t += PD) {
#pragma unroll
        for (int d = 0; d < PD; d++) step(t + d, d);
        if constexpr (kFlush > 0) {
            if ((t + PD) % kFlush == 0) {
#pragma unroll
                for (int rt = 0; rt < RT; rt++)
#pragma unroll
                    for (int mt = 0; mt < MT; mt++) {
                        acc[rt][mt] += part[0][rt][mt];
                        part[0][rt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
                    }
            }
        }
    }
    if constexpr (kTail) {
        if (t < nt) step(t, 0);
    }
#pragma unroll
    for (int rt = 0; rt < RT; rt++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            if constexpr (kSets == 4) acc[rt][mt] = (part[0][rt][mt] + part[1][rt][mt]) + (part[2][rt][mt] + part[3][rt][mt]);
            else if constexpr (kSets == 2) acc[rt][mt] = part[0][rt][mt] + part[1][rt][mt];
            else if constexpr (kFlush > 0) acc[rt][mt] += part[0][rt][mt];
            else acc[rt][mt] = part[0][rt][mt];
        }

    if constexpr (KG > 1) {
        // the K groups' partial tiles, added in group order
        f32x4* red = (f32x4*)lds;
        if (kg > 0) {
#pragma unroll
            for (int rt = 0; rt < RT; rt++)
#pragma unroll
                for (int mt = 0; mt < MT; mt++)
                    red[((((kg - 1) * NWN + wn) * RT + rt) * MT + mt) * WAVE + lane] = acc[rt][mt];
        }
        lds_barrier();
        if (!fin) return;
#pragma unroll
        for (int q = 0; q < KG - 1; q++)
#pragma unroll
            for (int rt = 0; rt < RT; rt++)
#pragma unroll
                for (int mt = 0; mt < MT; mt++) acc[rt][mt] += red[(((q * NWN + wn) * RT + rt) * MT + mt) * WAVE + lane];
    }
    const bool vec = (sg.ldy % 4) == 0 && ((uintptr_t)sg.Y % 16) == 0;
#pragma unroll
    for (int rt = 0; rt < RT; rt++) {
        const int n = n0 + 16 * (RT * wn + rt) + 4 * g;
        float sc[4];
#pragma unroll
        for (int j = 0; j < 4; j++) sc[j] = sg.scale ? bf2f(sraw[rt][j]) : 1.f;
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            const int m = m0 + 16 * mt + r16;
            if (m >= M) continue;
            float* y = sg.Y + (size_t)m * sg.ldy + n;
            if (vec && n + 3 < N) {
                f32x4 v = acc[rt][mt];
#pragma unroll
                for (int j = 0; j < 4; j++) v[j] *= sc[j];
                if (ga.accumulate) v += *(const f32x4*)y;
                *(f32x4*)y = v;
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if (n + j < N) y[j] = (ga.accumulate ? y[j] : 0.f) + acc[rt][mt][j] * sc[j];
            }
        }
    }
}

// One form of the kernel and its cost: us of one 64-k step of a round of workgroups (one per CU; `base`: the
// part that does not grow with the rounds, for the form without K groups, whose workgroups share a CU), the fastest
// estimate base + ceil(tiles / 256) x cost is taken. Bf16 X: the median over a sweep of M 20 .. 1500 and N x K 512 ..
// 8192 x 2048 and 2048 x 4096. fp32 X: fitted to 236 sizes of M 17 .. 2048, N x K 512 .. 12352 x 256 .. 8192
// (int8 and bf16 W alike), where the choice is 1.5% above the fastest form on average (2.8% with a first fit to few
// rounds, which sent 2048 x 5120 x 1536 int8 to the form without K groups: 110 us, 256 x 256 tiles 97, here 80) and 16
// sizes are more than 5% above it, bf16 W with 420 to 1500 rows mostly (at most 1.38).
struct MidForm {
    int rt, mt, nwn, kg;
    float cost, base = 0.f;
};
// fp32 X: staging and splitting X is the larger part of a step
constexpr MidForm kFormsF32[] = {{1, 2, 1, 8, 0.156f}, {1, 2, 2, 8, 0.18f}, {2, 2, 2, 8, 0.265f}, {2, 2, 4, 4, 0.42f},
                                 {2, 2, 4, 1, 0.33f, 0.15f}, {2, 4, 4, 2, 0.70f}, {2, 4, 8, 1, 1.15f}, {4, 4, 8, 1, 1.80f}};
constexpr MidForm kFormsBf16[] = {{1, 2, 1, 8, 0.100f}, {1, 2, 2, 4, 0.157f}, {1, 4, 2, 4, 0.205f}, {1, 4, 4, 2, 0.312f},
                                  {2, 4, 4, 2, 0.548f}, {2, 8, 4, 1, 0.90f},  {2, 8, 8, 1, 1.21f}};
// (bf16 X, the second form: 8 K groups for int8 W. bf16 W is fuller with 4 of them, whose workgroups take half the
// threads: 17 x 8192 x 2048 12.1 -> 10.8 us (row-tile kernel 11.4), 100 x 2048 x 2048 9.4 -> 9.0; int8 150 x 1024 x 8192 15.5 -> 18.0)
constexpr int kNF32 = 8, kNBf16 = 7, kForms = 8;  // entries of the two tables; codes of the sized forms
// 16 rows of X a tile, after the sized forms: up to 16 rows chosen by rows of W and K, see small_form; past
// them where all tiles run in one round, see one_round_form
constexpr MidForm kFormsSmall[] = {{1, 1, 1, 8, 0.f}, {1, 1, 1, 4, 0.f}, {1, 1, 2, 4, 0.f}, {2, 1, 2, 4, 0.f}};

// Measured (us, 16 rows, weights from HBM; fp32 X with int8 W, then bf16 both), row-tile kernel -> here:
//   8192 x 2048 9.5 -> 7.6, 10.1 -> 8.8    4096 x 2048 8.4 -> 7.0, 7.0 -> 6.1
//   2048 x 4096 13.4 -> 9.3, 10.3 -> 7.9   512 x 2048 8.0 -> 5.5, 6.1 -> 4.9
// 4 K groups instead of 8 where K is short and past 4096 rows of W, where tiles of 16 of them open a second
// round: for fp32 X, whose stage costs most, with tiles of 32 (3 rows of 5120 x 1536: int8, fp32 X 9.0 -> 6.6, bf16
// both 8.2 -> 7.3; row-tile kernel 8.7, 7.3). Tiles of 32 and 64 rows where even these are more than two
// workgroups per CU (bf16 W, fp32 X 32768 x 2048: 36.2 -> 33.0).
// K is short up to 1280: 5 steps of 4 K groups against 3 of 8 (us, 8 and 4 groups, 16 x 1000 x 1040 bf16 W, fp32 X 5.4, 5.1,
// bf16 both 4.4, 4.2; 3 x 2048 x 1024 5.3, 5.4; 16 x 1024 x 1536 5.4, 5.7)
constexpr int kShortK = 1280;
int small_form(bool f32, long long rows, int K) {
    if (rows > 16384) return kForms + 3;
    if (f32 ? rows > 4096 : rows > 8192) return kForms + 2;
    if (K <= kShortK || rows > 4096) return kForms + 1;
    return kForms;
}
// the 256 x 256 tiles of gemm.hip, in the same unit: int8 W with fp32 X, bf16 W with bf16 X
constexpr float kTile256F32 = 3.7f, kTile256Bf16 = 1.5f;

long long mid_tiles(const MidForm& f, const MidArgs& ga) {
    long long t = 0;
    for (int i = 0; i < ga.nseg; i++) t += (ga.seg[i].N + 16 * f.rt * f.nwn - 1) / (16 * f.rt * f.nwn);
    return t * ((ga.M + 16 * f.mt - 1) / (16 * f.mt));
}

// The 16-row form for more than 16 rows of X, or -1. A workgroup of 32 and more rows stages that much X before
// its first product and takes most of a CU's LDS; where the chip runs all tiles of 16 rows in one round, they are
// done sooner, and short rows of K were slower on the larger tiles than on the row-tile kernel before those.
// Measured (us; row-tile kernel, sized form, here):
//   int8 W, fp32 X   17 x 2048 x 512 4.8, 6.3, 4.2   64 x 2048 x 512 5.6, 6.4, 4.4   17 x 1000 x 1040 5.5, 7.9, 5.3
//   bf16 W, bf16 X   17 x 2048 x 512 4.4, 5.0, 3.6   17 x 1000 x 1040 4.4, 6.1, 4.5   17 x 1024 x 8192 -, 15.0, 12.5
// Over 968 sizes this form took 0.84 of the sized one's time on average, 1.08 at most. The limits on K: past them 4
// K groups walk too long (bf16 X 33 x 2048 x 4096 10.1 sized, 12.2 here; bf16 W, fp32 X 100 x 1536 x 6144 23.6, 27.4).
int one_round_form(bool f32, const MidArgs& ga) {
    auto one_round = [&](int i) { return mid_tiles(kFormsSmall[i], ga) <= 256; };
    if (one_round(0)) return kForms + (ga.K <= kShortK ? 1 : 0);
    if ((f32 || ga.K < 1024) && one_round(2)) return kForms + 2;
    if (f32 && ga.K <= 1024 && one_round(3)) return kForms + 3;
    return -1;
}

template <typename TW, typename TX, int RT, int MT, int NWN, int KG, int PD>
int launch_mid(MidArgs ga, hipStream_t st) {
    constexpr int BM = 16 * MT, BN = 16 * RT * NWN;
    ga.tiles_m = (ga.M + BM - 1) / BM;
    int t = 0;
    for (int i = 0; i < ga.nseg; i++) {
        ga.seg[i].t0 = t;
        t += (ga.seg[i].N + BN - 1) / BN;
    }
    ga.ntiles = ga.tiles_m * t;
    ga.per_xcd = (ga.ntiles + 7) / 8;
    // (one instance where both would be the same)
    constexpr bool both = MidSums<TW, TX, RT, MT, KG, true>::kSets > 1 && sizeof(TW) == 2 && MT > 1 && !(KG == 4 && MT == 2);
    if (both && ga.M > 64)
        gemm_mid_kernel<TW, TX, RT, MT, NWN, KG, PD, !both><<<8 * ga.per_xcd, 64 * NWN * KG, 0, st>>>(ga);
    else
        gemm_mid_kernel<TW, TX, RT, MT, NWN, KG, PD, true><<<8 * ga.per_xcd, 64 * NWN * KG, 0, st>>>(ga);
    return after_launch("gemm_mid");
}

template <typename TW, typename TX>
int run_mid(int form, const MidArgs& ga, hipStream_t st) {
    constexpr bool f32 = std::is_same<TX, float>::value;
#define AEG_MID(I)                                                                                              \
    case I: {                                                                                                   \
        constexpr MidForm f = f32 ? kFormsF32[I] : kFormsBf16[I < kNBf16 ? I : 0];                              \
        constexpr int kg = !f32 && I == 1 && sizeof(TW) == 1 ? 8 : f.kg;                                        \
        return launch_mid<TW, TX, f.rt, f.mt, f.nwn, kg, 2>(ga, st);                                            \
    }
#define AEG_MID_SMALL(I)                                                                                        \
    case kForms + I: return launch_mid<TW, TX, kFormsSmall[I].rt, 1, kFormsSmall[I].nwn, kFormsSmall[I].kg, 2>(ga, st);
    switch (form) {
        AEG_MID_SMALL(0) AEG_MID_SMALL(1) AEG_MID_SMALL(2) AEG_MID_SMALL(3)
        AEG_MID(0) AEG_MID(1) AEG_MID(2) AEG_MID(3) AEG_MID(4) AEG_MID(5) AEG_MID(6) AEG_MID(7)
    }
#undef AEG_MID
#undef AEG_MID_SMALL
    return fail(AEGIST_ERR_SHAPE, "gemm_mid: no such form");
}

}  // namespace

namespace aegist {

// The form this file's kernel would take the product in, or -1 if the 256 x 256 tiles of gemm.hip are
// estimated faster (`tile256`: they could take it; `stacked`: as one launch of all weights, else one after the
// other, each in rounds of its own: bf16 8192, 4096, 32 and 32 rows x 2048 at 1024 rows of X take
// 176 us that way and 85 here). Every operand is below 2^31 - 16 bytes (the caller splits larger ones),
// K % 16 == 0, rows 16-byte aligned.
int gemm_mid_form(int x_dtype, int nseg, const int* N, int M, int K, bool tile256, bool stacked) {
    if (M <= 16) {
        long long rows = 0;
        for (int i = 0; i < nseg; i++) rows += N[i];
        return small_form(x_dtype == AEGIST_F32, rows, K);
    }
    MidArgs ga{};
    ga.nseg = nseg;
    ga.M = M;
    ga.K = K;
    const long long tm = (M + 255) / 256;
    auto rounds256 = [&](long long n) { return ((n + 255) / 256 * tm + 255) / 256; };
    long long rows = 0, r256 = 0;
    for (int i = 0; i < nseg; i++) {
        ga.seg[i].N = N[i];
        rows += N[i];
        r256 += rounds256(N[i]);
    }
    const int one = one_round_form(x_dtype == AEGIST_F32, ga);
    if (one >= 0) return one;
    if (stacked) r256 = rounds256(rows);
    const MidForm* forms = x_dtype == AEGIST_F32 ? kFormsF32 : kFormsBf16;
    int best = -1;
    float least = tile256 ? r256 * (x_dtype == AEGIST_F32 ? kTile256F32 : kTile256Bf16) : 3.4e38f;
    for (int i = 0; i < (x_dtype == AEGIST_F32 ? kNF32 : kNBf16); i++) {
        const long long t = mid_tiles(forms[i], ga);
        const float est = forms[i].base + ((t + 255) / 256) * forms[i].cost;
        if (est <= least) {
            least = est;
            best = i;
        }
    }
    return best;
}

int launch_gemm_mid(int form, const void* X, int x_dtype, long long ldx, int w_dtype, int nseg, const void* const* W,
                    const uint16_t* const* scale, float* const* Y, const long long* ldy, const int* N, int M, int K,
                    int accumulate, hipStream_t st) {
    if (nseg < 1 || nseg > MID_SEG || form < 0) return fail(AEGIST_ERR_SHAPE, "gemm_mid: 1 to 4 weights per launch");
    MidArgs ga{};
    ga.X = X;
    ga.nseg = nseg;
    ga.ldx = (int)ldx;
    ga.M = M;
    ga.K = K;
    ga.accumulate = accumulate;
    for (int i = 0; i < nseg; i++) ga.seg[i] = MidSeg{W[i], scale[i], Y[i], ldy[i], N[i], 0};
    if (w_dtype == AEGIST_I8)
        return x_dtype == AEGIST_F32 ? run_mid<int8_t, float>(form, ga, st) : run_mid<int8_t, uint16_t>(form, ga, st);
    return x_dtype == AEGIST_F32 ? run_mid<uint16_t, float>(form, ga, st) : run_mid<uint16_t, uint16_t>(form, ga, st);
}

}  // namespace aegist
