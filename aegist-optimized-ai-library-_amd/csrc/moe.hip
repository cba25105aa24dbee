// Mixture-of-experts block for gfx950: router top-k, device-side grouping of the picks by
// expert, and the 4-bit SwiGLU experts on MFMA.
//
// Semantics (aegist/hybrid.py):
//   route        MoE.route :637-641          logits = h W_r^T; p = softmax(logits) in fp32; the K
//                                             largest (ties to the lower expert, hybrid.cu:35);
//                                             weights p / sum(top p)
//   experts      ExpertBank.forward :608-628 per pick: y = W_dn (silu(W_g h) * (W_u h)) * weight
//   dequantise   q4_dequantize :463-469       w = code * scale + min per 64-value group, codes
//                                             packed two per byte, even index in the low nibble
//   layout       expert_layout :472-482       [gu_q 2I x D/2 | gu_s 2I x D/64 f16 | gu_m | dn_q
//                                             D x I/2 | dn_s D x I/64 f16 | dn_m]
//   combine      MoE.forward :647-652         x += sum_k y_k + sigmoid(h . w_sg) * shared(h)
// Engine counterparts: router_topk hybrid.cu:317-362, moe_gu_* / moe_dn_* :386-558,
// moe_reduce :560-567, shared_gate_add :569-577; the host grouping of hybrid.rs:875-913 runs on
// the device here (no host sync per layer).
//
// Expert products on MFMA, exactly in the reference's fp32 sense: a 4-bit code c becomes the
// bf16 bit pattern 0x4300 | c = 128 + c (exact), the activations enter as bf16 hi + lo (~16
// significant bits), and per 64-value group the fp32 result is
//   y += s * (sum (128 + c)(x_hi + x_lo)) + (m - 128 s) * sum (x_hi + x_lo),
// i.e. s * sum c x + m * sum x with the scale and min applied per group in fp32.
// A dword of 8 codes (code j in bits 4j) yields the bf16 pairs (c0,c4) (c1,c5) (c2,c6)
// (c3,c7) with one and-or each, so the activations are stored in the same order within every
// 8-value chunk: x'[8q + 2j] = x[8q + j], x'[8q + 2j + 1] = x[8q + j + 4].
#include "common.h"
#include "moe_tiles.h"

#include <algorithm>
#include <type_traits>

namespace aegist {
int launch_proj(const void* X, int x_dtype, long long ldx, const void* W, int w_dtype, const uint16_t* scale, float* Y,
                long long ldy, int M, int N, int K, int accumulate, hipStream_t st);
bool moe_decode_fits(int T, int D, int I, int E, int K);
int launch_moe_decode(const float* h, const unsigned long long* eptr, const int* idx, const float* wts, int T, int D,
                      int I, int E, int K, long long gu_s, long long gu_m, long long dn_q, long long dn_s,
                      long long dn_m, float* act, float* ypick, hipStream_t st);
}  // namespace aegist

using namespace aegist;

namespace {

constexpr int PB = 32;            // picks per expert tile (two 16-column MFMA tiles)
constexpr int PBB = 64;           // picks per big (prefill) tile: four 16-column MFMA tiles
constexpr int RB = 64;            // output rows per workgroup (4 waves x 16)
constexpr int MAX_E = 1024;       // experts per layer the grouping kernel handles

struct MoeTile {                  // one block of <= PB grouped picks of one expert
    unsigned long long base;      // the expert's row address (resolved from the pointer table)
    int p0, p1;                   // grouped positions [p0, p1)
};

struct ExpertOffsets {            // byte offsets inside one expert row (expert_layout)
    long long gu_s, gu_m, dn_q, dn_s, dn_m;
};
static ExpertOffsets expert_offsets(int D, int I) {
    ExpertOffsets o;
    o.gu_s = (long long)2 * I * (D / 2);
    o.gu_m = o.gu_s + (long long)2 * I * (D / 64) * 2;
    o.dn_q = o.gu_m + (long long)2 * I * (D / 64) * 2;
    o.dn_s = o.dn_q + (long long)D * (I / 2);
    o.dn_m = o.dn_s + (long long)D * (I / 64) * 2;
    return o;
}

__device__ __forceinline__ float h2f(uint16_t h) { return (float)__builtin_bit_cast(_Float16, h); }

// Loads through expert-row addresses taken from the pointer table: the compiler cannot tell
// those are global memory and would emit flat loads, which also count against the LDS wait
// counter (every LDS wait would then drain the prefetched code stream). Global address space.
template <typename T>
__device__ __forceinline__ T ld_global(const void* p) {
    return *(const __attribute__((address_space(1))) T*)p;
}

// Maximum over the wave by DPP moves (row shifts, then row broadcasts) instead of LDS permutes, whose
// round trips made up most of the router's rounds; the total is the last lane's. No NaN inputs.
__device__ __forceinline__ float wave_max_dpp(float v) {
    auto step = [](float x, auto ctrl, auto rows) {
        return fmaxf(x, __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(x), __float_as_int(x),
                                                                   decltype(ctrl)::value, decltype(rows)::value, 0xF, false)));
    };
    using std::integral_constant;
    v = step(v, integral_constant<int, 0x111>{}, integral_constant<int, 0xF>{});  // row_shr:1
    v = step(v, integral_constant<int, 0x112>{}, integral_constant<int, 0xF>{});
    v = step(v, integral_constant<int, 0x114>{}, integral_constant<int, 0xF>{});
    v = step(v, integral_constant<int, 0x118>{}, integral_constant<int, 0xF>{});
    v = step(v, integral_constant<int, 0x142>{}, integral_constant<int, 0xA>{});  // row_bcast:15 to rows 1, 3
    v = step(v, integral_constant<int, 0x143>{}, integral_constant<int, 0xC>{});  // row_bcast:31 to rows 2, 3
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), WAVE - 1));
}

// The least value of the wave, in the same way.
__device__ __forceinline__ int wave_min_dpp(int v) {
    auto step = [](int x, auto ctrl, auto rows) {
        return min(x, __builtin_amdgcn_update_dpp(x, x, decltype(ctrl)::value, decltype(rows)::value, 0xF, false));
    };
    using std::integral_constant;
    v = step(v, integral_constant<int, 0x111>{}, integral_constant<int, 0xF>{});
    v = step(v, integral_constant<int, 0x112>{}, integral_constant<int, 0xF>{});
    v = step(v, integral_constant<int, 0x114>{}, integral_constant<int, 0xF>{});
    v = step(v, integral_constant<int, 0x118>{}, integral_constant<int, 0xF>{});
    v = step(v, integral_constant<int, 0x142>{}, integral_constant<int, 0xA>{});
    v = step(v, integral_constant<int, 0x143>{}, integral_constant<int, 0xC>{});
    return __builtin_amdgcn_readlane(v, WAVE - 1);
}

// ---------------------------------------------------------------------------------------------
// Router top-K over precomputed logits [T, E] (the projection kernel computes h W^T): one wave
// per token, lane holds the probabilities of experts lane + 64 i in registers; softmax in fp32;
// K rounds of a wave argmax that prefers the lower expert on equal probabilities.
template <int NPER>  // experts per lane held in registers (E <= 64 NPER)
__global__ void __launch_bounds__(256) router_topk_kernel(const float* __restrict__ logits, int* __restrict__ idx,
                                                          float* __restrict__ wts, int T, int E, int K) {
    const int lane = threadIdx.x % WAVE, t = blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE;
    if (t >= T) return;
    const float* l = logits + (size_t)t * E;
    float p[NPER];
    float m = -INFINITY;
#pragma unroll
    for (int i = 0; i < NPER; i++) {
        const int e = lane + WAVE * i;
        p[i] = e < E ? l[e] : -INFINITY;
        m = fmaxf(m, p[i]);
    }
    m = wave_max(m);
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < NPER; i++) {
        p[i] = lane + WAVE * i < E ? expf(p[i] - m) : 0.f;
        s += p[i];
    }
    s = wave_sum(s);
#pragma unroll
    for (int i = 0; i < NPER; i++) p[i] = lane + WAVE * i < E ? p[i] / s : -1.f;  // -1: not an expert
    float sel = 0.f;  // sum of the picked probabilities
    float myv = 0.f;  // lane k keeps pick k
    int mye = 0;
    for (int k = 0; k < K; k++) {
        // the largest probability of the wave, then the lowest expert that has it (experts lane + 64 i);
        // NaN and taken entries never compare greater
        float lv = -1.f;
        int li = 0x7fffffff, bi = 0x7fffffff;  // the lane's first holder of its largest
#pragma unroll
        for (int i = 0; i < NPER; i++) {
            if (NPER > 4 && p[i] > lv) li = lane + WAVE * i;
            lv = p[i] > lv ? p[i] : lv;
        }
        const float bv = wave_max_dpp(lv);
        if constexpr (NPER > 4) {
            bi = wave_min_dpp(lv == bv && bv > -1.f ? li : 0x7fffffff);
        } else if (bv > -1.f) {
            // few registers: the first i with a holder, its lowest lane
#pragma unroll
            for (int i = 0; i < NPER; i++) {
                const unsigned long long m = __ballot(p[i] == bv);
                if (m != 0 && bi == 0x7fffffff) bi = WAVE * i + __builtin_ctzll(m);
            }
        }
#pragma unroll
        for (int i = 0; i < NPER; i++)
            if (bi == lane + WAVE * i) p[i] = -2.f;  // taken
        if (lane == k) {
            myv = bv;
            mye = bi;
        }
        sel += bv;
    }
    if (lane < K) {
        idx[(size_t)t * K + lane] = mye;
        wts[(size_t)t * K + lane] = myv / sel;
    }
}

// ---------------------------------------------------------------------------------------------
// Grouping: picks i = t K + k with expert idx[i]; out of range experts are dropped. ptok / psrc: token and
// pick index of each grouped position. Two launches, each over blocks of `per` picks: moe_count_kernel counts the block's picks per
// expert in LDS (its other workgroups split the activations), moe_place_kernel adds the blocks'
// counts up, scans them over the experts and places its block's picks. (One workgroup doing all of it
// took 32 us for 16384 picks, twice through LDS atomics; 8 us each in blocks of 1024, the activation
// split's 8 us included.)
// An expert's positions are cut into tiles: with a `cap` all into ceil(c / cap) balanced ones (tiles3,
// meta[2] of them), else into blocks of 17..32 (tiles2, meta[1]) and a last one of <= 16 (tiles1,
// meta[0]). The order of positions inside an expert is unspecified (atomics);
// no result depends on it (every pick's sums run in the same order whatever tile it lands in with whom).
__device__ __forceinline__ int block_excl_scan(int v, int* wsum, int* total) {
    const int lane = threadIdx.x % WAVE, w = threadIdx.x / WAVE, nw = blockDim.x / WAVE;
    int x = v;
#pragma unroll
    for (int d = 1; d < WAVE; d <<= 1) {
        const int y = __shfl_up(x, d, WAVE);
        if (lane >= d) x += y;
    }
    if (lane == WAVE - 1) wsum[w] = x;
    __syncthreads();
    int off = 0, tot = 0;
    for (int i = 0; i < nw; i++) {
        if (i < w) off += wsum[i];
        tot += wsum[i];
    }
    __syncthreads();
    *total = tot;
    return off + x - v;
}

__device__ __forceinline__ void xprep_chunk(long long q, long long nq, const float* __restrict__ h,
                                            uint16_t* __restrict__ xh, uint16_t* __restrict__ xl, float* __restrict__ xs);

__global__ void __launch_bounds__(256) moe_count_kernel(const int* __restrict__ idx, int N, int E, int per, int nb,
                                                        int* __restrict__ cnt, const float* __restrict__ h, int T, int D,
                                                        uint16_t* __restrict__ xh, uint16_t* __restrict__ xl,
                                                        float* __restrict__ xs) {
    __shared__ int c[MAX_E];
    const int b = blockIdx.x;
    if (b >= nb) {
        xprep_chunk((long long)(b - nb) * blockDim.x + threadIdx.x, (long long)T * (D / 8), h, xh, xl, xs);
        return;
    }
    for (int e = threadIdx.x; e < E; e += blockDim.x) c[e] = 0;
    __syncthreads();
    for (int i = b * per + threadIdx.x; i < min(N, (b + 1) * per); i += blockDim.x) {
        const int e = idx[i];
        if (e >= 0 && e < E) atomicAdd(&c[e], 1);
    }
    __syncthreads();
    for (int e = threadIdx.x; e < E; e += blockDim.x) cnt[(size_t)b * E + e] = c[e];
}

__global__ void __launch_bounds__(1024) moe_place_kernel(const int* __restrict__ idx, int N, int K, int E, int per, int nb,
                                                         const int* __restrict__ cnt,
                                                         const unsigned long long* __restrict__ eptr,
                                                         int* __restrict__ ptok, int* __restrict__ psrc,
                                                         MoeTile* __restrict__ tiles1, MoeTile* __restrict__ tiles2,
                                                         MoeTile* __restrict__ tiles3, int cap,
                                                         int* __restrict__ meta) {
    __shared__ int cur[MAX_E], wsum[16];
    const int tid = threadIdx.x, b = blockIdx.x;
    int c = 0, mine = 0;  // the expert's picks; those of the blocks before this one
    if (tid < E) {
#pragma unroll 8
        for (int k = 0; k < nb; k++) {
            const int v = cnt[(size_t)k * E + tid];
            mine += k < b ? v : 0;
            c += v;
        }
    }
    int total;
    const int off = block_excl_scan(c, wsum, &total);
    if (tid < E) cur[tid] = off + mine;
    if (b == 0) {
        const int n3 = cap ? (c + cap - 1) / cap : 0;
        const int c3 = n3 > 0 ? c : 0, cr = c - c3, rem = cr % PB;
        const int small = rem > 0 && rem <= 16 ? 1 : 0;      // the last block, if it is small
        const int big = cr / PB + (rem > 16 ? 1 : 0);        // full blocks and a large last block
        int tot_1, tot_2, tot_3;
        const int off1 = block_excl_scan(small, wsum, &tot_1);
        const int off2 = block_excl_scan(big, wsum, &tot_2);
        const int off3 = block_excl_scan(n3, wsum, &tot_3);
        if (tid < E) {
            const unsigned long long base = c > 0 ? eptr[tid] : 0ull;
            for (int j = 0; j < n3; j++)
                tiles3[off3 + j] = MoeTile{base, off + tile_begin(c3, j, n3), off + tile_begin(c3, j + 1, n3)};
            for (int j = 0; j < big; j++)
                tiles2[off2 + j] = MoeTile{base, off + c3 + j * PB, off + c3 + min(cr, (j + 1) * PB)};
            if (small) tiles1[off1] = MoeTile{base, off + c - rem, off + c};
        }
        if (tid == 0) {
            meta[0] = tot_1;
            meta[1] = tot_2;
            meta[2] = tot_3;
        }
    }
    __syncthreads();
    for (int i = b * per + tid; i < min(N, (b + 1) * per); i += blockDim.x) {
        const int e = idx[i];
        if (e < 0 || e >= E) continue;
        const int pos = atomicAdd(&cur[e], 1);
        ptok[pos] = i / K;
        psrc[pos] = i;
    }
}

// ---------------------------------------------------------------------------------------------
// Activations for the expert products: xh / xl [rows][D] bf16 (hi truncated, lo = rounded
// remainder) in the chunk order above, xs [rows][D / 64] = sum over the group of (hi + lo).
// One thread per 8-value chunk; 8 threads of a 64-group reduce their sums by shuffles.
__device__ __forceinline__ void split8(const float* v, uint4& hi, uint4& lo, float& sum) {
    // element order within the chunk: v0 v4 v1 v5 v2 v6 v3 v7
    uint32_t H[4], L[4];
    sum = 0.f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const float a = v[j], b = v[j + 4];
        const uint32_t ua = __float_as_uint(a) & 0xffff0000u, ub = __float_as_uint(b) & 0xffff0000u;
        const float ra = a - __uint_as_float(ua), rb = b - __uint_as_float(ub);
        typedef float f2 __attribute__((ext_vector_type(2)));
        typedef __bf16 b2 __attribute__((ext_vector_type(2)));
        const uint32_t lp = __builtin_bit_cast(uint32_t, __builtin_convertvector((f2{ra, rb}), b2));
        H[j] = (ua >> 16) | ub;
        L[j] = lp;
        sum += (__uint_as_float(ua) + bf_lo(lp)) + (__uint_as_float(ub) + bf_hi(lp));
    }
    hi = uint4{H[0], H[1], H[2], H[3]};
    lo = uint4{L[0], L[1], L[2], L[3]};
}

__device__ __forceinline__ void xprep_chunk(long long q, long long nq, const float* __restrict__ h,
                                            uint16_t* __restrict__ xh, uint16_t* __restrict__ xl, float* __restrict__ xs) {
    const bool ok = q < nq;
    const long long qq = ok ? q : nq - 1;
    const float* src = h + qq * 8;
    const float4 a = ((const float4*)src)[0], b = ((const float4*)src)[1];
    const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    uint4 hi, lo;
    float s;
    split8(v, hi, lo, s);
    s += __shfl_xor(s, 1, WAVE);
    s += __shfl_xor(s, 2, WAVE);
    s += __shfl_xor(s, 4, WAVE);
    if (!ok) return;
    ((uint4*)xh)[qq] = hi;
    ((uint4*)xl)[qq] = lo;
    if ((qq & 7) == 0) xs[qq / 8] = s;
}

// bf16 pairs (c_j, c_{j+4}) + 128 from a dword of 8 4-bit codes
__device__ __forceinline__ bf16x8 codes_bf16(uint32_t p) {
    const uint32_t d0 = (p & 0x000F000Fu) | 0x43004300u;
    const uint32_t d1 = ((p >> 4) & 0x000F000Fu) | 0x43004300u;
    const uint32_t d2 = ((p >> 8) & 0x000F000Fu) | 0x43004300u;
    const uint32_t d3 = ((p >> 12) & 0x000F000Fu) | 0x43004300u;
    typedef uint32_t u4v __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(bf16x8, (u4v{d0, d1, d2, d3}));
}
__device__ __forceinline__ bf16x8 ld_bf8(const uint16_t* p) { return *(const bf16x8*)p; }
__device__ __forceinline__ f32x4 mfma_bf(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// ---------------------------------------------------------------------------------------------
// One expert matrix block (NM = 1 or 2 matrices sharing the activations; RB = 64 rows each)
// times a tile of <= 16 NT picks. The 64-groups are split over the 4 waves (wave w takes
// groups w, w + 4, ...), so each activation fragment is read once per workgroup; every wave
// covers all 64 rows as 4 row tiles and the waves' partial sums are added in LDS afterwards.
// Lane (n, g) accumulates rows 16 rt + 4g + j (j < 4) for picks 16 t + n. Per 64-group a lane
// holds the 16 codes [64 grp + 16 g, +16) of its row (one 8-byte load): dword ks feeds the
// MFMA of step ks, so each MFMA's 32 codes (8 per lane group) lie in one group; the
// activations are read at the same k. Codes stream through a register ring (the HBM stream),
// activations through a 2-slot ring.
constexpr int RTL = RB / 16;  // row tiles per wave

template <int NM, int NT>
struct BlockAcc {
    f32x4 acc[NM][RTL][NT];
};

// `stage` fills sc and gs (LDS); it runs after this wave's first code and activation loads are
// issued, so its global round trip overlaps theirs, and is followed by the workgroup barrier.
template <int NM, int NT, typename Stage>
__device__ __forceinline__ void expert_block(const unsigned char* __restrict__ qbase, const long long* qrow0, int Kdim,
                                             const float2* sc, const uint16_t* __restrict__ xh,
                                             const uint16_t* __restrict__ xl, const long long* xrow, const float* gs,
                                             BlockAcc<NM, NT>& out, int ngroups, Stage stage) {
    // groups of codes in flight per lane (per row tile and matrix): two for decode-sized tiles,
    // where the weight stream is the whole cost; one for two pick tiles (register budget)
    constexpr int PD = NT == 1 ? 2 : 1;
    const int tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE, n = lane % 16, g = lane / 16;
#pragma unroll
    for (int m = 0; m < NM; m++)
#pragma unroll
        for (int rt = 0; rt < RTL; rt++)
#pragma unroll
            for (int t = 0; t < NT; t++) out.acc[m][rt][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int nmine = ngroups > wave ? (ngroups - wave + 3) / 4 : 0;  // this wave's groups
    if (nmine == 0) {
        stage();
        __syncthreads();
        return;
    }
    const size_t rowbytes = Kdim / 2;
    const unsigned char* arow[NM];
#pragma unroll
    for (int m = 0; m < NM; m++) arow[m] = qbase + (size_t)(qrow0[m] + n) * rowbytes + 8 * g;
    auto gaddr = [&](int i) { return 32 * (wave + 4 * min(i, nmine - 1)); };  // byte offset of my i-th group
    typedef uint32_t u2v __attribute__((ext_vector_type(2)));
    u2v ar[NM][RTL][PD];
#pragma unroll
    for (int u = 0; u < PD; u++)
#pragma unroll
        for (int m = 0; m < NM; m++)
#pragma unroll
            for (int rt = 0; rt < RTL; rt++) ar[m][rt][u] = ld_global<u2v>(arow[m] + 16 * rt * rowbytes + gaddr(u));
    constexpr int NB = NT == 1 ? 2 : 1;  // activation slots (prefetched a group ahead for one tile)
    bf16x8 bh[NB][NT][2], bl[NB][NT][2];  // [slot][tile][ks]
#define AEG_LOAD_B(slot, grp)                                                  \
    _Pragma("unroll") for (int t = 0; t < NT; t++)                             \
        _Pragma("unroll") for (int ks = 0; ks < 2; ks++) {                     \
            const long long k0 = xrow[t] + 64 * (grp) + 16 * g + 8 * ks;       \
            bh[slot][t][ks] = ld_bf8(xh + k0);                                 \
            bl[slot][t][ks] = ld_bf8(xl + k0);                                 \
        }
    AEG_LOAD_B(0, wave)
    stage();
    __syncthreads();
    for (int i0 = 0; i0 < nmine; i0 += PD) {
#pragma unroll
        for (int u = 0; u < PD; u++) {
            const int i = i0 + u;
            if (i >= nmine) break;
            const int grp = wave + 4 * i, slot = NB == 2 ? (u & 1) : 0;
            if constexpr (NB == 2) {
                if (i + 1 < nmine) {
                    AEG_LOAD_B((slot ^ 1), grp + 4)
                }
            } else if (i > 0) {
                AEG_LOAD_B(0, grp)
            }
            float X[NT];
#pragma unroll
            for (int t = 0; t < NT; t++) X[t] = gs[(16 * t + n) * ngroups + grp];
#pragma unroll
            for (int m = 0; m < NM; m++)
#pragma unroll
                for (int rt = 0; rt < RTL; rt++) {
                    const u2v a2 = ar[m][rt][u];
                    // refill this ring slot with my group PD ahead (clamped: static wait counts)
                    ar[m][rt][u] = ld_global<u2v>(arow[m] + 16 * rt * rowbytes + gaddr(i + PD));
                    f32x4 P[NT];
#pragma unroll
                    for (int t = 0; t < NT; t++) P[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int ks = 0; ks < 2; ks++) {
                        const bf16x8 a = codes_bf16(ks ? a2.y : a2.x);
#pragma unroll
                        for (int t = 0; t < NT; t++) {
                            P[t] = mfma_bf(a, bh[slot][t][ks], P[t]);
                            P[t] = mfma_bf(a, bl[slot][t][ks], P[t]);
                        }
                    }
                    // y += s P + (m - 128 s) X for this row tile's rows and every pick tile
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const float2 sm = sc[(m * RB + 16 * rt + 4 * g + j) * ngroups + grp];
#pragma unroll
                        for (int t = 0; t < NT; t++)
                            out.acc[m][rt][t][j] = fmaf(sm.x, P[t][j], fmaf(sm.y, X[t], out.acc[m][rt][t][j]));
                    }
                }
        }
    }
#undef AEG_LOAD_B
}

// Sum the 4 waves' partials of matrix m into red[pick][row] (row < RB), in wave order (the
// result does not depend on scheduling). red has PB rows of RB + 1 floats.
template <int NM, int NT>
__device__ __forceinline__ void reduce_waves(const BlockAcc<NM, NT>& a, int m, float (*red)[RB + 1]) {
    const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE, n = lane % 16, g = lane / 16;
    for (int w = 0; w < 4; w++) {
        if (wave == w) {
#pragma unroll
            for (int rt = 0; rt < RTL; rt++)
#pragma unroll
                for (int t = 0; t < NT; t++)
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        float& r = red[16 * t + n][16 * rt + 4 * g + j];
                        r = (w == 0 ? 0.f : r) + a.acc[m][rt][t][j];
                    }
        }
        __syncthreads();
    }
}

// Stage (s, m - 128 s) of rows [row0, row0 + RB) x groups [0, G) of one matrix into sc[RB][G]:
// the block's scale and min entries are one contiguous run of RB G halves each, read as 16-byte
// pieces (8 per load), all loads of a thread issued before any is used.
__device__ __forceinline__ void stage_scales(float2* sc, const uint16_t* __restrict__ s,
                                             const uint16_t* __restrict__ mn, long long row0, int G) {
    const uint16_t* s0 = s + (size_t)row0 * G;
    const uint16_t* m0 = mn + (size_t)row0 * G;
    const int n8 = RB * G / 8;  // 16-byte pieces (RB G is a multiple of 8: G = K / 64, RB = 64)
    constexpr int MAXP = RB * 64 / 8 / 256;  // pieces per thread at the largest G (64)
    typedef uint32_t u4v __attribute__((ext_vector_type(4)));
    u4v sv[MAXP], mv[MAXP];
#pragma unroll
    for (int u = 0; u < MAXP; u++) {
        const int i = threadIdx.x + 256 * u;
        if (i < n8) {
            sv[u] = ld_global<u4v>(s0 + 8 * i);
            mv[u] = ld_global<u4v>(m0 + 8 * i);
        }
    }
#pragma unroll
    for (int u = 0; u < MAXP; u++) {
        const int i = threadIdx.x + 256 * u;
        if (i < n8) {
            const uint32_t sw[4] = {sv[u].x, sv[u].y, sv[u].z, sv[u].w}, mw[4] = {mv[u].x, mv[u].y, mv[u].z, mv[u].w};
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float a = h2f((uint16_t)(sw[e / 2] >> (16 * (e & 1)))), b = h2f((uint16_t)(mw[e / 2] >> (16 * (e & 1))));
                sc[8 * i + e] = float2{a, b - 128.f * a};
            }
        }
    }
}

// Stage the activation group sums of the tile's picks: gs[pr][c] = src[row(pr) G + c] for
// pr < PB (rows past the tile repeat its last pick), all loads issued first.
__device__ __forceinline__ void stage_gsums(float* gs, const float* __restrict__ src, const int* __restrict__ rowmap,
                                            int p0, int np, int G) {
    constexpr int MAXP = PB * 64 / 256;
    float v[MAXP];
#pragma unroll
    for (int u = 0; u < MAXP; u++) {
        const int i = threadIdx.x + 256 * u;
        if (i < PB * G) {
            const int pr = i / G, c = i % G, p = p0 + min(pr, np - 1);
            v[u] = src[(size_t)(rowmap ? rowmap[p] : p) * G + c];
        }
    }
#pragma unroll
    for (int u = 0; u < MAXP; u++) {
        const int i = threadIdx.x + 256 * u;
        if (i < PB * G) gs[i] = v[u];
    }
}

// Gate / up: block (unit block ub of RB units) x tile. act[p][r] = silu(gate_r . x) * (up_r . x)
// for the tile's picks, stored as bf16 hi / lo in chunk order (ah, al [P][I]) with group sums
// as [P][I / 64] (the unit block is one 64-group of the down projection's input).
// Grid (I / RB unit blocks, tile-list capacity); the tile count and the tile record are read
// together, and the record carries the expert's row address (no pointer-table round trip).
template <int NT>  // pick tiles of 16: 1 for tiles of <= 16 picks, 2 for larger ones
__global__ void __launch_bounds__(256, 2) moe_gate_up_kernel(const MoeTile* __restrict__ tiles,
                                                          const int* __restrict__ ntiles,
                                                          const int* __restrict__ ptok, const uint16_t* __restrict__ xh,
                                                          const uint16_t* __restrict__ xl, const float* __restrict__ xs,
                                                          int D, int I, ExpertOffsets off, uint16_t* __restrict__ ah,
                                                          uint16_t* __restrict__ al, float* __restrict__ as) {
    // dynamic LDS: sc [2][RB][G] (s, m - 128 s) | gs [PB][G] activation group sums
    extern __shared__ float2 dyn[];
    __shared__ float ob[PB][RB + 1];     // gate sums, then act
    __shared__ float ub2[PB][RB + 1];    // up sums
    const int ub = blockIdx.x, tile = blockIdx.y;
    const MoeTile tl = tiles[tile];  // read before the count is known (capacity-sized list)
    if (tile >= *ntiles) return;
    const int G = D / 64, r0 = ub * RB;
    float2* sc = dyn;
    float* gs = (float*)(dyn + 2 * RB * G);
    const int p0 = tl.p0, np = tl.p1 - tl.p0;
    const unsigned char* base = (const unsigned char*)tl.base;
    auto stage = [&]() {
        stage_scales(sc, (const uint16_t*)(base + off.gu_s), (const uint16_t*)(base + off.gu_m), r0, G);
        stage_scales(sc + RB * G, (const uint16_t*)(base + off.gu_s), (const uint16_t*)(base + off.gu_m), I + r0, G);
        stage_gsums(gs, xs, ptok, p0, np, G);
    };
    const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE, n = lane % 16, g = lane / 16;
    long long xrow[2];
#pragma unroll
    for (int t = 0; t < 2; t++) xrow[t] = (long long)ptok[p0 + min(16 * t + n, np - 1)] * D;
    const long long qrow0[2] = {r0, I + r0};  // gate rows, up rows of this unit block
    BlockAcc<2, NT> acc;
    expert_block<2, NT>(base, qrow0, D, sc, xh, xl, xrow, gs, acc, G, stage);
    reduce_waves<2, NT>(acc, 0, ob);   // gate sums
    reduce_waves<2, NT>(acc, 1, ub2);  // up sums
    // 256 threads = 32 picks x 8 chunks of the 64 units
    const int pr = threadIdx.x / 8, q = threadIdx.x % 8;
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = silu_f(ob[pr][8 * q + i]) * ub2[pr][8 * q + i];
    uint4 hi, lo;
    float s;
    split8(v, hi, lo, s);
    s += __shfl_xor(s, 1, WAVE);
    s += __shfl_xor(s, 2, WAVE);
    s += __shfl_xor(s, 4, WAVE);
    if (pr < np) {
        const size_t p = p0 + pr;
        *(uint4*)(ah + p * I + r0 + 8 * q) = hi;
        *(uint4*)(al + p * I + r0 + 8 * q) = lo;
        if (q == 0) as[p * (I / 64) + ub] = s;
    }
}

// Down: block (output rows [RB ob, RB ob + RB)) x tile. ypick[src][o] = wts[src] * (dn_o . act).
// Grid (D / RB output blocks, tile-list capacity), tile records as for gate / up.
template <int NT>
__global__ void __launch_bounds__(256, 2) moe_down_kernel(const MoeTile* __restrict__ tiles,
                                                       const int* __restrict__ ntiles,
                                                       const int* __restrict__ psrc, const float* __restrict__ wts,
                                                       const uint16_t* __restrict__ ah, const uint16_t* __restrict__ al,
                                                       const float* __restrict__ as, int D, int I, ExpertOffsets off,
                                                       float* __restrict__ ypick) {
    // dynamic LDS: sc [RB][G] | gs [PB][G]
    extern __shared__ float2 dyn[];
    __shared__ float red[PB][RB + 1];  // the waves' summed outputs
    const int ob = blockIdx.x, tile = blockIdx.y;
    const MoeTile tl = tiles[tile];
    if (tile >= *ntiles) return;
    const int G = I / 64, o0 = ob * RB;
    float2* sc = dyn;
    float* gs = (float*)(dyn + RB * G);
    const int p0 = tl.p0, np = tl.p1 - tl.p0;
    const unsigned char* base = (const unsigned char*)tl.base;
    auto stage = [&]() {
        stage_scales(sc, (const uint16_t*)(base + off.dn_s), (const uint16_t*)(base + off.dn_m), o0, G);
        stage_gsums(gs, as, nullptr, p0, np, G);
    };
    const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE, n = lane % 16, g = lane / 16;
    long long xrow[2];
#pragma unroll
    for (int t = 0; t < 2; t++) xrow[t] = (long long)(p0 + min(16 * t + n, np - 1)) * I;
    const long long qrow0[1] = {o0};
    BlockAcc<1, NT> acc;
    expert_block<1, NT>(base + off.dn_q, qrow0, I, sc, ah, al, xrow, gs, acc, G, stage);
    reduce_waves<1, NT>(acc, 0, red);
    // 256 threads = 32 picks x 8 runs of 8 rows: ypick[src][o0 + 8 q ..] = w * y
    const int pr = threadIdx.x / 8, q = threadIdx.x % 8;
    if (pr < np) {
        const int src = psrc[p0 + pr];
        const float w = wts[src];
        float* dst = ypick + (size_t)src * D + o0 + 8 * q;
        const float* r = &red[pr][8 * q];
        ((float4*)dst)[0] = float4{w * r[0], w * r[1], w * r[2], w * r[3]};
        ((float4*)dst)[1] = float4{w * r[4], w * r[5], w * r[6], w * r[7]};
    }
}

// ---------------------------------------------------------------------------------------------
// Prefill-sized batches: every expert's picks in tiles of up to 64. A workgroup of 8 waves covers 512
// code rows for a tile's picks (gate / up: 256 units, i.e. 256 gate and 256 up rows; down: 512 output
// rows), each wave 64 rows as 4 row tiles, walking the 64-groups in order; the picks' activations of a
// group (hi and lo, 64 picks x 64 values) are staged once per workgroup in LDS (double-buffered, 16-byte
// slots XOR-swizzled by the pick row), so an activation byte is fetched once per workgroup and a
// code byte once per tile.
//
// Bound by the VALU beside the products (batch 2048: matrix cores busy 28% and vector units 42% of the
// cycles in the earlier form, which spent 6 vector instructions per product). Kept out of the loop:
//   - the min's term sum_g m X, which is itself a matrix product over the groups: it starts the
//     accumulators, m as two bf16 parts and the fp32 group sums X as three (both exact), 6 products
//     per tile instead of 4 FMAs per group and tile;
//   - the 128 of the codes: a group's products start from -128 X (one splat per pick tile and group, the
//     C operand of every row tile's first product), so what leaves them is sum c x, and the scale is
//     applied by one mixed-precision FMA per value with the fp16 scale as it stands;
//   - column tiles without picks: NT = 1 .. 4 by the tile's count.
// The codes stay two groups ahead over an LDS-only barrier per pair of groups.
// Measured, batch 2048 of 256 experts (gate / up + down, traced): 331 + 205 us before, 259 + 179 us now (over the
// benchmark's ring of layers, whose scales and mins are all alike, 230 + 159); with neither codes, activations nor LDS reads in the loop the whole op still takes 380 of its 415 us: the products
// and the vector work of the two waves of a SIMD overlap poorly (28% and 25% busy), and a workgroup's
// start is 8 us of its 40 (down) to 100 (gate / up).
constexpr int NWB = 8;         // waves per big workgroup (one workgroup per CU)
constexpr int RTB = 4;         // row tiles per wave
constexpr int UB = 32 * NWB;   // units per gate / up workgroup
constexpr int OB = 64 * NWB;   // output rows per down workgroup
static_assert(2 * UB == kMoeRows && OB == kMoeRows, "moe_tile_picks counts workgroups of this many rows");

// Scales and group sums lie group-major: a lane's 4 rows of scales are one 8-byte read, the picks' sums
// 16 consecutive words, and every offset is a constant.
constexpr int BSR = 64 * NWB + 4, BGR = PBB;
constexpr int kActBytes = 2 * PBB * 128;     // one group's activations: hi, lo x 64 picks x 128 B
struct BigSmem {
    __attribute__((aligned(1024))) unsigned char act[2][2][kActBytes];  // two pairs of groups
    __attribute__((aligned(16))) uint16_t sc[32 * BSR];  // fp16 scales [group][wave's row], G <= 32
    float gs[32 * BGR];                      // activation group sums [group][pick]
    float red[NWB][PBB];
};

// The tile's sums: acc[rt][t] of lane (n, g) = rows qrow[rt] + 4 g + j, pick 16 t + n, over the G groups of
// Kdim codes. row_of(pick): its row in xh / xl; sc_row(r): the code row of LDS scale row r (the wave's rows
// are 64 wave + 16 rt + ..); gs_of(pick, group): its group sum. A workgroup's start is a chain of round
// trips that its few groups have to pay for (down: 8), so every load of the start is issued before the
// first is used, and one barrier publishes all that is staged.
template <int NT, typename RowOf, typename ScRow, typename GsOf>
__device__ __forceinline__ void big_block(BigSmem& sm, RowOf row_of, ScRow sc_row, GsOf gs_of,
                                          const unsigned char* __restrict__ qbase, const unsigned char* __restrict__ sbase,
                                          const unsigned char* __restrict__ mbase, const int (&qrow)[RTB], int Kdim,
                                          const uint16_t* __restrict__ xh, const uint16_t* __restrict__ xl, int G,
                                          f32x4 (&acc)[RTB][4]) {
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
    const int n = lane % 16, g = lane / 16;
    typedef uint32_t u2v __attribute__((ext_vector_type(2)));
    typedef uint32_t u4w __attribute__((ext_vector_type(4)));
    unsigned arow[RTB];
#pragma unroll
    for (int rt = 0; rt < RTB; rt++) arow[rt] = (unsigned)(qrow[rt] + n) * (Kdim / 2) + 8 * g;
    // activation pieces: 16 per group (8 per part, 8 picks x 128 B each), 16 / NWB per wave (pieces of
    // picks past the tile's column tiles are skipped: uniform); lane L of piece q holds slot L % 8 of pick
    // 8 (q % 8) + L / 8, which goes to LDS slot (L % 8) ^ sw(pick). Through registers: with direct
    // global -> LDS copies the compiler drains every load in flight, the codes' prefetch too, at each
    // group's barrier
    constexpr int PPW = 16 / NWB;
    unsigned src[PPW];
    int dst[PPW];
#pragma unroll
    for (int u = 0; u < PPW; u++) {
        const int q = PPW * wave + u, pk = 8 * (q % 8) + lane / 8;
        src[u] = (unsigned)row_of(pk) * (2 * Kdim) + (lane % 8) * 16;
        dst[u] = (q / 8 * PBB + pk) * 128 + ((lane % 8) ^ ((pk >> 1) & 7)) * 16;
    }
    u4w st[2][PPW];  // a pair of groups in flight
    auto fetch = [&](int set, int grp) {
#pragma unroll
        for (int u = 0; u < PPW; u++) {
            const int q = PPW * wave + u;
            if ((q % 8) < 2 * NT)
                st[set][u] = ld_global<u4w>((const unsigned char*)(q < 8 ? xh : xl) + (src[u] + 128 * min(grp, G - 1)));
        }
    };
    auto store = [&](int set, unsigned char* buf) {
#pragma unroll
        for (int u = 0; u < PPW; u++)
            if (((PPW * wave + u) % 8) < 2 * NT) *(u4w*)(buf + dst[u]) = st[set][u];
    };
    // codes of group grp for every row tile (ring of 2 groups)
    u2v ar[2][RTB];
    fetch(0, 0);
    fetch(1, 1);
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
        for (int rt = 0; rt < RTB; rt++) ar[u][rt] = ld_global<u2v>(qbase + (arow[rt] + 32 * min(u, G - 1)));
    // the row mins of groups 8 g .. 8 g + 7, all requested at once (clamped: a guarded load waits in its branch)
    u4w mraw[RTB];
    if (G % 8 == 0) {
#pragma unroll
        for (int rt = 0; rt < RTB; rt++)
            mraw[rt] = ld_global<u4w>(mbase + ((unsigned)(qrow[rt] + n) * G + min(8 * g, G - 8)) * 2);
    } else {
#pragma unroll
        for (int rt = 0; rt < RTB; rt++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const unsigned row = (unsigned)(qrow[rt] + n) * G;
                const uint32_t a = ld_global<uint16_t>(mbase + (row + min(8 * g + 2 * e, G - 1)) * 2);
                const uint32_t b = ld_global<uint16_t>(mbase + (row + min(8 * g + 2 * e + 1, G - 1)) * 2);
                mraw[rt][e] = a | (b << 16);
            }
    }
    // scales: 8 halves of a row per piece, G / 8 (rounded up) pieces a row; group sums: 64 picks a group
    constexpr int NTH = 64 * NWB, SMAX = 64 * NWB * 32 / 8 / NTH, GMAX = PBB * 32 / NTH;
    u4w sv[SMAX];
    float gv[GMAX];
    const int npc = 64 * NWB * G / 8;
#pragma unroll
    for (int u = 0; u < SMAX; u++) {
        const int i = min(tid + NTH * u, npc - 1), r = 8 * i / G;  // a piece may end in the next row: the same run
        if (NTH * u < npc) sv[u] = ld_global<u4w>(sbase + ((unsigned)sc_row(r / 32 * 32) * G + (8 * i - r / 32 * 32 * G)) * 2);
    }
#pragma unroll
    for (int u = 0; u < GMAX; u++) {
        const int i = tid + NTH * u;
        if (NTH * u < PBB * G) gv[u] = gs_of(i % PBB, min(i / PBB, G - 1));
    }
    store(0, sm.act[0][0]);
    store(1, sm.act[0][1]);
#pragma unroll
    for (int u = 0; u < SMAX; u++) {
        const int i = tid + NTH * u;
        if (i < npc) {
#pragma unroll
            for (int e = 0; e < 8; e++)
                sm.sc[(8 * i + e) % G * BSR + (8 * i + e) / G] = (uint16_t)(sv[u][e / 2] >> (16 * (e & 1)));
        }
    }
#pragma unroll
    for (int u = 0; u < GMAX; u++) {
        const int i = tid + NTH * u;
        if (i < PBB * G) sm.gs[i / PBB * BGR + i % PBB] = gv[u];
    }
    fetch(0, 2);
    fetch(1, 3);
    lds_barrier();
    // acc = sum over groups of m X: A = m [row][8 g .. 8 g + 7], B = X [pick][same groups], zeros past G
    {
        bf16x8 xb[3][NT];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            uint32_t p1[4], p2[4], p3[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                float x[2], r[2], q[2];
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const int k = 8 * g + 2 * e + h;
                    const float xk = sm.gs[min(k, G - 1) * BGR + 16 * t + n];
                    x[h] = k < G ? xk : 0.f;
                    r[h] = x[h] - __uint_as_float(__float_as_uint(x[h]) & 0xffff0000u);
                    q[h] = r[h] - __uint_as_float(__float_as_uint(r[h]) & 0xffff0000u);
                }
                p1[e] = __builtin_amdgcn_perm(__float_as_uint(x[1]), __float_as_uint(x[0]), 0x07060302u);
                p2[e] = __builtin_amdgcn_perm(__float_as_uint(r[1]), __float_as_uint(r[0]), 0x07060302u);
                p3[e] = f2bf2(q[0], q[1]);
            }
            xb[0][t] = __builtin_bit_cast(bf16x8, p1);
            xb[1][t] = __builtin_bit_cast(bf16x8, p2);
            xb[2][t] = __builtin_bit_cast(bf16x8, p3);
        }
#pragma unroll
        for (int rt = 0; rt < RTB; rt++) {
            uint32_t hi[4], lo[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                float m[2], l[2];
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    m[h] = 8 * g + 2 * e + h < G ? h2f((uint16_t)(mraw[rt][e] >> (16 * h))) : 0.f;
                    l[h] = m[h] - __uint_as_float(__float_as_uint(m[h]) & 0xffff0000u);
                }
                hi[e] = __builtin_amdgcn_perm(__float_as_uint(m[1]), __float_as_uint(m[0]), 0x07060302u);
                lo[e] = __builtin_amdgcn_perm(__float_as_uint(l[1]), __float_as_uint(l[0]), 0x07060302u);
            }
            const bf16x8 ah = __builtin_bit_cast(bf16x8, hi), al = __builtin_bit_cast(bf16x8, lo);
#pragma unroll
            for (int t = 0; t < NT; t++) {
                f32x4 v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int p = 2; p >= 0; p--) {  // smallest parts first
                    v = mfma_bf(al, xb[p][t], v);
                    v = mfma_bf(ah, xb[p][t], v);
                }
                acc[rt][t] = v;
            }
#pragma unroll
            for (int t = 0; t < NT; t++) asm volatile("" : "+v"(acc[rt][t]));
        }
    }
    uint32_t mask = 0x000F000Fu, magic = 0x43004300u;
    asm volatile("" : "+s"(mask), "+v"(magic));  // in registers: one and-or per pair of codes
    auto codes = [&](uint32_t p) {
        u4w d;
#pragma unroll
        for (int j = 0; j < 4; j++) d[j] = ((p >> (4 * j)) & mask) | magic;
        return __builtin_bit_cast(bf16x8, d);
    };
    auto group = [&](int grp, int slot, const unsigned char* cur) {
        // this group's activation fragments: pick tile t, k step ks: LDS slot (2 g + ks) ^ sw(row)
        bf16x8 bh[NT][2], bl[NT][2];
        f32x4 c0[NT];  // -128 X of the pick in all four rows
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const int row = 16 * t + n;
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
                const int off = row * 128 + (((2 * g + ks) ^ ((row >> 1) & 7)) * 16);
                bh[t][ks] = *(const bf16x8*)(cur + off);
                bl[t][ks] = *(const bf16x8*)(cur + PBB * 128 + off);
            }
            const float x = -128.f * sm.gs[grp * BGR + row];
            c0[t] = f32x4{x, x, x, x};
        }
#pragma unroll
        for (int rt = 0; rt < RTB; rt++) {
            const u2v a2 = ar[slot][rt];
            const uint2 sv = *(const uint2*)&sm.sc[grp * BSR + 64 * wave + 16 * rt + 4 * g];
            const bf16x8 a0 = codes(a2.x), a1 = codes(a2.y);
            f32x4 P[NT];
#pragma unroll
            for (int t = 0; t < NT; t++) P[t] = mfma_bf(a0, bh[t][0], c0[t]);
#pragma unroll
            for (int t = 0; t < NT; t++) P[t] = mfma_bf(a0, bl[t][0], P[t]);
#pragma unroll
            for (int t = 0; t < NT; t++) P[t] = mfma_bf(a1, bh[t][1], P[t]);
#pragma unroll
            for (int t = 0; t < NT; t++) P[t] = mfma_bf(a1, bl[t][1], P[t]);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float s = h2f((uint16_t)((j < 2 ? sv.x : sv.y) >> (16 * (j & 1))));
#pragma unroll
                for (int t = 0; t < NT; t++) acc[rt][t][j] = fmaf(s, P[t][j], acc[rt][t][j]);
            }
            // this row tile is done: without the fence its sums drift past the store and the barrier,
            // with every row tile's products alive (340 spilled registers)
#pragma unroll
            for (int t = 0; t < NT; t++) asm volatile("" : "+v"(acc[rt][t]));
        }
        // refill this ring slot with the codes two groups ahead (past the end: the last group's)
#pragma unroll
        for (int rt = 0; rt < RTB; rt++) ar[slot][rt] = ld_global<u2v>(qbase + (arow[rt] + 32 * min(grp + 2, G - 1)));
    };
    // G is even (rows of 128 codes): one barrier per pair of groups; the next pair's activations, in
    // flight during this one, go to the other half of the buffer
    int buf = 0;
#pragma unroll 1
    for (int grp = 0; grp < G; grp += 2) {
#pragma unroll
        for (int u = 0; u < 2; u++) group(grp + u, u, sm.act[buf][u]);
        buf ^= 1;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            store(u, sm.act[buf][u]);
            fetch(u, grp + 4 + u);
        }
        lds_barrier();
    }
}

// Gate / up for big tiles: units [UB ub, UB ub + UB) x one tile of <= 64 picks. act as in
// moe_gate_up_kernel (bf16 hi / lo in chunk order, group sums over 64 units).
template <int NT>
__device__ __forceinline__ void big_gate_up(BigSmem& sm, const unsigned char* base, const ExpertOffsets& off, int p0, int np,
                                            const int* __restrict__ ptok, const float* __restrict__ xs,
                                            const uint16_t* __restrict__ xh, const uint16_t* __restrict__ xl, int D, int I,
                                            uint16_t* __restrict__ ah, uint16_t* __restrict__ al, float* __restrict__ as) {
    const int tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE, n = lane % 16, g = lane / 16;
    const int ub = blockIdx.x, u0 = ub * UB;
    // wave w: units u0 + 32 w .. + 32: gate row tiles 0, 1 and up row tiles 2, 3
    // (I is a multiple of 128: waves past it repeat the last units, unstored)
    const bool mine = u0 + 32 * wave < I;
    const int wu = mine ? u0 + 32 * wave : I - 32;
    const int qrow[RTB] = {wu, wu + 16, I + wu, I + wu + 16};
    f32x4 acc[RTB][4];
    // picks past the tile repeat its last one (their results are not stored); LDS scale row
    // 64 w + 32 m + r is matrix m's row u0 + 32 w + r
    const int G = D / 64;
    auto row_of = [&](int pk) { return ptok[p0 + min(pk, np - 1)]; };
    auto sc_row = [&](int r) { return r / 32 % 2 * I + min(u0 + r / 64 * 32, I - 32) + r % 32; };
    auto gs_of = [&](int pk, int k) { return xs[(size_t)row_of(pk) * G + k]; };
    big_block<NT>(sm, row_of, sc_row, gs_of, base, base + off.gu_s, base + off.gu_m, qrow, D, xh, xl, G, acc);
    // act = silu(gate) * up; lane (n, g) of tile (rt, t) holds units wu + 16 rt + 4 g + j of pick
    // 16 t + n. A chunk of 8 units lies in lanes g = 2c and 2c + 1: the even lane takes the odd
    // lane's 4 values and writes the chunk (hi, lo in chunk order) and its sum.
    float wsum[NT];  // per pick tile: this lane's chunk sums
#pragma unroll
    for (int t = 0; t < NT; t++) wsum[t] = 0.f;
#pragma unroll
    for (int rt = 0; rt < 2; rt++)
#pragma unroll
        for (int t = 0; t < NT; t++) {
            float a[4], o[4];
#pragma unroll
            for (int j = 0; j < 4; j++) a[j] = silu_f(acc[rt][t][j]) * acc[rt + 2][t][j];
#pragma unroll
            for (int j = 0; j < 4; j++) o[j] = __shfl_xor(a[j], 16, WAVE);
            if ((g & 1) == 0) {
                const float v[8] = {a[0], a[1], a[2], a[3], o[0], o[1], o[2], o[3]};
                uint4 hi, lo;
                float sum;
                split8(v, hi, lo, sum);
                wsum[t] += sum;
                const int pr = 16 * t + n;
                if (pr < np && mine) {
                    const size_t p = p0 + pr;
                    const int u = wu + 16 * rt + 4 * g;  // the chunk's first unit
                    *(uint4*)(ah + p * I + u) = hi;
                    *(uint4*)(al + p * I + u) = lo;
                }
            }
        }
    // group sums: a 64-unit group is waves 2 k and 2 k + 1; per wave, the even lanes g = 0, 2 of
    // pick n hold its chunk sums
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const float s2 = wsum[t] + __shfl_xor(wsum[t], 32, WAVE);
        if (g == 0) sm.red[wave][16 * t + n] = s2;
    }
    __syncthreads();
    if (tid < (UB / 64) * PBB) {
        const int k = tid / PBB, pr = tid % PBB;
        if (pr < np && u0 + 64 * k < I) as[(size_t)(p0 + pr) * (I / 64) + (u0 / 64) + k] = sm.red[2 * k][pr] + sm.red[2 * k + 1][pr];
    }
}

__global__ void __launch_bounds__(64 * NWB, 2) moe_gate_up_big_kernel(const MoeTile* __restrict__ tiles,
                                                              const int* __restrict__ ntiles,
                                                              const int* __restrict__ ptok,
                                                              const uint16_t* __restrict__ xh,
                                                              const uint16_t* __restrict__ xl,
                                                              const float* __restrict__ xs, int D, int I,
                                                              ExpertOffsets off, uint16_t* __restrict__ ah,
                                                              uint16_t* __restrict__ al, float* __restrict__ as) {
    __shared__ BigSmem sm;
    const MoeTile tl = tiles[blockIdx.y];
    if ((int)blockIdx.y >= *ntiles) return;
    const int p0 = tl.p0, np = tl.p1 - tl.p0;
    const unsigned char* base = (const unsigned char*)tl.base;
    switch ((np + 15) / 16) {
        case 1: big_gate_up<1>(sm, base, off, p0, np, ptok, xs, xh, xl, D, I, ah, al, as); break;
        case 2: big_gate_up<2>(sm, base, off, p0, np, ptok, xs, xh, xl, D, I, ah, al, as); break;
        case 3: big_gate_up<3>(sm, base, off, p0, np, ptok, xs, xh, xl, D, I, ah, al, as); break;
        default: big_gate_up<4>(sm, base, off, p0, np, ptok, xs, xh, xl, D, I, ah, al, as);
    }
}

// Down for big tiles: output rows [OB ob, OB ob + OB) x one tile of <= 64 picks; ypick[src][o] =
// wts[src] * (dn_o . act), as moe_down_kernel.
template <int NT>
__device__ __forceinline__ void big_down(BigSmem& sm, const unsigned char* base, const ExpertOffsets& off, int p0, int np,
                                         const int* __restrict__ psrc, const float* __restrict__ wts,
                                         const float* __restrict__ as, const uint16_t* __restrict__ ah, const uint16_t* __restrict__ al, int D, int I,
                                         float* __restrict__ ypick) {
    const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE, n = lane % 16, g = lane / 16;
    const int wo = blockIdx.x * OB + 64 * wave;
    // D is a multiple of 128: the last workgroup's upper waves repeat its last rows, unstored
    const int qrow[RTB] = {min(wo, D - 16), min(wo + 16, D - 16), min(wo + 32, D - 16), min(wo + 48, D - 16)};
    f32x4 acc[RTB][4];
    const int G = I / 64;
    int src[NT];  // the lane's picks, wanted only at the end
#pragma unroll
    for (int t = 0; t < NT; t++) src[t] = psrc[p0 + min(16 * t + n, np - 1)];
    auto row_of = [&](int pk) { return p0 + min(pk, np - 1); };
    auto sc_row = [&](int r) { return min((int)blockIdx.x * OB + r / 32 * 32, D - 32) + r % 32; };
    auto gs_of = [&](int pk, int k) { return as[(size_t)row_of(pk) * G + k]; };
    big_block<NT>(sm, row_of, sc_row, gs_of, base + off.dn_q, base + off.dn_s, base + off.dn_m, qrow, I, ah, al, G, acc);
    float w[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) w[t] = wts[src[t]];
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const int pr = 16 * t + n;
        if (pr >= np) continue;
#pragma unroll
        for (int rt = 0; rt < RTB; rt++) {
            if (wo + 16 * rt >= D) break;
            const f32x4 v = acc[rt][t] * w[t];
            *(f32x4*)(ypick + (size_t)src[t] * D + wo + 16 * rt + 4 * g) = v;
        }
    }
}

__global__ void __launch_bounds__(64 * NWB, 2) moe_down_big_kernel(const MoeTile* __restrict__ tiles,
                                                           const int* __restrict__ ntiles, const int* __restrict__ psrc,
                                                           const float* __restrict__ wts,
                                                           const uint16_t* __restrict__ ah,
                                                           const uint16_t* __restrict__ al,
                                                           const float* __restrict__ as, int D, int I,
                                                           ExpertOffsets off, float* __restrict__ ypick) {
    __shared__ BigSmem sm;
    const MoeTile tl = tiles[blockIdx.y];
    if ((int)blockIdx.y >= *ntiles) return;
    const int p0 = tl.p0, np = tl.p1 - tl.p0;
    const unsigned char* base = (const unsigned char*)tl.base;
    switch ((np + 15) / 16) {
        case 1: big_down<1>(sm, base, off, p0, np, psrc, wts, as, ah, al, D, I, ypick); break;
        case 2: big_down<2>(sm, base, off, p0, np, psrc, wts, as, ah, al, D, I, ypick); break;
        case 3: big_down<3>(sm, base, off, p0, np, psrc, wts, as, ah, al, D, I, ypick); break;
        default: big_down<4>(sm, base, off, p0, np, psrc, wts, as, ah, al, D, I, ypick);
    }
}

// x[t] += sum_k ypick[t K + k] (k in order) and, with a shared expert, + sigmoid(h_t . wg) ysh[t].
// Grid (T, D / 256): one thread per column; the K pick rows are loaded together.
__global__ void __launch_bounds__(256) moe_combine_kernel(float* __restrict__ x, const float* __restrict__ ypick,
                                                          const int* __restrict__ idx, int E,
                                                          const float* __restrict__ ysh, const float* __restrict__ h,
                                                          const uint16_t* __restrict__ wg, int D, int K) {
    __shared__ float red[8];
    const int t = blockIdx.x, i = blockIdx.y * blockDim.x + threadIdx.x, ii = min(i, D - 1);
    // every load is issued before the gate's reduction (a workgroup is a chain of round trips at
    // decode sizes); dropped picks read a row that is not added
    float v[16];
    bool ok[16];
#pragma unroll
    for (int k = 0; k < 16; k++) {
        if (k < K) {
            const int e = idx[(size_t)t * K + k];
            ok[k] = e >= 0 && e < E;
            v[k] = ypick[((size_t)t * K + k) * D + ii];
        }
    }
    const float x0 = x[(size_t)t * D + ii], y0 = ysh ? ysh[(size_t)t * D + ii] : 0.f;
    float gate = 0.f;
    if (ysh) {
        float a = 0.f;
        for (int c = threadIdx.x; c < D; c += blockDim.x) a += h[(size_t)t * D + c] * bf2f(wg[c]);
        gate = sigmoid_f(block_sum(a, red));
    }
    if (i >= D) return;
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < 16; k++)
        if (k < K) s += ok[k] ? v[k] : 0.f;
    float r = x0 + s;
    if (ysh) r += gate * y0;
    x[(size_t)t * D + i] = r;
}

// x[t] += sigmoid(h_t . wg) y[t] (the engine's shared_gate_add)
__global__ void __launch_bounds__(256) shared_gate_add_kernel(float* __restrict__ x, const float* __restrict__ y,
                                                              const float* __restrict__ h,
                                                              const uint16_t* __restrict__ wg, int D) {
    __shared__ float red[8];
    const int t = blockIdx.x;
    float a = 0.f;
    for (int i = threadIdx.x; i < D; i += blockDim.x) a += h[(size_t)t * D + i] * bf2f(wg[i]);
    const float gate = sigmoid_f(block_sum(a, red));
    for (int i = threadIdx.x; i < D; i += blockDim.x) x[(size_t)t * D + i] += gate * y[(size_t)t * D + i];
}

__global__ void silu_mul_kernel(const float* __restrict__ g, const float* __restrict__ u, float* __restrict__ out,
                                long long n) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = silu_f(g[i]) * u[i];
}

// AEGIST_MOE_BIG=0 keeps every tile at <= 32 picks (A/B runs).
static bool big_tiles_enabled() {
    const char* e = getenv("AEGIST_MOE_BIG");
    return !(e && e[0] == '0');
}

// Workspace plan of aegist_moe_experts.
struct MoePlan {
    size_t xh, xl, xs, ah, al, as, yp, cnt, ptok, psrc, tiles1, tiles2, tiles3, meta, total;
    int per, nb;           // grouping: picks per block, blocks (at most 64: each reads all the blocks' counts)
    int cap;               // picks per prefill tile, 0: the tiles of <= 32 picks
    int max1, max2, max3;  // tile-list capacities: <= 16 picks (one per expert), 17..32, prefill tiles
};
static size_t al256(size_t x) { return (x + 255) / 256 * 256; }
static MoePlan moe_plan(int T, int K, int D, int I, int E) {
    MoePlan p;
    const size_t N = (size_t)T * K;
    p.max1 = (int)std::min<size_t>(N, (size_t)E);
    // an expert with c picks has floor(c / PB) + [c % PB > 16] <= c / 17 large blocks
    p.max2 = (int)(N / 17);
    // the prefill tiles' rows are whole pairs of groups up to 2048, addressed through 32-bit byte offsets
    const bool fits = D % 128 == 0 && I % 128 == 0 && D / 64 <= 32 && I / 64 <= 32 && (size_t)T * D * 2 < (1ull << 32) &&
                      N * I * 2 < (1ull << 32);
    p.cap = fits ? moe_tile_picks(T, K, E, D, I) : 0;
    p.max3 = p.cap ? (int)(N / p.cap + std::min<size_t>(N, (size_t)E)) : 0;  // sum of ceil(c / cap)
    // room for the smallest tiles whatever this batch takes: a workspace for more tokens serves fewer
    const size_t room3 = N / 16 + std::min<size_t>(N, (size_t)E);
    p.per = (int)std::max<size_t>(1024, (N + 63) / 64);
    p.nb = (int)((N + p.per - 1) / p.per);
    size_t o = 0;
    auto take = [&](size_t bytes) {
        const size_t at = o;
        o += al256(bytes);
        return at;
    };
    p.xh = take((size_t)T * D * 2);
    p.xl = take((size_t)T * D * 2);
    p.xs = take((size_t)T * (D / 64) * 4);
    p.ah = take(N * I * 2);
    p.al = take(N * I * 2);
    p.as = take(N * (I / 64) * 4);
    p.yp = take(N * D * 4);
    p.cnt = take((size_t)p.nb * E * 4);
    p.ptok = take(N * 4);
    p.psrc = take(N * 4);
    p.tiles1 = take((size_t)p.max1 * sizeof(MoeTile));
    p.tiles2 = take((size_t)std::max(p.max2, 1) * sizeof(MoeTile));
    p.tiles3 = take(room3 * sizeof(MoeTile));
    p.meta = take(16);
    p.total = o;
    return p;
}

}  // namespace

extern "C" {

size_t aegist_router_topk_workspace_bytes(int T, int E) {
    return T > 0 && E > 0 ? (size_t)T * E * 4 : 0;
}

int aegist_router_topk_ws(const float* h, const uint16_t* W, int* idx, float* wts, int T, int D, int E, int K,
                          void* ws, size_t ws_bytes, void* stream) {
    AEG_REQUIRE(T >= 0 && D > 0 && D % 16 == 0, "router_topk: need D % 16 == 0");
    AEG_REQUIRE(E > 0 && E <= 64 * 64, "router_topk: need 0 < E <= 4096");
    AEG_REQUIRE(K > 0 && K <= 16 && K <= E, "router_topk: need 0 < K <= min(16, E)");
    if (T == 0) return 0;
    // logits [T, E] = h W^T on the projection kernel (fp32 h as bf16 hi + lo against the exact
    // bf16 W), in the workspace
    int rc = check_workspace(ws, ws_bytes, aegist_router_topk_workspace_bytes(T, E), "router_topk");
    if (rc) return rc;
    float* logits = (float*)ws;
    hipStream_t st = AEG_STREAM(stream);
    rc = launch_proj(h, AEGIST_F32, D, W, AEGIST_BF16, nullptr, logits, E, T, E, D, 0, st);
    if (rc) return rc;
    const unsigned grid = (T + 3) / 4;
    if (E <= 64) router_topk_kernel<1><<<grid, 256, 0, st>>>(logits, idx, wts, T, E, K);
    else if (E <= 256) router_topk_kernel<4><<<grid, 256, 0, st>>>(logits, idx, wts, T, E, K);
    else if (E <= 1024) router_topk_kernel<16><<<grid, 256, 0, st>>>(logits, idx, wts, T, E, K);
    else router_topk_kernel<64><<<grid, 256, 0, st>>>(logits, idx, wts, T, E, K);
    return after_launch("router_topk");
}

int aegist_router_topk(const float* h, const uint16_t* W, int* idx, float* wts, int T, int D, int E, int K,
                       void* stream) {
    size_t bound = 0;
    void* ws = bound_workspace(&bound);
    return aegist_router_topk_ws(h, W, idx, wts, T, D, E, K, ws, bound, stream);
}

size_t aegist_moe_workspace_bytes(int T, int K, int D, int I, int E) {
    if (T <= 0 || K <= 0 || D <= 0 || I <= 0 || E <= 0) return 256;
    return moe_plan(T, K, D, I, E).total;
}

int aegist_moe_experts(const float* h, const unsigned long long* eptr, const int* idx, const float* wts, float* x,
                       int T, int D, int I, int E, int K, const float* ysh, const uint16_t* wg, void* ws,
                       size_t ws_bytes, void* stream) {
    AEG_REQUIRE(T >= 0 && K > 0 && K <= 16, "moe_experts: need T >= 0, 0 < K <= 16");
    AEG_REQUIRE(D % 64 == 0 && D >= 64 && D <= 64 * 64, "moe_experts: need D % 64 == 0 and D <= 4096");
    AEG_REQUIRE(I % 64 == 0 && I >= 64 && I <= 64 * 64, "moe_experts: need I % 64 == 0 and I <= 4096");
    AEG_REQUIRE(E > 0 && E <= MAX_E, "moe_experts: need 0 < E <= 1024");
    AEG_REQUIRE((ysh == nullptr) == (wg == nullptr), "moe_experts: the shared output and its gate come together");
    AEG_REQUIRE((long long)T * K < (1LL << 31) / 2, "moe_experts: too many picks");
    if (T == 0) return 0;
    const MoePlan p = moe_plan(T, K, D, I, E);
    if (!ws || ws_bytes < p.total) return fail(AEGIST_ERR_WORKSPACE, "moe_experts: workspace too small");
    AEG_REQUIRE((uintptr_t)h % 16 == 0 && (uintptr_t)x % 16 == 0, "moe_experts: h and x must be 16-byte aligned");
    unsigned char* w = (unsigned char*)ws;
    hipStream_t st = AEG_STREAM(stream);
    const ExpertOffsets off = expert_offsets(D, I);
    const int N = T * K;
    int* ptok = (int*)(w + p.ptok);
    int* psrc = (int*)(w + p.psrc);
    MoeTile* tiles1 = (MoeTile*)(w + p.tiles1);
    MoeTile* tiles2 = (MoeTile*)(w + p.tiles2);
    MoeTile* tiles3 = (MoeTile*)(w + p.tiles3);
    int* meta = (int*)(w + p.meta);
    uint16_t* xh = (uint16_t*)(w + p.xh);
    uint16_t* xl = (uint16_t*)(w + p.xl);
    float* xs = (float*)(w + p.xs);
    uint16_t* ah = (uint16_t*)(w + p.ah);
    uint16_t* al = (uint16_t*)(w + p.al);
    float* as = (float*)(w + p.as);
    float* yp = (float*)(w + p.yp);

    if (moe_decode_fits(T, D, I, E, K)) {
        // fp32 activations in the place of the hi / lo parts
        int rc = launch_moe_decode(h, eptr, idx, wts, T, D, I, E, K, off.gu_s, off.gu_m, off.dn_q, off.dn_s, off.dn_m,
                                   (float*)ah, yp, st);
        if (rc) return rc;
        moe_combine_kernel<<<dim3(T, (D + 255) / 256), 256, 0, st>>>(x, yp, idx, E, ysh, h, wg, D, K);
        return after_launch("moe_combine");
    }
    const int cap = big_tiles_enabled() ? p.cap : 0;
    int* cnt = (int*)(w + p.cnt);
    const long long nq = (long long)T * (D / 8);
    moe_count_kernel<<<p.nb + (unsigned)((nq + 255) / 256), 256, 0, st>>>(idx, N, E, p.per, p.nb, cnt, h, T, D, xh, xl, xs);
    int rc = after_launch("moe_count");
    if (rc) return rc;
    moe_place_kernel<<<p.nb, 1024, 0, st>>>(idx, N, K, E, p.per, p.nb, cnt, eptr, ptok, psrc, tiles1, tiles2, tiles3, cap, meta);
    if ((rc = after_launch("moe_place"))) return rc;
    if (cap) {
        moe_gate_up_big_kernel<<<dim3((I + UB - 1) / UB, p.max3), 64 * NWB, 0, st>>>(tiles3, meta + 2, ptok, xh, xl, xs, D, I, off, ah,
                                                                   al, as);
        if ((rc = after_launch("moe_gate_up_big"))) return rc;
        moe_down_big_kernel<<<dim3((D + OB - 1) / OB, p.max3), 64 * NWB, 0, st>>>(tiles3, meta + 2, psrc, wts, ah, al, as, D,
                                                                                  I, off, yp);
        if ((rc = after_launch("moe_down_big"))) return rc;
        moe_combine_kernel<<<dim3(T, (D + 255) / 256), 256, 0, st>>>(x, yp, idx, E, ysh, h, wg, D, K);
        return after_launch("moe_combine");
    }
    // Picks with an out-of-range expert id are dropped: no tile covers them and the combine
    // skips their rows, so nothing has to be cleared.
    const size_t lds_gu = (size_t)(2 * RB + PB) * (D / 64) * 8, lds_dn = (size_t)(RB + PB) * (I / 64) * 8;
    // two launches per projection: tiles of <= 16 picks (one MFMA column tile, the decode case)
    // and larger tiles (two); a workgroup past its list's count exits at once
    moe_gate_up_kernel<1><<<dim3(I / RB, p.max1), 256, lds_gu, st>>>(tiles1, meta, ptok, xh, xl, xs, D, I, off, ah, al,
                                                                     as);
    if ((rc = after_launch("moe_gate_up"))) return rc;
    if (p.max2 > 0) {
        moe_gate_up_kernel<2><<<dim3(I / RB, p.max2), 256, lds_gu, st>>>(tiles2, meta + 1, ptok, xh, xl, xs, D, I, off,
                                                                         ah, al, as);
        if ((rc = after_launch("moe_gate_up"))) return rc;
    }
    moe_down_kernel<1><<<dim3(D / RB, p.max1), 256, lds_dn, st>>>(tiles1, meta, psrc, wts, ah, al, as, D, I, off, yp);
    if ((rc = after_launch("moe_down"))) return rc;
    if (p.max2 > 0) {
        moe_down_kernel<2><<<dim3(D / RB, p.max2), 256, lds_dn, st>>>(tiles2, meta + 1, psrc, wts, ah, al, as, D, I,
                                                                      off, yp);
        if ((rc = after_launch("moe_down"))) return rc;
    }
    moe_combine_kernel<<<dim3(T, (D + 255) / 256), 256, 0, st>>>(x, yp, idx, E, ysh, h, wg, D, K);
    return after_launch("moe_combine");
}

int aegist_shared_gate_add(float* x, const float* y, const float* h, const uint16_t* wg, int T, int D, void* stream) {
    AEG_REQUIRE(T >= 0 && D > 0, "shared_gate_add: bad shape");
    if (T == 0) return 0;
    shared_gate_add_kernel<<<T, 256, 0, AEG_STREAM(stream)>>>(x, y, h, wg, D);
    return after_launch("shared_gate_add");
}

int aegist_silu_mul(const float* g, const float* u, float* out, long long n, void* stream) {
    AEG_REQUIRE(n >= 0, "silu_mul: bad size");
    if (n == 0) return 0;
    silu_mul_kernel<<<(unsigned)((n + 255) / 256), 256, 0, AEG_STREAM(stream)>>>(g, u, out, n);
    return after_launch("silu_mul");
}

}  // extern "C"
