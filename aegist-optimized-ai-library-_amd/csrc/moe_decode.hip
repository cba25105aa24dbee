// The 4-bit SwiGLU experts at decode batches (hybrid.py:608-628 for a handful of tokens; engine
// moe_gu_* / moe_dn_*, hybrid.cu:386-558): few picks, each of its own expert or nearly so, so the
// op is a stream of the touched experts' rows from HBM (1.77 MB each at 2048 x 512).
//
// Tiles of 16 rows against 16 columns on v_mfma_f32_16x16x32_bf16, where the columns are not 16 picks
// (there are one or two) but 4 picks x 2 parts of the activation (bf16 hi, lo) x 2 quantisation groups:
// a lane loads 16 bytes (32 codes) of a row, 4 lanes of a row a run of 128 codes = two 64-groups, and
// each of the run's 4 products mixes codes of both groups; a column whose group a lane's codes do not
// belong to reads zeros there. So a load covers 64 consecutive bytes of 16 rows (32 in the form that
// keeps a product within one group), one product per 8 codes and lane serves up to 4 picks with both
// parts, and the scale and min of a group are applied to 4 values per lane:
//   y += s sum (128 + c) x + (m - 128 s) sum x, per group and part, the parts and groups added last,
// the same fp32 formula as moe.hip's tiles. Row scales and activation parts are staged in LDS once per
// workgroup; codes stream through registers, 4 runs (8 KB per wave) in flight.
//
// No grouping launch: a workgroup belongs to one pick, finds the other picks of its expert among
// all picks by ballots, and works for up to MDP of them at once (weights read once for all) if it is
// the first of its four, or exits. Results do not depend on which picks share a workgroup: every
// pick's sums run in the same order whatever the company.
//
// Measured (experts and combine, one launch sequence in a graph): batch 1 41 -> 17 us, batch 16
// (105 experts, 186 MB) 128 -> 49 us, batch 64 (223 experts) 228 -> 125 us. A VALU form (whole-row loads,
// fp32 dot products) was as fast at batch 1 and 91 against 44 us at batch 16: without packed fp32
// it needs three vector instructions per code.
#include "common.h"

#include <type_traits>

using namespace aegist;

namespace {

constexpr int MDP = 4;       // picks per workgroup
constexpr int kMaxPicks = 512;

typedef uint32_t u4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float h2f(uint16_t h) { return (float)__builtin_bit_cast(_Float16, h); }

// Loads through addresses taken from the pointer table: in the global address space, so they do
// not count against the LDS wait counter as flat loads would.
template <typename T>
__device__ __forceinline__ T ld_global(const void* p) {
    return *(const __attribute__((address_space(1))) T*)p;
}

// Picks that share a workgroup: those of pick i's expert, in pick order, cut into fours; the first of
// each four works. Returns how many picks this workgroup has (0: none, exit), mem[0 .. n) in pick
// order. Every thread of the workgroup gets the same answer.
__device__ __forceinline__ int pick_group(const int* __restrict__ idx, int N, int i, int E, int* mem, int* expert) {
    __shared__ unsigned long long mask[kMaxPicks / WAVE];
    const int tid = threadIdx.x, e = idx[i];
    for (int j = tid; j < kMaxPicks; j += blockDim.x) {
        const unsigned long long m = __ballot(j < N && idx[min(j, N - 1)] == e);
        if (tid % WAVE == 0) mask[j / WAVE] = m;
    }
    __syncthreads();
    *expert = e;
    if (e < 0 || e >= E) return 0;  // dropped: adds nothing
    int rank = 0;
    const int wi = i / WAVE, bi = i % WAVE;
    for (int w = 0; w < wi; w++) rank += __popcll(mask[w]);
    rank += __popcll(mask[wi] & ((1ull << bi) - 1));
    if (rank % MDP) return 0;
    int n = 0;
    unsigned long long m = mask[wi] & ~((1ull << bi) - 1);
    for (int w = wi; w < (N + WAVE - 1) / WAVE; w++) {
        if (w > wi) m = mask[w];
        while (m && n < MDP) {
            mem[n++] = w * WAVE + __builtin_ctzll(m);
            m &= m - 1;
        }
    }
    return n;
}

// bf16 pairs (c_j, c_{j + 4}) + 128 from a dword of 8 4-bit codes: one and-or per pair (the mask in a
// scalar, the exponent bits in a vector register: the instruction takes no literals)
__device__ __forceinline__ bf16x8 codes_bf16(uint32_t p, uint32_t mask, uint32_t magic) {
    u4v d;
#pragma unroll
    for (int j = 0; j < 4; j++) d[j] = ((p >> (4 * j)) & mask) | magic;
    return __builtin_bit_cast(bf16x8, d);
}

// 8 activations as bf16 hi (truncated) and lo (rounded remainder) in the order of codes_bf16
// (v0 v4 v1 v5 v2 v6 v3 v7), and the sums of the parts
__device__ __forceinline__ void split8(const float* v, uint4& hi, uint4& lo, float& sh, float& sl) {
    uint32_t H[4], L[4];
    sh = sl = 0.f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const float a = v[j], b = v[j + 4];
        const uint32_t ua = __float_as_uint(a) & 0xffff0000u, ub = __float_as_uint(b) & 0xffff0000u;
        H[j] = (ua >> 16) | ub;
        L[j] = f2bf2(a - __uint_as_float(ua), b - __uint_as_float(ub));
        sh += __uint_as_float(ua) + __uint_as_float(ub);
        sl += bf_lo(L[j]) + bf_hi(L[j]);
    }
    hi = uint4{H[0], H[1], H[2], H[3]};
    lo = uint4{L[0], L[1], L[2], L[3]};
}

// LDS of a workgroup for rows of Kd codes, `rows` scale rows per wave: the picks' activation parts
// (row 4 part + pick, padded by 16 bytes so that the 8 rows of a read lie in different banks), 64
// bytes of zeros, the part sums [chunk][16 columns], the waves' (s, m) fp16 pairs [row][group + 1].
__host__ __device__ constexpr int x_stride(int Kd) { return 2 * Kd + 16; }
__host__ __device__ constexpr int lds_sum(int Kd) { return 2 * MDP * x_stride(Kd) + 64; }
__host__ __device__ constexpr int lds_scale(int Kd) { return lds_sum(Kd) + Kd / 128 * 64; }
__host__ __device__ constexpr int lds_bytes(int Kd, int rows, int waves) {
    return lds_scale(Kd) + waves * rows * (Kd / 64 + 1) * 4;
}

// kGu: gate / up, act[pick][u] = silu(gate_u . x) (up_u . x) for 16 units per pair of row tiles (Kd = D).
// Otherwise down, out[pick][o] = wts[pick] (dn_o . act[pick]) for 32 outputs per pair (Kd = I).
// Grid (N picks, row blocks), NW waves of npair pairs each; src: the picks' fp32 inputs (h of the
// pick's token, act of the pick).
template <bool kGu, int NW, int npair, int Kd, int OCC>
__global__ void __launch_bounds__(64 * NW, OCC) moe_decode_kernel(
    const float* __restrict__ src, const unsigned long long* __restrict__ eptr, const int* __restrict__ idx,
    const float* __restrict__ wts, int N, int K, int E, int rows, long long off_q, long long off_s,
    long long off_m, float* __restrict__ out) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    int mem[MDP], e;
    const int np = pick_group(idx, N, blockIdx.x, E, mem, &e);
    if (np == 0) return;
    const unsigned char* base = (const unsigned char*)eptr[e];
    const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int n = lane % 16, g = lane / 16;
    constexpr int G = Kd / 64, nch = Kd / 128;
    constexpr int kUnit = kGu ? 16 : 32;  // outputs per pair
    const int o0 = (blockIdx.y * NW + wave) * npair * kUnit;
    const int nw = min(npair, max(0, rows - o0) / kUnit);  // this wave's pairs: rows is a multiple of a pair

    // codes: tile t of pair pr, chunk c: row0 + lane % 16, bytes 64 c + 16 (lane / 16); one load
    // covers 64 consecutive bytes of 16 rows
    auto row0 = [&](int pr, int t) { return kGu ? t * rows + o0 + 16 * pr : o0 + 32 * pr + 16 * t; };
    auto load = [&](int pr, int t, int c) {
        return ld_global<u4v>(base + off_q + ((unsigned)(row0(pr, t) + n) * (Kd / 2) + 64 * c + 16 * g));
    };
    constexpr int PD = 4;  // chunks in flight
    u4v q[PD][2];
    if (nw > 0) {
#pragma unroll
        for (int u = 0; u < PD; u++)
#pragma unroll
            for (int t = 0; t < 2; t++) q[u][t] = load(0, t, u);
    }
    // scales and mins of the wave's rows: every 16 rows are one run of 16 G halves, 8 per lane and
    // load; requested here, unpacked after the activations so that both round trips overlap
    uint32_t* sc = (uint32_t*)(lds + lds_scale(Kd)) + wave * npair * 32 * (G + 1);
    constexpr int SP = npair * 4 * G, SI = (SP + WAVE - 1) / WAVE;
    u4v sv[SI], mv[SI];
#pragma unroll
    for (int k = 0; k < SI; k++) {
        const int i = min(lane + WAVE * k, nw * 4 * G - 1), r = 8 * i / G, gr = 8 * i % G;  // LDS row 32 pr + 16 t + ..
        if (nw > 0) {
            const unsigned at = ((row0(r / 32, (r / 16) % 2) + r % 16) * G + gr) * 2;
            sv[k] = ld_global<u4v>(base + off_s + at);
            mv[k] = ld_global<u4v>(base + off_m + at);
        }
    }
    // activations
    for (int i = tid; i < np * (Kd / 8); i += 64 * NW) {
        const int p = i / (Kd / 8), k = i % (Kd / 8);
        const float4* xp = (const float4*)(src + (size_t)(kGu ? mem[p] / K : mem[p]) * Kd + 8 * k);
        const float4 a = xp[0], b = xp[1];
        const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        uint4 hi, lo;
        float sh, sl;
        split8(v, hi, lo, sh, sl);
        *(uint4*)(lds + p * x_stride(Kd) + 16 * k) = hi;
        *(uint4*)(lds + (MDP + p) * x_stride(Kd) + 16 * k) = lo;
#pragma unroll
        for (int o = 1; o < 8; o <<= 1) {  // the 8 threads of a 64-group (Kd / 8 is a multiple of 64)
            sh += __shfl_xor(sh, o, WAVE);
            sl += __shfl_xor(sl, o, WAVE);
        }
        if (k % 8 == 0) {
            float* xs = (float*)(lds + lds_sum(Kd)) + k / 16 * 16 + (k / 8 % 2) * 8 + p;
            xs[0] = sh;
            xs[MDP] = sl;
        }
    }
    if (tid < 4) *(uint4*)(lds + 2 * MDP * x_stride(Kd) + 16 * tid) = uint4{0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < SI; k++) {
        const int i = lane + WAVE * k, r = 8 * i / G, gr = 8 * i % G;
        if (i < nw * 4 * G) {
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const uint32_t a = sv[k][e / 2] >> (16 * (e & 1)), b = mv[k][e / 2] >> (16 * (e & 1));
                sc[r * (G + 1) + gr + e] = (a & 0xffffu) | (b << 16);
            }
        }
    }
    lds_barrier();

    // column n: pick n % 4, part (n / 4) % 2, group n / 8 of the chunk: lanes whose codes lie in the
    // other group read zeros
    const bool mine = g / 2 == n / 8;
    const unsigned char* xl = mine ? lds + (n % 8) * x_stride(Kd) + 64 * g : lds + 2 * MDP * x_stride(Kd);
    const int xstep = mine ? 256 : 0;
    const float* xs = (const float*)(lds + lds_sum(Kd)) + n;
    uint32_t magic = 0x43004300u, mask = 0x000F000Fu;
    asm volatile("" : "+v"(magic), "+s"(mask));  // in registers: see codes_bf16
#pragma unroll 1
    for (int pr = 0; pr < nw; pr++) {
        f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
        const uint32_t* scp = sc + (32 * pr + 4 * g) * (G + 1) + n / 8;
#pragma unroll 1
        for (int c0 = 0; c0 < nch; c0 += PD) {
            const bool wrap = c0 + PD >= nch;  // the chunks PD ahead are the next pair's first
            const int pn = wrap ? pr + 1 : pr, cn = wrap ? 0 : c0 + PD;
            const bool more = pn < nw;
#pragma unroll
            for (int u = 0; u < PD; u++) {
                const int c = c0 + u;
                bf16x8 x[4];
#pragma unroll
                for (int j = 0; j < 4; j++) x[j] = *(const bf16x8*)(xl + c * xstep + 16 * j);
                const float X = xs[16 * c];
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    f32x4 P{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        P = __builtin_amdgcn_mfma_f32_16x16x32_bf16(codes_bf16(q[u][t][j], mask, magic), x[j], P, 0, 0, 0);
                    if (more) q[u][t] = load(pn, t, cn + u);
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const uint32_t w = scp[(16 * t + j) * (G + 1) + 2 * c];
                        const float s = h2f((uint16_t)w), m = h2f((uint16_t)(w >> 16));
                        acc[t][j] = fmaf(s, P[j], fmaf(fmaf(-128.f, s, m), X, acc[t][j]));
                    }
                }
            }
        }
        // the four columns of a pick (two groups, two parts)
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                float v = acc[t][j];
                v += __shfl_xor(v, 4, WAVE);
                acc[t][j] = v + lane_xor<8>(v);
            }
        if (n < np) {
            int mp = mem[0];
#pragma unroll
            for (int i = 1; i < MDP; i++) mp = n == i ? mem[i] : mp;
            float* o = out + (size_t)mp * rows + o0 + kUnit * pr + 4 * g;
            if constexpr (kGu) {
                *(float4*)o = float4{silu_f(acc[0][0]) * acc[1][0], silu_f(acc[0][1]) * acc[1][1],
                                     silu_f(acc[0][2]) * acc[1][2], silu_f(acc[0][3]) * acc[1][3]};
            } else {
                const float w = wts[mp];
#pragma unroll
                for (int t = 0; t < 2; t++)
                    *(float4*)(o + 16 * t) = float4{w * acc[t][0], w * acc[t][1], w * acc[t][2], w * acc[t][3]};
            }
        }
    }
}

bool row_fits(int n) { return n == 512 || n == 1024 || n == 2048; }

template <bool kGu, int NW, int npair, int OCC>
int launch(const float* src, const unsigned long long* eptr, const int* idx, const float* wts, int N, int K, int E, int Kd,
           int rows, long long q, long long s, long long m, float* out, hipStream_t st) {
    constexpr int per = NW * npair * (kGu ? 16 : 32);
    const dim3 grid(N, (rows + per - 1) / per);
#define AEG_KD(KD)                                                                                             \
    if (Kd == KD)                                                                                              \
        moe_decode_kernel<kGu, NW, npair, KD, OCC><<<grid, 64 * NW, lds_bytes(KD, 32 * npair, NW), st>>>(          \
            src, eptr, idx, wts, N, K, E, rows, q, s, m, out);
    AEG_KD(512) AEG_KD(1024) AEG_KD(2048)
#undef AEG_KD
    return after_launch(kGu ? "moe_decode_gate_up" : "moe_decode_down");
}

}  // namespace

namespace aegist {

// Whether the decode kernels take the batch: up to 512 picks, at most two per expert on average
// (beyond that the MFMA tiles of moe.hip read each expert once for more picks), row lengths
// of whole rounds of 4 chunks of 128 codes. The host does not know which experts were picked: where all tokens
// pick the same ones, an expert's picks go four to a workgroup, and the call takes about as long as for experts
// drawn alike (2048 x 512, 8 of 256 experts, 64 tokens: 134 and 124 us; the tiles of moe.hip 61 and 204).
bool moe_decode_fits(int T, int D, int I, int E, int K) {
    const long long N = (long long)T * K;
    return N <= kMaxPicks && N <= 2LL * E && row_fits(D) && row_fits(I);
}

int launch_moe_decode(const float* h, const unsigned long long* eptr, const int* idx, const float* wts, int T, int D,
                      int I, int E, int K, long long gu_s, long long gu_m, long long dn_q, long long dn_s,
                      long long dn_m, float* act, float* ypick, hipStream_t st) {
    const int N = T * K;
    // gate / up: two pairs of row tiles per wave once there are enough workgroups (batch 16: 2 us less
    // than one pair; 8 waves or 2 waves per workgroup 2 to 9 us more); down: one pair (two or four
    // leave too few waves in flight: batch 16, 11 and 28 us more)
    const int rc = N > 64 ? launch<true, 4, 2, 3>(h, eptr, idx, wts, N, K, E, D, I, 0, gu_s, gu_m, act, st)
                          : launch<true, 4, 1, 3>(h, eptr, idx, wts, N, K, E, D, I, 0, gu_s, gu_m, act, st);
    return rc ? rc : launch<false, 4, 1, 3>(act, eptr, idx, wts, N, K, E, I, D, dn_q, dn_s, dn_m, ypick, st);
}

}  // namespace aegist
