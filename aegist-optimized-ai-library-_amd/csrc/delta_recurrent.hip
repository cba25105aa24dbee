// Gated delta rule, token by token (the recurrent form), for short sequences and the
// correctness configuration: S *= e^g; kv = S^T k; delta = (v - kv) beta; S += k delta^T;
// o = S^T q (hybrid.py:318-324 looped; the engine's delta_scan, hybrid.cu:240-300).
//
// The columns of S evolve independently (column j only needs k, q, v_j), so the work is split
// by column block: one wave64 per (sequence, value head, block of 8 or 16 columns) holds 128 x 8 or
// 128 x 16 of the state in VGPRs (16 or 32 rows x 1 column per lane) for the whole sequence. B = 1 with 32
// value heads gives 512 or 256 waves instead of the 32 workgroups of a head-per-block scan.
//
// Latency-bound: one wave's chain per token. Both column sums are taken over the old state (S^T k and
// S^T q), so the output does not wait for the update: o = e^g S^T q + (k . q) delta. Everything that
// does not depend on the state runs a token ahead, beside the sums: the norms (DPP sums instead of
// LDS permutes), q and k staged in the wave's own LDS (no workgroup barrier, which also waited for the
// prefetch of the next token's inputs), the loads two tokens ahead. In the layer stack 37 tokens, 32 heads, batch 1:
// 44 -> 36 us.
#include "common.h"

using namespace aegist;

namespace {

constexpr int D = 128;

struct SeqArgs {
    long long sb_qk, st_qk, sh_qk, sb_v, st_v, sh_v, sb_o, st_o, sh_o;
    long long sb_g, st_g;  // g / beta strides by sequence and token (value head contiguous)
};

template <typename Tin, typename Tout, int CB>  // CB: columns per workgroup (one wave), 8 or 16
__global__ void __launch_bounds__(64) delta_recurrent_kernel(const Tin* __restrict__ q, const Tin* __restrict__ k,
                                                             const Tin* __restrict__ v, const float* __restrict__ g,
                                                             const float* __restrict__ beta, float* __restrict__ state,
                                                             Tout* __restrict__ out, SeqArgs a, int T, int HK, int HV,
                                                             int normalize, float qscale, float eps) {
    constexpr int RPL = D * CB / WAVE;  // state rows per lane
    __shared__ __attribute__((aligned(16))) float sk[2][D], sq[2][D];  // wave-private, two tokens
    const int cb = blockIdx.x, hv = blockIdx.y, b = blockIdx.z, lane = threadIdx.x;
    const int c = lane % CB, rg = lane / CB;  // column within block, row group (RPL rows)
    const int col = cb * CB + c;
    const int kh = hv / (HV / HK);
    float* S = state ? state + ((size_t)b * HV + hv) * D * D : nullptr;

    float s[RPL];
#pragma unroll
    for (int r = 0; r < RPL; r++) s[r] = S ? S[(size_t)(rg * RPL + r) * D + col] : 0.f;

    const Tin* qb = q + b * a.sb_qk + kh * a.sh_qk;
    const Tin* kb = k + b * a.sb_qk + kh * a.sh_qk;
    const Tin* vb = v + b * a.sb_v + hv * a.sh_v;
    const float* gb = g + b * a.sb_g + hv;
    const float* bb = beta + b * a.sb_g + hv;

    // registers for the token being prefetched
    float nq0 = 0.f, nq1 = 0.f, nk0 = 0.f, nk1 = 0.f, nv = 0.f, ng = 0.f, nb = 0.f;
    auto fetch = [&](int t) {
        nq0 = Act<Tin>::ld(qb, t * a.st_qk + lane);
        nq1 = Act<Tin>::ld(qb, t * a.st_qk + lane + 64);
        nk0 = Act<Tin>::ld(kb, t * a.st_qk + lane);
        nk1 = Act<Tin>::ld(kb, t * a.st_qk + lane + 64);
        nv = Act<Tin>::ld(vb, t * a.st_v + col);
        ng = gb[t * a.st_g];
        nb = bb[t * a.st_g];
    };
    // the prefetched token's scalars and its normalised q and k (LDS), one token ahead of their use
    float vv = 0.f, decay = 0.f, bt = 0.f, kq = 0.f;
    auto stage = [&](int buf) {
        float q0 = nq0, q1 = nq1, k0 = nk0, k1 = nk1;
        if (normalize) {
            const float rq = rsqrtf(wave_sum_dpp(q0 * q0 + q1 * q1) + eps);
            const float rk = rsqrtf(wave_sum_dpp(k0 * k0 + k1 * k1) + eps);
            q0 = (q0 * rq) * qscale;
            q1 = (q1 * rq) * qscale;
            k0 *= rk;
            k1 *= rk;
        }
        kq = wave_sum_dpp(q0 * k0 + q1 * k1);
        sq[buf][lane] = q0;
        sq[buf][lane + 64] = q1;
        sk[buf][lane] = k0;
        sk[buf][lane + 64] = k1;
        vv = nv;
        decay = expf(ng);
        bt = nb;
    };
    if (T > 0) {
        fetch(0);
        stage(0);
        if (T > 1) fetch(1);
    }
    for (int t = 0; t < T; t++) {
        wave_sync();
        float kr[RPL], qr[RPL];
#pragma unroll
        for (int r = 0; r < RPL; r += 4) {
            const float4 x = *(const float4*)&sk[t & 1][rg * RPL + r], y = *(const float4*)&sq[t & 1][rg * RPL + r];
            kr[r] = x.x; kr[r + 1] = x.y; kr[r + 2] = x.z; kr[r + 3] = x.w;
            qr[r] = y.x; qr[r + 1] = y.y; qr[r + 2] = y.z; qr[r + 3] = y.w;
        }
        const float cv = vv, cd = decay, cbt = bt, ckq = kq;
        // the next token is normalised and staged, and the one after it requested, beside this
        // token's sums
        if (t + 1 < T) {
            stage((t + 1) & 1);
            if (t + 2 < T) fetch(t + 2);
        }
        // both column sums over the old state: S^T k and S^T q, so that the output does not wait for
        // the update: o = e^g S^T q + (k . q) delta
        float pk[2] = {0.f, 0.f}, pq[2] = {0.f, 0.f};
#pragma unroll
        for (int r = 0; r < RPL; r++) {
            pk[r & 1] = fmaf(s[r], kr[r], pk[r & 1]);
            pq[r & 1] = fmaf(s[r], qr[r], pq[r & 1]);
        }
        float SK = pk[0] + pk[1], SQ = pq[0] + pq[1];
        if constexpr (CB == 8) {
            SK += lane_xor<8>(SK);
            SQ += lane_xor<8>(SQ);
        }
        SK = pair_sum32(pair_sum16(SK));
        SQ = pair_sum32(pair_sum16(SQ));
        const float delta = (cv - cd * SK) * cbt;
#pragma unroll
        for (int r = 0; r < RPL; r++) s[r] = fmaf(kr[r], delta, cd * s[r]);
        if (rg == 0) Act<Tout>::st(out, b * a.sb_o + t * a.st_o + hv * a.sh_o + col, fmaf(ckq, delta, cd * SQ));
    }
    if (S) {
#pragma unroll
        for (int r = 0; r < RPL; r++) S[(size_t)(rg * RPL + r) * D + col] = s[r];
    }
}

// Blocks of 8 columns shorten a token's chain, but read and write the state in pieces of 32 bytes instead of 64
// and stage q and k twice as often: they pay for few heads over many tokens. Measured (fp32, us, 16 and 8
// columns): 32 heads 1 token 6.0, 7.4; 12 18.1, 18.5; 16 22.6, 21.9; 63 66, 61; 64 heads 24 32.8, 34.8; 63 69, 65;
// 128 heads 37 49.0, 48.8; 63 73.7, 72.2; 256 heads 63 83, 102; 2048 heads 1 token 65.8, 132. (The first form, 16 columns
// with two barriers a token, took 6.2, 20.9, 25.8, 78; 38, 82; 55, 86; 89 and 65.5 us.)
constexpr bool narrow_columns(long long heads, int T) { return heads <= 128 && 2LL * T >= heads; }
static_assert(!narrow_columns(64 * 32, 1) && !narrow_columns(32, 1) && narrow_columns(32, 37) && !narrow_columns(256, 200),
              "a step of many heads takes 16 columns");

template <typename Tin, typename Tout>
int launch2(const void* q, const void* k, const void* v, const float* g, const float* beta, float* state, void* out,
            const SeqArgs& a, int B, int T, int HK, int HV, int normalize, float qscale, float eps, hipStream_t st) {
    if (narrow_columns((long long)B * HV, T))
        delta_recurrent_kernel<Tin, Tout, 8><<<dim3(D / 8, HV, B), 64, 0, st>>>(
            (const Tin*)q, (const Tin*)k, (const Tin*)v, g, beta, state, (Tout*)out, a, T, HK, HV, normalize, qscale, eps);
    else
        delta_recurrent_kernel<Tin, Tout, 16><<<dim3(D / 16, HV, B), 64, 0, st>>>(
            (const Tin*)q, (const Tin*)k, (const Tin*)v, g, beta, state, (Tout*)out, a, T, HK, HV, normalize, qscale, eps);
    return after_launch("delta_recurrent");
}

}  // namespace

namespace aegist {
int launch_delta_recurrent(const void* q, const void* k, const void* v, int in_dtype, long long sb_qk, long long st_qk,
                           long long sh_qk, long long sb_v, long long st_v, long long sh_v, const float* g,
                           const float* beta, float* state, void* out, int out_dtype, long long sb_o, long long st_o,
                           long long sh_o, int B, int T, int HK, int HV, int normalize, float qscale, float eps,
                           hipStream_t st) {
    if (B < 0 || T < 0 || HK <= 0 || HV <= 0 || HV % HK) return fail(AEGIST_ERR_SHAPE, "delta_recurrent: need HV % HK == 0");
    if (B == 0) return 0;
    if (T == 0) return 0;
    SeqArgs a{sb_qk, st_qk, sh_qk, sb_v, st_v, sh_v, sb_o, st_o, sh_o, (long long)T * HV, HV};
    if (in_dtype == AEGIST_F32 && out_dtype == AEGIST_F32)
        return launch2<float, float>(q, k, v, g, beta, state, out, a, B, T, HK, HV, normalize, qscale, eps, st);
    if (in_dtype == AEGIST_F32 && out_dtype == AEGIST_BF16)
        return launch2<float, uint16_t>(q, k, v, g, beta, state, out, a, B, T, HK, HV, normalize, qscale, eps, st);
    if (in_dtype == AEGIST_BF16 && out_dtype == AEGIST_F32)
        return launch2<uint16_t, float>(q, k, v, g, beta, state, out, a, B, T, HK, HV, normalize, qscale, eps, st);
    if (in_dtype == AEGIST_BF16 && out_dtype == AEGIST_BF16)
        return launch2<uint16_t, uint16_t>(q, k, v, g, beta, state, out, a, B, T, HK, HV, normalize, qscale, eps, st);
    return fail(AEGIST_ERR_DTYPE, "delta_recurrent: dtypes must be AEGIST_F32 or AEGIST_BF16");
}
}  // namespace aegist

extern "C" int aegist_delta_recurrent(const void* q, const void* k, const void* v, int in_dtype, long long sb_qk,
                                      long long st_qk, long long sh_qk, long long sb_v, long long st_v, long long sh_v,
                                      const float* g, const float* beta, float* state, void* out, int out_dtype,
                                      long long sb_o, long long st_o, long long sh_o, int B, int T, int HK, int HV,
                                      int normalize, float qscale, float eps, void* stream) {
    return launch_delta_recurrent(q, k, v, in_dtype, sb_qk, st_qk, sh_qk, sb_v, st_v, sh_v, g, beta, state, out,
                                  out_dtype, sb_o, st_o, sh_o, B, T, HK, HV, normalize, qscale, eps,
                                  AEG_STREAM(stream));
}

// Engine mirror: y [T, C] fp32 rows q | k | v (already L2-normalised), gb [T, 2HV] (g, then
// beta), state [HV, 128, 128], o [T, HV, 128]. Sequences of 64+ tokens take the chunked path.
namespace aegist {
size_t delta_scan_chunked_ws_bytes(int T, int HK, int HV);
int delta_scan_chunked(const float* y, const float* gb, float* state, float* o, int T, int C, int HK, int HV,
                       void* ws, size_t ws_bytes,
                       hipStream_t st);
}

extern "C" size_t aegist_delta_scan_workspace_bytes(int T, int HK, int HV) {
    if (T < 64 || HK <= 0 || HV <= 0) return 0;
    return delta_scan_chunked_ws_bytes(T, HK, HV);
}

extern "C" int aegist_delta_scan_ws(const float* y, const float* gb, float* state, float* o, int T, int C, int HK,
                                    int HV, void* ws, size_t ws_bytes, void* stream) {
    if (T < 0 || HK <= 0 || HV <= 0 || HV % HK || C != 2 * HK * D + HV * D)
        return fail(AEGIST_ERR_SHAPE, "delta_scan: need C == 2*HK*128 + HV*128 and HV % HK == 0");
    if (T == 0) return 0;
    hipStream_t st = AEG_STREAM(stream);
    if (T >= 64) {
        int rc = check_workspace(ws, ws_bytes, delta_scan_chunked_ws_bytes(T, HK, HV), "delta_scan");
        if (rc) return rc;
        return delta_scan_chunked(y, gb, state, o, T, C, HK, HV, ws, ws_bytes, st);
    }
    // g and beta are interleaved per token in gb: present them through the strided kernel
    // by pointing g at gb and beta at gb + HV with a token stride of 2*HV.
    SeqArgs a{0, C, D, 0, C, D, 0, (long long)HV * D, D, 0, 2 * HV};
    return launch2<float, float>(y, y + (size_t)HK * D, y + (size_t)2 * HK * D, gb, gb + HV, state, o, a, 1, T, HK, HV, 0,
                                 1.f, 0.f, st);
}

// The reference signature (no workspace argument): T >= 64 takes the workspace bound to this
// thread (aegist_bind_workspace).
extern "C" int aegist_delta_scan(const float* y, const float* gb, float* state, float* o, int T, int C, int HK, int HV,
                                 void* stream) {
    size_t bound = 0;
    void* ws = bound_workspace(&bound);
    return aegist_delta_scan_ws(y, gb, state, o, T, C, HK, HV, ws, bound, stream);
}
