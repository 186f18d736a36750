// fp32 GQA prefill on the matrix cores (D = 64, blocks of 64 or 32 keys, up to
// 16 query heads per KV head): block-sparse lists, or no lists (dense).
//
// One workgroup of 4 wavefronts per (sequence b, KV head g, tile of 16 / R
// consecutive query tokens): the tile's tokens x R heads are the 16 columns of
// v_mfma_f32_16x16x4_f32 (column c -> token c / R, head c % R). The workgroup
// forms the union of the tokens' lists in LDS, each entry with the mask of the
// tokens that listed the block, and its wavefronts take the entries in turn
// (u = w, w + 4, ...), each with its own running (m, l, O); the four partials
// are merged in wavefront order at the end, so the result does not depend on
// timing. Per entry
//     S^T[key, col] = K[key, :] . Q[col, :]      (BS MFMA)
//     P = exp2(S scale log2 e - m[col]), fp32     (masked by list, causality, length)
//     O^T[d, col] += V^T[d, key] . P^T[key, col]  (BS MFMA)
// K and V go straight from memory to the operand registers: lane l of the K
// operand holds dims 16 (l / 16) .. +15 of key l % 16 (any order of the
// contraction serves, as Q's is the same), and row r of O^T tile t is dim
// 4 r + t, so that a lane's four V operands of a key are one 16-byte load and
// its 16 outputs are consecutive. The score layout of the product is already the
// operand layout of P, so nothing passes through LDS.
//
// Bound by the fp32 matrix rate (32 cycles an MFMA, 128 of them an entry at
// BS = 64) and, for short prompts, by the latency of a wavefront's few entries:
// hence four wavefronts per tile rather than more columns per wavefront. The
// VALU kernel it stands in for served one token per workgroup through LDS: a
// layer of T=1024, 12/4 heads, top-8 of 64-key blocks (compressor and router
// included) 206 us then, 47 us now; T=2048 420 and 102 (the attention 38 and 92).
//
// A masked column's P is 0, but 0 x V is NaN where V is infinite or NaN: an
// entry whose V holds such values is added token by token, with the rows that
// a token may not attend cleared.
#include "common.h"
#include "kernels.h"
#include "mfma.h"

namespace sparda {

namespace {

constexpr int kFWaves = 4;
constexpr int kFThreads = kFWaves * kWave;
constexpr int kFMaxNB = 2048;                       // KV blocks a token mask array covers
constexpr float kFLog2e = 1.4426950408889634f;

struct F32Merge {
    float o[kFWaves - 1][16][kWave];
    float m[kFWaves - 1][kWave], l[kFWaves - 1][kWave];
};
struct F32Smem {
    union {
        uint32_t mask[kFMaxNB];                     // tokens that listed block j (set-up)
        F32Merge mg;                                // the later wavefronts' partials (after the walk)
    };
    uint32_t ent[kFMaxNB];                          // block << 16 | token mask
    int n_ent;
};

}  // namespace

template <int BS>
__global__ void __launch_bounds__(kFThreads, 2)
prefill_f32_kernel(const float* __restrict__ q, int64_t q_sb, int64_t q_st, int64_t q_sh,
                   const float* __restrict__ k, const float* __restrict__ v, int64_t kv_sb, int64_t kv_st,
                   int64_t kv_sh, const int32_t* __restrict__ sel, const int32_t* __restrict__ n_sel, int cap,
                   int64_t T, int H, int R, int64_t NT, int causal, float scale_log2, float* __restrict__ out,
                   int64_t out_sb, int64_t out_st) {
    constexpr int kSub = BS / 16;                   // 16-key sub-tiles of a block
    __shared__ F32Smem sm;
    const int tid = threadIdx.x;
    const int lane = tid % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int col16 = lane % 16;
    const int grp = lane / 16;
    // latest (heaviest) tiles first
    const int64_t BH = static_cast<int64_t>(gridDim.x) / NT;
    const int64_t bg = blockIdx.x % BH;
    const int b = static_cast<int>(bg / H);
    const int g = static_cast<int>(bg % H);
    const int tpt = 16 / R;                         // tokens per tile
    const int64_t t0 = (NT - 1 - blockIdx.x / BH) * tpt;
    const int nt = static_cast<int>(T - t0 < tpt ? T - t0 : tpt);
    const int64_t NB = cdiv(T, BS);
    const int jmax = static_cast<int>(causal ? (t0 + nt - 1) / BS : NB - 1);
    const float* kbase = k + b * kv_sb + static_cast<int64_t>(g) * kv_sh;
    const float* vbase = v + b * kv_sb + static_cast<int64_t>(g) * kv_sh;

    // this lane's column; columns past the tile's tokens repeat its first one, masked
    const bool live = col16 / R < nt && col16 / R < tpt;
    const int tk = live ? col16 / R : 0;
    const int hh = live ? col16 % R : 0;
    const int64_t t = t0 + tk;
    const int64_t key_end = causal ? t + 1 : T;     // keys [0, key_end) are allowed
    float qr[16];
    {
        const float4* qp = reinterpret_cast<const float4*>(q + b * q_sb + t * q_st +
                                                           static_cast<int64_t>(g * R + hh) * q_sh + 16 * grp);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float4 w = qp[i];
            qr[4 * i] = w.x; qr[4 * i + 1] = w.y; qr[4 * i + 2] = w.z; qr[4 * i + 3] = w.w;
        }
    }

    // ---- the entries: every block of [0, jmax] without lists, else the union of the tokens' lists ----
    int n_ent = jmax + 1;
    if (sel != nullptr) {
        for (int i = tid; i <= jmax; i += kFThreads) sm.mask[i] = 0u;
        __syncthreads();
        const int64_t row0 = bg * T + t0;
        for (int e = tid; e < nt * cap; e += kFThreads) {
            const int tt = e / cap, i = e - tt * cap;
            const int j = sel[(row0 + tt) * cap + i];
            const int tlim = causal ? static_cast<int>((t0 + tt) / BS) : jmax;  // later blocks hold no allowed key
            if (i < n_sel[row0 + tt] && j >= 0 && j <= tlim) atomicOr(&sm.mask[j], 1u << tt);  // a repeat counts once
        }
        __syncthreads();
        if (wave == 0) {
            int n = 0;
            for (int c0 = 0; c0 <= jmax; c0 += kWave) {
                const int j = c0 + lane;
                const uint32_t mk = j <= jmax ? sm.mask[j] : 0u;
                const uint64_t bal = __ballot(mk != 0u);
                if (mk != 0u)
                    sm.ent[n + __popcll(bal & ((1ull << lane) - 1ull))] = static_cast<uint32_t>(j) << 16 | mk;
                n += __popcll(bal);
            }
            if (lane == 0) sm.n_ent = n;
        }
        __syncthreads();
        n_ent = sm.n_ent;
    }

    const int kv_st32 = static_cast<int>(kv_st);
    // K operand: key 16 n + col16, dims 16 grp .. +15. Rows past T read row T-1 (masked).
    typedef float F16 __attribute__((ext_vector_type(16)));
    auto load_k = [&](int j, F16 (&kr)[kSub]) __attribute__((always_inline)) {
        // uniform block base, 32-bit lane offsets (checked by the host)
        const int64_t r0 = static_cast<int64_t>(j) * BS;
        const int last = static_cast<int>(T - 1 - r0 < BS - 1 ? T - 1 - r0 : BS - 1);
        const float* kb = kbase + r0 * kv_st;
#pragma unroll
        for (int n = 0; n < kSub; ++n) {
            const int r = 16 * n + col16 < last ? 16 * n + col16 : last;
            const float4* p = reinterpret_cast<const float4*>(kb + static_cast<uint32_t>(r * kv_st32 + 16 * grp));
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float4 w = p[i];
                kr[n][4 * i] = w.x; kr[n][4 * i + 1] = w.y; kr[n][4 * i + 2] = w.z; kr[n][4 * i + 3] = w.w;
            }
        }
    };
    auto entry = [&](int u, int& j, uint32_t& mk) __attribute__((always_inline)) {
        if (sel != nullptr) {
            const uint32_t e = __builtin_amdgcn_readfirstlane(static_cast<int>(sm.ent[u]));
            j = static_cast<int>(e >> 16);
            mk = e & 0xffffu;
        } else {
            j = u;
            mk = 0xffffu;
        }
    };

    float m = -__builtin_inff(), l = 0.0f;          // the column's running maximum (log2 units); this lane's part of its sum
    f32x4 o[4];
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    F16 kr[kSub];
    int j = 0;
    uint32_t mk = 0;
    if (wave < n_ent) {
        entry(wave, j, mk);
        load_k(j, kr);
    }
    for (int u = wave; u < n_ent; u += kFWaves) {   // wave-uniform
        const int64_t r0 = static_cast<int64_t>(j) * BS;
        // V operands: key 16 n + 4 grp + i, dims 4 col16 .. +3
        f32x4 vr[kSub][4];
        const int last = static_cast<int>(T - 1 - r0 < BS - 1 ? T - 1 - r0 : BS - 1);
        const float* vb = vbase + r0 * kv_st;
#pragma unroll
        for (int n = 0; n < kSub; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int key = 16 * n + 4 * grp + i;
                vr[n][i] = *reinterpret_cast<const f32x4*>(
                    vb + static_cast<uint32_t>((key < last ? key : last) * kv_st32 + 4 * col16));
            }
        f32x4 s[kSub];
#pragma unroll
        for (int n = 0; n < kSub; ++n) s[n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 16; ++e)
#pragma unroll
            for (int n = 0; n < kSub; ++n)
                s[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[n][e], qr[e], s[n], 0, 0, 0);
        const bool listed = live && (mk >> tk & 1u) != 0u;
        const int lim = listed ? static_cast<int>(key_end - r0 < BS ? key_end - r0 : BS) : 0;  // allowed keys of the block
        int jn = 0;
        uint32_t mkn = 0;
        if (u + kFWaves < n_ent) {
            entry(u + kFWaves, jn, mkn);
            load_k(jn, kr);                         // in flight under the softmax and the second product
        }
        float mx = -__builtin_inff();
#pragma unroll
        for (int n = 0; n < kSub; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s[n][i] = 16 * n + 4 * grp + i < lim ? s[n][i] * scale_log2 : -__builtin_inff();
                mx = fmaxf(mx, s[n][i]);
            }
        mx = pair32_max(pair16_max(mx));
        const float m_new = fmaxf(m, mx);
        const float ref = m_new == -__builtin_inff() ? 0.0f : m_new;  // nothing allowed yet: every P is 0
        const float alpha = __builtin_amdgcn_exp2f(m - ref);
        m = m_new;
        l *= alpha;
#pragma unroll
        for (int n = 0; n < kSub; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s[n][i] = __builtin_amdgcn_exp2f(s[n][i] - ref);
                l += s[n][i];
            }
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) o[dt] *= alpha;
        float vm = 0.0f;
#pragma unroll
        for (int n = 0; n < kSub; ++n)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int dt = 0; dt < 4; ++dt) vm = __builtin_elementwise_maximum(vm, __builtin_fabsf(vr[n][i][dt]));
        if (__ballot(!(vm < __builtin_inff())) == 0ull) {
#pragma unroll
            for (int n = 0; n < kSub; ++n)
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int dt = 0; dt < 4; ++dt)
                        o[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(vr[n][i][dt], s[n][i], o[dt], 0, 0, 0);
        } else {
            for (int x = 0; x < nt; ++x) {
                if ((mk >> x & 1u) == 0u) continue;  // wave-uniform
                const int64_t end = (causal ? t0 + x + 1 : T) - r0;
                f32x4 d[4];
#pragma unroll
                for (int dt = 0; dt < 4; ++dt) d[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int n = 0; n < kSub; ++n)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int dt = 0; dt < 4; ++dt)
                            d[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                                16 * n + 4 * grp + i < end ? vr[n][i][dt] : 0.0f, s[n][i], d[dt], 0, 0, 0);
#pragma unroll
                for (int dt = 0; dt < 4; ++dt)
                    if (live && tk == x) o[dt] += d[dt];
            }
        }
        j = jn;
        mk = mkn;
    }
    l = pair32_sum(pair16_sum(l));

    // ---- merge the wavefronts' partials, in order ----
    if (wave > 0) {
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i) sm.mg.o[wave - 1][4 * i + dt][lane] = o[dt][i];
        sm.mg.m[wave - 1][lane] = m;
        sm.mg.l[wave - 1][lane] = l;
    }
    __syncthreads();
    if (wave > 0) return;
    float M = m;
#pragma unroll
    for (int w = 0; w < kFWaves - 1; ++w) M = fmaxf(M, sm.mg.m[w][lane]);
    const float ref = M == -__builtin_inff() ? 0.0f : M;
    float wt = __builtin_amdgcn_exp2f(m - ref);
    l *= wt;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) o[dt] *= wt;
#pragma unroll
    for (int w = 0; w < kFWaves - 1; ++w) {
        wt = __builtin_amdgcn_exp2f(sm.mg.m[w][lane] - ref);
        l = __builtin_fmaf(wt, sm.mg.l[w][lane], l);
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
#pragma unroll
            for (int i = 0; i < 4; ++i) o[dt][i] = __builtin_fmaf(wt, sm.mg.o[w][4 * i + dt][lane], o[dt][i]);
    }
    if (!live) return;
    const float inv = 1.0f / l;
    float4* op = reinterpret_cast<float4*>(out + b * out_sb + t * out_st + static_cast<int64_t>(g * R + hh) * 64 + 16 * grp);
#pragma unroll
    for (int i = 0; i < 4; ++i) op[i] = make_float4(o[0][i] * inv, o[1][i] * inv, o[2][i] * inv, o[3][i] * inv);
}

bool prefill_f32_supported(int dtype, int64_t T, int64_t Hq, int64_t Hkv, int64_t D, int64_t bs, int64_t B,
                           const int32_t* sel, int64_t cap, int64_t q_sb, int64_t q_st, int64_t q_sh, int64_t kv_sb,
                           int64_t kv_st, int64_t kv_sh, int64_t out_sb, int64_t out_st, const void* q,
                           const void* k, const void* v, const void* out) {
    if (dtype != SPARDA_F32 || D != 64 || (bs != 64 && bs != 32) || Hq % Hkv != 0 || Hq / Hkv > 16) return false;
    // short prompts in few workgroups go to the general kernel, which has one
    // memory latency less before its keys and little else to do: us there / here
    // for 6/2 heads, T=1 4.0 / 6.4, T=16 4.9 / 6.8, T=33 6.2 / 7.3, T=64 8.2 / 7.1;
    // 32-key blocks T=16 5.0 / 5.6, T=33 7.2 / 5.7; 16/2 heads T=16 6.5 / 6.9, T=33
    // 8.1 / 7.0; B=64, T=16 9.9 / 8.0.
    if (T * (Hq / Hkv > 4 ? 4 : 1) <= (bs == 64 ? 40 : 16) && B * Hkv * T <= 512) return false;
    // a tile's list entries are counted in 32 bits, its blocks in the mask array
    if (sel != nullptr && (cdiv(T, bs) > kFMaxNB || cap >= (int64_t(1) << 27))) return false;
    if (B * Hkv * cdiv(T, 16 / (Hq / Hkv)) >= (int64_t(1) << 31)) return false;
    if (kv_st < 0 || kv_st >= (int64_t(1) << 22)) return false;  // offsets inside a block are 32-bit, unsigned
    auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    if (!al16(q) || !al16(k) || !al16(v) || !al16(out)) return false;
    return q_sb % 4 == 0 && q_st % 4 == 0 && q_sh % 4 == 0 && kv_sb % 4 == 0 && kv_st % 4 == 0 && kv_sh % 4 == 0 &&
           out_sb % 4 == 0 && out_st % 4 == 0;
}

int launch_prefill_f32(const void* q, int64_t q_sb, int64_t q_st, int64_t q_sh, const void* k, const void* v,
                       int64_t kv_sb, int64_t kv_st, int64_t kv_sh, const int32_t* sel, const int32_t* n_sel,
                       int64_t cap, int64_t B, int64_t T, int64_t Hq, int64_t Hkv, int64_t bs, int causal,
                       float scale, void* out, int64_t out_sb, int64_t out_st, hipStream_t stream) {
    const int64_t R = Hq / Hkv;
    const int64_t NT = cdiv(T, 16 / R);
    dim3 grid(static_cast<unsigned>(B * Hkv * NT));
#define SPARDA_F32K(BS_)                                                                                    \
    hipLaunchKernelGGL((prefill_f32_kernel<BS_>), grid, dim3(kFThreads), 0, stream,                         \
                       static_cast<const float*>(q), q_sb, q_st, q_sh, static_cast<const float*>(k),        \
                       static_cast<const float*>(v), kv_sb, kv_st, kv_sh, sel, n_sel, static_cast<int>(cap), \
                       T, static_cast<int>(Hkv), static_cast<int>(R), NT, causal, scale * kFLog2e,          \
                       static_cast<float*>(out), out_sb, out_st)
    if (bs == 64) SPARDA_F32K(64);
    else SPARDA_F32K(32);
#undef SPARDA_F32K
    return check_hip(hipGetLastError(), "prefill_f32_kernel");
}

}  // namespace sparda
