// bf16 dense GQA prefill on the gfx950 matrix cores (D = 64), causal or not:
// the reference's dense fallback (model/attention/sparse.py:201-224: layer 0,
// no forecast, or at most two KV blocks) without selection lists.
//
// One workgroup of CW x KG = 8 wavefronts serves one (sequence b, KV head g,
// window of 16 CW query tokens): CW token waves, each with the tokens
// [16w, 16w+16) of the window for all R = Hq/Hkv query heads of the group: 16R
// columns (column c -> token c / R, head c % R), R tiles of 16 columns whose Q
// operands stay in registers; and KG key groups of CW waves, of which group kg
// walks the KV blocks kg, kg + KG, ... of 64 keys in ascending order up to the
// window's last token's block. Each block's K and V are staged once in LDS by
// their group (double-buffered; the next block is loaded into registers while
// the current one is computed) and shared by the window's tokens and R heads.
// The groups share the columns' references, so their O and row sums are added
// at the end, in group order. Where windows are few, small ones times key groups
// keep the number of workgroups well past one per CU, so that the causal triangle
// balances: at B=1, T=8192, 12/4 heads 128 us (800 TFLOP/s) against 231 with one
// group and 128-token windows (256 workgroups, the heaviest twice the mean); where
// they are many, one group stages a block for the most tokens (the launcher's
// rule, with its times). Bound by issue: a wave's
// exponentials and products take turns, so that the matrix cores are busy about
// 40% of the time. Per tile and block, with v_mfma_f32_16x16x32_bf16:
//     S^T[key, col] = K[key, :] . Q[col, :]           (8 MFMA)
//     P = exp2(S * scale log2 e - ref[col]), bf16      (fp32 exponent)
//     O^T[d, col]  += V^T[d, key] . P^T[key, col]      (8 MFMA)
//     l[col]       += 1^T P^T                           (2 MFMA, a ones A operand)
// ref[col] is the column's maximum over block 0 (which every column attends,
// key 0 being allowed to every token), taken when block 0 is computed; later
// blocks take no maxima and never rescale. A score more than 64 log2-units
// above the reference shows as a row sum past 2^64 at the end; the window is
// then walked once for the exact column maxima and again against them (every
// P <= 1).
// A wavefront whose tokens all lie before a block skips it (the causal
// triangle is not computed); the diagonal block masks the keys past each
// column's token. No per-token membership logic: every key up to the token
// (or every key) is attended.
//
// The chunked-gather prefill (model/attention/sparse.py:284-364) runs the same
// kernel with LISTED: one workgroup of 4 wavefronts per query block of 64
// tokens, which builds the block's list in LDS first (chunk.h: {0, own} U the
// union of its rows' non-causal top-k, cut to min(NB, k+2)) and walks the
// listed blocks instead of every block up to the diagonal; all 64 tokens share
// the list, so every tile is full. The first listed block sets the references
// (its key 0 is allowed to every token, since listed blocks never lie past
// the own one).
#include "chunk.h"
#include "common.h"
#include "kernels.h"
#include "mfma.h"

namespace sparda {

namespace {

constexpr int kDBs = 64;                 // keys per KV block
constexpr int kDD = 64;                  // head dim
constexpr int64_t kDCus = 256;           // compute units: one dense workgroup each
constexpr int kLTok = 4;                 // token waves of a listed workgroup (one 64-token query block)
constexpr int kDKRow = kDD + 8;          // K row in LDS, bf16 elements (144 B)
constexpr int kDVRow = kDD + 16;         // V row in LDS, bf16 elements (160 B)
constexpr float kDLog2e = 1.4426950408889634f;
constexpr float kDGuard = 18446744073709551616.0f;  // 2^64: a row sum past it means a score far above ref

template <int KG>
struct DenseStage {
    uint16_t k[2][KG][kDBs * kDKRow];
    uint16_t v[2][KG][kDBs * kDVRow];
};

// partial O and row sums of the KG - 1 later key groups, added into the first
// group's after the walk (lane-linear: every access is one row of 64 lanes)
template <int R, int CW, int KG>
struct DenseMerge {
    f32x4 o[KG - 1][CW][R * 4][kWave];
    float l[KG - 1][CW][R][16];
};
template <int R, int CW>
struct DenseMerge<R, CW, 1> {};

template <int R, int CW, int KG>
struct DenseSmem {
    union {
        DenseStage<KG> st;
        DenseMerge<R, CW, KG> mg;
    };
    int flag;                             // some column's row sum passed kDGuard
    int arrived[KG];                      // waves of a key group past its barriers
};

// the chunked lists' inputs and outputs (LISTED only)
struct ChunkArgs {
    const int32_t* topk;  // [B, Hkv, T, ke] non-causal top-k, or nullptr: the static window
    int ke, k, cut;       // top-k width, top_k, list length cap min(NB, k + 2)
    int32_t* sel;         // optional [B, Hkv, T, cap] / [B, Hkv, T]: the lists as sparda_select_chunked writes them
    int32_t* n_sel;
    int cap;
};

}  // namespace

template <int R, bool LISTED, int CW, int KG>
__global__ void __launch_bounds__(CW * KG * kWave, 2)
prefill_dense_kernel(const uint16_t* __restrict__ q, int64_t q_sb, int64_t q_st, int64_t q_sh,
                     const uint16_t* __restrict__ k, const uint16_t* __restrict__ v, int64_t kv_sb, int64_t kv_st,
                     int64_t kv_sh, int64_t T, int H, int64_t NBq, int causal, float scale_log2,
                     uint16_t* __restrict__ out, int64_t out_sb, int64_t out_st, ChunkArgs ch) {
    constexpr int kThreads = CW * kWave;         // threads of a key group: they stage its block
    constexpr int kWin = 16 * CW;                // query tokens per workgroup
    constexpr int kSR = kDBs * 8 / kThreads;     // 16-byte K (and V) chunks each thread stages per block
    static_assert(!LISTED || (CW == kLTok && KG == 1), "a listed workgroup is one 64-token query block");
    __shared__ DenseSmem<R, CW, KG> sm;
    __shared__ ChunkLds cl;
    const int lane = threadIdx.x % kWave;
    // wave-uniform (scalar registers): the token wave, and the key group, which
    // walks the blocks kg, kg + KG, ...
    const int wv = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
    constexpr bool kOne = KG == 1 && !LISTED;  // (the listed form spills ten registers more with the index folded)
    const int wave = kOne ? wv : wv % CW, kg = kOne ? 0 : wv / CW;
    const int tid = wave * kWave + lane;         // thread within its key group
    const int col16 = lane % 16;
    const int grp = lane / 16;

    // heaviest windows first, XCD-aware when there are few (b, g) pairs
    const int64_t BH = static_cast<int64_t>(gridDim.x) / NBq;
    int64_t bg, qw;
    window_order(blockIdx.x, BH, NBq, bg, qw);
    const int b = static_cast<int>(bg / H);
    const int g = static_cast<int>(bg % H);
    const int64_t t0 = qw * kWin;
    const int64_t NB = cdiv(T, kDBs);
    const int t_valid = static_cast<int>(T - t0 < kWin ? T - t0 : kWin);
    const int64_t w_first = t0 + 16 * wave;  // this wavefront's first token
    int64_t w_last = w_first + 15;
    w_last = w_last < T - 1 ? w_last : T - 1;
    const bool w_live = w_first < T;
    // Q operands of this wavefront's tiles (column col16 of tile tt; rows past T read row T-1)
    int tok[R];
    bf16x8 qreg[R][2];
#pragma unroll
    for (int tt = 0; tt < R; ++tt) {
        const int c = 16 * tt + col16;
        tok[tt] = 16 * wave + c / R;
        int64_t t = t0 + tok[tt];
        t = t < T ? t : T - 1;
        const uint16_t* qp = q + b * q_sb + t * q_st + static_cast<int64_t>(g * R + c % R) * q_sh + 8 * grp;
        qreg[tt][0] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(qp));
        qreg[tt][1] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(qp + 32));
    }

    f32x4 o[R][4], ol[R];
    float ref[R];  // the columns' references, log2 units
    bf16x8 ones_a;
#pragma unroll
    for (int e = 0; e < 8; ++e) ones_a[e] = static_cast<__bf16>(col16 == 0 ? 1.0f : 0.0f);
    auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int tt = 0; tt < R; ++tt) {
            ol[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) o[tt][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    };
    clear();
#pragma unroll
    for (int tt = 0; tt < R; ++tt) ref[tt] = -__builtin_inff();
    if (threadIdx.x < KG) sm.arrived[threadIdx.x] = 0;
    if (threadIdx.x == 0) sm.flag = 0;  // ordered before its uses by the staging barrier

    // staging: thread -> 16-byte chunks (rows tid / 8 + i * kThreads / 8, column
    // tid % 8) of K and of V; rows past T (a ragged last block) read row T-1
    // (finite values, masked)
    const uint16_t* kbase = k + b * kv_sb + static_cast<int64_t>(g) * kv_sh;
    const uint16_t* vbase = v + b * kv_sb + static_cast<int64_t>(g) * kv_sh;
    const int srow = tid / 8, scol = (tid % 8) * 8;
    constexpr int kRowStep = kThreads / 8;
    // the chunks in flight live in one vector register tuple (an array of
    // uint4 handed between the lambdas would be placed in scratch memory)
    typedef unsigned int StageV __attribute__((ext_vector_type(4 * kSR)));
    auto fetch = [&](int j, StageV& kv_k, StageV& kv_v) __attribute__((always_inline)) {
        // dense: the block's base is scalar; listed: the block index comes from LDS and
        // the addresses are formed by lane (1 to 3% faster there, as much slower for dense)
        const int64_t row0 = static_cast<int64_t>(j) * kDBs;
        const int last = static_cast<int>(T - 1 - row0 < kDBs - 1 ? T - 1 - row0 : kDBs - 1);
        const uint16_t* kb = kbase + row0 * kv_st;
        const uint16_t* vb = vbase + row0 * kv_st;
#pragma unroll
        for (int i = 0; i < kSR; ++i) {
            uint4 a, c;
            if constexpr (LISTED) {
                int64_t r = row0 + srow + i * kRowStep;
                r = r < T ? r : T - 1;
                a = *reinterpret_cast<const uint4*>(kbase + r * kv_st + scol);
                c = *reinterpret_cast<const uint4*>(vbase + r * kv_st + scol);
            } else {
                int r = srow + i * kRowStep;
                r = r < last ? r : last;
                a = *reinterpret_cast<const uint4*>(kb + (r * kv_st + scol));
                c = *reinterpret_cast<const uint4*>(vb + (r * kv_st + scol));
            }
            kv_k[4 * i] = a.x; kv_k[4 * i + 1] = a.y; kv_k[4 * i + 2] = a.z; kv_k[4 * i + 3] = a.w;
            kv_v[4 * i] = c.x; kv_v[4 * i + 1] = c.y; kv_v[4 * i + 2] = c.z; kv_v[4 * i + 3] = c.w;
        }
    };
    auto stash = [&](int buf, const StageV& kv_k, const StageV& kv_v) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kSR; ++i) {
            *reinterpret_cast<uint4*>(&sm.st.k[buf][kg][(srow + i * kRowStep) * kDKRow + scol]) =
                uint4{kv_k[4 * i], kv_k[4 * i + 1], kv_k[4 * i + 2], kv_k[4 * i + 3]};
            *reinterpret_cast<uint4*>(&sm.st.v[buf][kg][(srow + i * kRowStep) * kDVRow + scol]) =
                uint4{kv_v[4 * i], kv_v[4 * i + 1], kv_v[4 * i + 2], kv_v[4 * i + 3]};
        }
    };

    // blocks of the workgroup and of this wavefront: dense causal, every block up
    // to the last token's; dense non-causal, every block; listed, the list, built
    // while the Q rows and block 0 (the first entry of every list) are in flight
    int nblk, w_nblk;
    StageV nk0{}, nv0{};
    if constexpr (LISTED) {
        fetch(0, nk0, nv0);
        const int64_t row0 = bg * T + t0;  // (b * Hkv + g) * T + t0
        chunk_list(cl, ch.topk != nullptr ? ch.topk + row0 * ch.ke : nullptr, t_valid, ch.ke, static_cast<int>(qw),
                   ch.k, NB, ch.cut);
        if (ch.sel != nullptr) chunk_write(cl, row0, t_valid, ch.cap, ch.sel, ch.n_sel);
        nblk = cl.m;
        w_nblk = w_live ? nblk : 0;
    } else {
        const int64_t last_tok = t0 + t_valid - 1;
        nblk = static_cast<int>(causal ? last_tok / kDBs + 1 : NB);
        w_nblk = !w_live ? 0 : static_cast<int>(causal ? w_last / kDBs + 1 : NB);
    }
    // the u-th block walked
    auto blk = [&](int u) __attribute__((always_inline)) -> int {
        if constexpr (LISTED) return cl.lst[u];
        else return u;
    };

    // the columns' scores against the first block walked, which every key group
    // takes its references from (one group's slot, read by all)
    auto set_refs = [&](int j) __attribute__((always_inline)) {
        bf16x8 ka[4][2];
#pragma unroll
        for (int n = 0; n < 4; ++n)
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
                ka[n][kk] = lds_read8(&sm.st.k[0][0][(16 * n + col16) * kDKRow + 32 * kk + 8 * grp]);
        const int64_t key0 = static_cast<int64_t>(j) * kDBs;
        const bool edge = causal ? key0 + kDBs - 1 > w_first : key0 + kDBs > T;
#pragma unroll
        for (int tt = 0; tt < R; ++tt) {
            f32x4 s[4];
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                s[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[n][0], qreg[tt][0], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                s[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[n][1], qreg[tt][1], s[n], 0, 0, 0);
            }
            if (edge) {
                const int64_t lim64 = causal ? t0 + tok[tt] - key0 : T - 1 - key0;
                const int lim = static_cast<int>(lim64 < kDBs ? lim64 : kDBs);
#pragma unroll
                for (int n = 0; n < 4; ++n)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (16 * n + 4 * grp + i > lim) s[n][i] = -__builtin_inff();
            }
            ref[tt] = pair32_max(pair16_max(max_acc(s, -__builtin_inff()))) * scale_log2;  // block's column max, log2 units
        }
    };

    // mode 0: P against the references (with one key group the first block
    // walked sets them unless `keep`); mode 1: scores only, the exact column
    // maxima of the group's blocks into ref
    auto compute = [&](int buf, int j, bool first, int mode, bool keep) __attribute__((always_inline)) {
        // K A operands: key 16n + col16, dims 32kk + 8grp .. +7
        bf16x8 ka[4][2];
#pragma unroll
        for (int n = 0; n < 4; ++n)
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
                ka[n][kk] = lds_read8(&sm.st.k[buf][kg][(16 * n + col16) * kDKRow + 32 * kk + 8 * grp]);
        // V^T A operands, read transposed from the row-major tile
        bf16x8 va[4][2];
        if (mode == 0) {
            const int rsub = 4 * grp + col16 / 4;
            const int csub = 4 * (col16 % 4);
#pragma unroll
            for (int dt = 0; dt < 4; ++dt)
#pragma unroll
                for (int m = 0; m < 2; ++m) {
                    const uint16_t* base = &sm.st.v[buf][kg][(32 * m + rsub) * kDVRow + 16 * dt + csub];
                    const i16x4 lo = lds_read_tr(base);
                    const i16x4 hi = lds_read_tr(base + 16 * kDVRow);
                    va[dt][m] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                }
        }
        // keys past a column's token (causal diagonal) or past T (ragged tail) are masked
        const int64_t key0 = static_cast<int64_t>(j) * kDBs;
        const bool edge = causal ? key0 + kDBs - 1 > w_first : key0 + kDBs > T;
#pragma unroll
        for (int tt = 0; tt < R; ++tt) {
            f32x4 s[4];
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                s[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[n][0], qreg[tt][0], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                s[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[n][1], qreg[tt][1], s[n], 0, 0, 0);
            }
            if (edge) {
                const int64_t lim64 = causal ? t0 + tok[tt] - key0 : T - 1 - key0;  // keys <= lim are allowed
                const int lim = static_cast<int>(lim64 < kDBs ? lim64 : kDBs);
#pragma unroll
                for (int n = 0; n < 4; ++n)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (16 * n + 4 * grp + i > lim) s[n][i] = -__builtin_inff();
            }
            if (mode == 1 || (KG == 1 && first && !keep)) {  // wave-uniform
                const float cand = pair32_max(pair16_max(max_acc(s, -__builtin_inff()))) * scale_log2;  // block's column max, log2 units
                ref[tt] = mode == 1 ? fmaxf(ref[tt], cand) : cand;
                if (mode == 1) continue;
            }
            // a column with no allowed key (ref -inf) gets P = 0 throughout
            const float neg = ref[tt] == -__builtin_inff() ? -__builtin_inff() : -ref[tt];
            uint4 pw[2];
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                bf16x8 pb;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    pb[i] = static_cast<__bf16>(__builtin_amdgcn_exp2f(__builtin_fmaf(s[2 * m][i], scale_log2, neg)));
                    pb[4 + i] =
                        static_cast<__bf16>(__builtin_amdgcn_exp2f(__builtin_fmaf(s[2 * m + 1][i], scale_log2, neg)));
                }
                pw[m] = __builtin_bit_cast(uint4, pb);
            }
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) {
                o[tt][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va[dt][0], __builtin_bit_cast(bf16x8, pw[0]),
                                                                    o[tt][dt], 0, 0, 0);
                o[tt][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va[dt][1], __builtin_bit_cast(bf16x8, pw[1]),
                                                                    o[tt][dt], 0, 0, 0);
            }
            ol[tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones_a, __builtin_bit_cast(bf16x8, pw[0]), ol[tt], 0, 0, 0);
            ol[tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones_a, __builtin_bit_cast(bf16x8, pw[1]), ol[tt], 0, 0, 0);
        }
    };

    // step i: group kg computes block i KG + kg from buffer i & 1 while its
    // block of the next step is in registers; one barrier per step orders its
    // stash before the reads of the next (nk, nv: block blk(0) already loaded
    // when have0, one key group only)
    // The barrier of a step joins the waves of one key group only: the groups share
    // nothing until the merge, and out of step one group's exponentials run
    // beside the other's products (in step, every wave of a SIMD wants the same
    // unit: 4 to 12% slower). A wave arrives once its LDS accesses of the step are done; all waves of
    // the workgroup are resident, so every one arrives.
    int phase = 0;
    auto group_sync = [&]() __attribute__((always_inline)) {
        if constexpr (KG == 1) {
            __syncthreads();
        } else {
            phase += CW;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            if (lane == 0) __hip_atomic_fetch_add(&sm.arrived[kg], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            while (__builtin_amdgcn_readfirstlane(__hip_atomic_load(&sm.arrived[kg], __ATOMIC_RELAXED,
                                                                    __HIP_MEMORY_SCOPE_WORKGROUP)) < phase)
                __builtin_amdgcn_s_sleep(1);
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        }
    };
    const int steps = (nblk + KG - 1) / KG;  // workgroup-uniform
    auto walk = [&](int mode, bool keep, StageV nk, StageV nv, bool have0) __attribute__((always_inline)) {
        if (!have0 && kg < nblk) fetch(blk(kg), nk, nv);
        if (kg < nblk) stash(0, nk, nv);
        if (kg + KG < nblk) fetch(blk(kg + KG), nk, nv);
        __syncthreads();
        if (KG > 1 && mode == 0 && !keep) {
            if (w_live) set_refs(blk(0));
            __syncthreads();  // the first block has been read by every group
        }
        for (int i = 0; i < steps; ++i) {
            const int buf = i & 1;
            const int u = i * KG + kg;
            // wave-uniform: blocks past this wavefront's tokens are skipped
            if (u < w_nblk) compute(buf, blk(u), u == 0, mode, keep);
            if (u + KG < nblk) {
                stash(buf ^ 1, nk, nv);
                if (u + 2 * KG < nblk) fetch(blk(u + 2 * KG), nk, nv);
            }
            group_sync();
        }
        if (KG > 1) __syncthreads();  // every group's last reads of the staging bytes
    };
    walk(0, false, nk0, nv0, LISTED);
    // a row sum past 2^64 (or not finite): a score more than 64 log2-units above
    // its column's reference somewhere; the row sums sit in lanes 0..15, element 0
    {
        bool bad = false;
#pragma unroll
        for (int tt = 0; tt < R; ++tt) bad = bad || (w_live && lane < 16 && !(ol[tt][0] <= kDGuard));
        if (__ballot(bad) != 0ull && lane == 0) atomicOr(&sm.flag, 1);
    }
    __syncthreads();
    if (sm.flag != 0) {  // workgroup-uniform: every wave walks again
#pragma unroll
        for (int tt = 0; tt < R; ++tt) ref[tt] = -__builtin_inff();
        walk(1, true, nk0, nv0, false);  // the exact column maxima
        if constexpr (KG > 1) {
            // of every group's blocks (the walk's last barrier freed the staging bytes)
#pragma unroll
            for (int tt = 0; tt < R; ++tt)
                if (grp == 0) reinterpret_cast<float*>(&sm.st)[((kg * CW + wave) * R + tt) * 16 + col16] = ref[tt];
            __syncthreads();
#pragma unroll
            for (int tt = 0; tt < R; ++tt)
                for (int o_ = 0; o_ < KG; ++o_)
                    ref[tt] = fmaxf(ref[tt], reinterpret_cast<float*>(&sm.st)[((o_ * CW + wave) * R + tt) * 16 + col16]);
            __syncthreads();
        }
        clear();
        walk(0, true, nk0, nv0, false);  // against them: every P <= 1
    }
    if constexpr (KG > 1) {
        // the groups' sums share their references: plain additions, in group order
        if (kg > 0) {
#pragma unroll
            for (int tt = 0; tt < R; ++tt) {
#pragma unroll
                for (int dt = 0; dt < 4; ++dt) sm.mg.o[kg - 1][wave][4 * tt + dt][lane] = o[tt][dt];
                if (lane < 16) sm.mg.l[kg - 1][wave][tt][lane] = ol[tt][0];
            }
        }
        __syncthreads();
        if (kg > 0) return;
#pragma unroll
        for (int o_ = 0; o_ < KG - 1; ++o_)
#pragma unroll
            for (int tt = 0; tt < R; ++tt) {
#pragma unroll
                for (int dt = 0; dt < 4; ++dt) o[tt][dt] += sm.mg.o[o_][wave][4 * tt + dt][lane];
                ol[tt][0] += sm.mg.l[o_][wave][tt][col16];
            }
    }

    // ---- epilogue: out[b, t, h*64 + d] = O / l ----
#pragma unroll
    for (int tt = 0; tt < R; ++tt) {
        // the row sum of column col16 sits in lane col16 (lane group 0), element 0
        const float lsum = __shfl(ol[tt][0], col16, kWave);
        if (tok[tt] >= t_valid) continue;
        const int c = 16 * tt + col16;
        const float inv = 1.0f / lsum;
        uint16_t* orow = out + b * out_sb + (t0 + tok[tt]) * out_st + static_cast<int64_t>(g * R + c % R) * kDD;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) {
            bf16x4 w;
#pragma unroll
            for (int i = 0; i < 4; ++i) w[i] = static_cast<__bf16>(o[tt][dt][i] * inv);
            *reinterpret_cast<bf16x4*>(orow + 16 * dt + 4 * grp) = w;
        }
    }
}

bool prefill_dense_supported(int dtype, int64_t Hq, int64_t Hkv, int64_t D, int64_t q_sb, int64_t q_st,
                             int64_t q_sh, int64_t kv_sb, int64_t kv_st, int64_t kv_sh, int64_t out_sb,
                             int64_t out_st, const void* q, const void* k, const void* v, const void* out) {
    if (dtype != SPARDA_BF16 || D != kDD || Hq % Hkv != 0) return false;
    const int64_t R = Hq / Hkv;
    if (R < 1 || R > 4) return false;
    auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    if (!al16(q) || !al16(k) || !al16(v) || (reinterpret_cast<uintptr_t>(out) & 7u)) return false;
    if ((q_sb % 8) || (q_st % 8) || (q_sh % 8) || (kv_sb % 8) || (kv_st % 8) || (kv_sh % 8)) return false;
    if ((out_sb % 4) || (out_st % 4)) return false;
    return true;
}

int launch_prefill_dense(const void* q, int64_t q_sb, int64_t q_st, int64_t q_sh, const void* k, const void* v,
                         int64_t kv_sb, int64_t kv_st, int64_t kv_sh, int64_t B, int64_t T, int64_t Hq,
                         int64_t Hkv, int causal, float scale, void* out, int64_t out_sb, int64_t out_st,
                         hipStream_t stream) {
    const int64_t R = Hq / Hkv;
    const float sl = scale * kDLog2e;
#define SPARDA_DN(R_, CW_, KG_)                                                                            \
    hipLaunchKernelGGL((prefill_dense_kernel<R_, false, CW_, KG_>),                                        \
                       dim3(static_cast<unsigned>(B * Hkv * cdiv(T, 16 * CW_))), dim3(CW_ * KG_ * kWave), 0, stream, \
                       static_cast<const uint16_t*>(q), q_sb, q_st, q_sh, static_cast<const uint16_t*>(k), \
                       static_cast<const uint16_t*>(v), kv_sb, kv_st, kv_sh, T, static_cast<int>(Hkv),     \
                       cdiv(T, 16 * CW_), causal, sl, static_cast<uint16_t*>(out), out_sb, out_st, ChunkArgs{})
#define SPARDA_DN_W(R_)                         \
    if (groups == 4) SPARDA_DN(R_, 2, 4);       \
    else if (groups == 2) SPARDA_DN(R_, 4, 2);  \
    else SPARDA_DN(R_, 8, 1);
    // Windows of 128 tokens stage a block for the most tokens, key groups cut a
    // window's serial walk: groups where windows are few against the CUs and the
    // walk is long. W 128-token windows of up to NB blocks; times in us of
    // 1 / 2 / 4 groups, 12/4 heads, causal.
    //  - one block: nothing to share (T=64, B=1: 7.8 / 9.3 / 9.1).
    //  - up to a quarter of a window a CU: four groups (T=2048: 66 / 36 / 24; for
    //    R = 4, whose four-group form spills, from 4 blocks on: B=16, T=128 14.0 /
    //    12.6 / 14.9), up to half a window on long causal walks (T=4096: 125 / 64 / 48).
    //  - past that the longest walk against the sum of all walks: one group takes
    //    the time of NB blocks at W = 256, as many as W / 256 NB / 2 above, and two
    //    groups half a walk and a fixed cost: they cross at NB = 12 (W / 256)^2
    //    (W = 256: T=512 25 / 25, T=1024 39 / 32; W = 512: T=2048 82 / 85, T=4096
    //    145 / 142) or 80 (W = 1024: T=4096 275 / 280, T=8192 514 / 500). With one or
    //    two heads a tile's products hide less staging: not past 3/2 windows a CU
    //    (8/4 heads, W = 512, T=2048: 59 / 67).
    //  - without the mask every walk is the same: two groups up to half a window a
    //    CU, or on long walks of three and four heads (B=4, T=3000: 187 / 149).
    const int64_t NB = cdiv(T, kDBs);
    const int64_t windows = B * Hkv * cdiv(T, 128), W = windows < (1 << 20) ? windows : (1 << 20);
    const bool crossed = causal ? (NB * kDCus * kDCus >= 12 * W * W || NB >= 80) && (R >= 3 || 2 * W <= 3 * kDCus)
                                : 2 * W <= kDCus || (R >= 3 && NB >= 24);
    const int groups = NB == 1 ? 1
                       : (R < 4 || NB >= 4) && (4 * W <= kDCus || (causal && 2 * W <= kDCus && NB >= 20)) ? 4
                       : crossed ? 2
                                 : 1;
    switch (R) {
        case 1: SPARDA_DN_W(1); break;
        case 2: SPARDA_DN_W(2); break;
        case 3: SPARDA_DN_W(3); break;
        default: SPARDA_DN_W(4); break;
    }
#undef SPARDA_DN_W
#undef SPARDA_DN
    return check_hip(hipGetLastError(), "prefill_dense_kernel");
}

int launch_prefill_chunked(const void* q, int64_t q_sb, int64_t q_st, int64_t q_sh, const void* k, const void* v,
                           int64_t kv_sb, int64_t kv_st, int64_t kv_sh, const int32_t* topk, int64_t ke,
                           int64_t top_k, int32_t* sel, int32_t* n_sel, int64_t cap, int64_t B, int64_t T,
                           int64_t Hq, int64_t Hkv, float scale, void* out, int64_t out_sb, int64_t out_st,
                           hipStream_t stream) {
    const int64_t NB = cdiv(T, kDBs);
    if (NB > kChunkMaxNB)
        return set_error(SPARDA_ERR_SHAPE, "prefill_chunked: more than %d blocks", kChunkMaxNB);
    const int64_t cut = NB < top_k + 2 ? NB : top_k + 2;
    if (sel != nullptr && (cap < cut || cap > kMaxSelCap))
        return set_error(SPARDA_ERR_SHAPE, "prefill_chunked: sel_cap %lld outside [%lld, %d]", (long long)cap,
                         (long long)cut, kMaxSelCap);
    const int64_t NBq = NB;  // one workgroup per 64-token query block
    const int64_t R = Hq / Hkv;
    dim3 grid(static_cast<unsigned>(B * Hkv * NBq));
    const float sl = scale * kDLog2e;
    const ChunkArgs ch{topk, static_cast<int>(ke), static_cast<int>(top_k), static_cast<int>(cut), sel, n_sel,
                       static_cast<int>(sel != nullptr ? cap : 0)};
#define SPARDA_CH(R_)                                                                                      \
    hipLaunchKernelGGL((prefill_dense_kernel<R_, true, kLTok, 1>), grid, dim3(kLTok * kWave), 0, stream,   \
                       static_cast<const uint16_t*>(q), q_sb, q_st, q_sh, static_cast<const uint16_t*>(k), \
                       static_cast<const uint16_t*>(v), kv_sb, kv_st, kv_sh, T, static_cast<int>(Hkv), NBq, \
                       1, sl, static_cast<uint16_t*>(out), out_sb, out_st, ch)
    switch (R) {
        case 1: SPARDA_CH(1); break;
        case 2: SPARDA_CH(2); break;
        case 3: SPARDA_CH(3); break;
        default: SPARDA_CH(4); break;
    }
#undef SPARDA_CH
    return check_hip(hipGetLastError(), "prefill_dense_kernel (chunked)");
}

}  // namespace sparda
