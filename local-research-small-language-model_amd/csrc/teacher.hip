// Teacher block mass for routing-quality evaluation (model/forecast.py:133-193,
// TeacherBlockSelector): the dense attention probability of every query row on
// every KV block, averaged over the query heads of a KV head,
//
//   mass[b, g, t, j] = (1/R) sum_{h in g} sum_{s in block j} softmax_s(q[b,t,h] . k[b,s,g] / sqrt(D))
//
// (causal: keys s <= t, blocks j > t / bs get 0), without materialising the
// [B, Hq, T, T] weights the reference builds. bf16 inputs, D = 64, bs = 64.
//
// One workgroup of NW wavefronts per (b, g, window of 16 NW tokens); wavefront
// w owns tokens 16w .. 16w+15 for all R heads as R tiles of 16 columns (column
// c -> token c / R, head c % R), like the sparse prefill. K blocks are staged in
// LDS (double-buffered, the next block in flight in registers) and shared by
// the wavefronts; S^T = K Q^T per block and tile with v_mfma_f32_16x16x32_bf16.
// Bound by the exponentials and the matrix products of the scores, so each score
// is formed and exponentiated once: against the column's reference, its maximum
// over block 0 (which every column attends, key 0 being allowed to every token),
// the block sums fp32 per column in LDS, and with them the row sums; the window's
// rows are normalised and written at the end, coalesced along the blocks. Where a
// score lies so far above the reference that its exponent would cost precision
// (kTGuard), the wavefront raises its references to the block's maxima, scales
// what it holds and forms that block's sums again: one walk whatever the scores
// are. The 4 lane groups' partial sums of a column are added by one fp32 matrix
// product with ones (v_mfma_f32_16x16x4_f32, exact products) per tile, whose
// results hold their own column only (an infinite or NaN row stays alone). Windows
// of more than kTKeep blocks do not keep every block sum: they walk once for the
// row sums and references and again for the block sums, written kTKeep blocks at a time.
// B=4, T=4096, 12/4 heads: 106 us (485 TFLOP/s), 119 with a raise in every window
// (scores that peak at the token itself); 204 with two walks that both
// exponentiated, a running maximum and lane-pair sums per block. B=1, T=8192 (two
// walks) 253 us, from 325; one block (T=64) 5.5 us.
#include "common.h"
#include "kernels.h"
#include "mfma.h"

namespace sparda {

constexpr int kTBs = 64;           // block size
constexpr int kTD = 64;            // head dim
constexpr int kTKRow = kTD + 8;    // K row in LDS (bf16 elements, 144 B)
constexpr int kTKeep = 64;         // block sums kept per column (50 KB of LDS for 4 wavefronts, two workgroups per CU)
constexpr int kTSRow = 49;         // LDS row of one block's column sums (odd: reads along the blocks are conflict-free)
constexpr float kTGuard = 16384.0f; // 2^14: a lane's part of a block sum past it raises the references
constexpr int64_t kTCus = 256;

template <int R, int NW>
__global__ void __launch_bounds__(NW * kWave, 2)
teacher_mass_kernel(const uint16_t* __restrict__ q, int64_t q_sb, int64_t q_st, int64_t q_sh,
                    const uint16_t* __restrict__ k, int64_t k_sb, int64_t k_st, int64_t k_sh,
                    int64_t T, int H, int64_t NBq, int64_t NB, int causal, float scale_log2,
                    float* __restrict__ mass) {
    static_assert(16 * R <= kTSRow, "columns of a wavefront");
    constexpr int kThreads = NW * kWave;
    constexpr int kWin = 16 * NW;                // tokens per workgroup
    constexpr int kCh = kTBs * 8 / kThreads;     // 16-byte K chunks each thread stages per block
    __shared__ uint16_t kst[2][kTBs * kTKRow];
    __shared__ float lrow[NW][16 * R];           // the columns' row sums
    extern __shared__ float sums[];              // [NW][min(NB, kTKeep)][kTSRow]
    const int tid = threadIdx.x;
    const int lane = tid % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int col16 = lane % 16;
    const int grp = lane / 16;
    // heaviest windows first
    const int64_t BH = static_cast<int64_t>(gridDim.x) / NBq;
    const int64_t bg = blockIdx.x % BH;
    const int64_t t0 = (NBq - 1 - blockIdx.x / BH) * kWin;
    const int b = static_cast<int>(bg / H);
    const int g = static_cast<int>(bg % H);
    const int64_t t_last = t0 + kWin - 1 < T - 1 ? t0 + kWin - 1 : T - 1;
    const int jmax = static_cast<int>(causal ? t_last / kTBs : NB - 1);

    // Q operands of this wavefront's tiles, straight from memory
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

    // K staging: chunk c = tid + i * kThreads -> row c / 8, 16-byte chunk c % 8;
    // rows past T repeat row T-1 (masked)
    const uint16_t* kbase = k + b * k_sb + static_cast<int64_t>(g) * k_sh;
    const int srow = tid / 8, scol = (tid % 8) * 8;
    typedef unsigned int StageV __attribute__((ext_vector_type(4 * kCh)));
    auto fetch = [&](int j, StageV& r) __attribute__((always_inline)) {
        const int64_t row0 = static_cast<int64_t>(j) * kTBs;
        const int last = static_cast<int>(T - 1 - row0 < kTBs - 1 ? T - 1 - row0 : kTBs - 1);
        const uint16_t* kb = kbase + row0 * k_st;
#pragma unroll
        for (int i = 0; i < kCh; ++i) {
            int s = srow + i * (kThreads / 8);
            s = s < last ? s : last;
            const uint4 a = *reinterpret_cast<const uint4*>(kb + (s * k_st + scol));
            r[4 * i] = a.x; r[4 * i + 1] = a.y; r[4 * i + 2] = a.z; r[4 * i + 3] = a.w;
        }
    };
    auto stash = [&](int buf, const StageV& r) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kCh; ++i)
            *reinterpret_cast<uint4*>(&kst[buf][(srow + i * (kThreads / 8)) * kTKRow + scol]) =
                uint4{r[4 * i], r[4 * i + 1], r[4 * i + 2], r[4 * i + 3]};
    };

    float m[R];     // the columns' references (log2 units)
    float l = 0.0f; // row sum of column col16 of tile grp (lanes with grp < R)

    // S^T of block j for every tile; masked keys at -inf
    const int64_t w_first = t0 + 16 * wave;
    auto scores = [&](int buf, int j, f32x4 (&s)[R][4]) __attribute__((always_inline)) {
        bf16x8 ka[4][2];
#pragma unroll
        for (int n = 0; n < 4; ++n)
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
                ka[n][kk] = lds_read8(&kst[buf][(16 * n + col16) * kTKRow + 32 * kk + 8 * grp]);
#pragma unroll
        for (int tt = 0; tt < R; ++tt)
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                s[tt][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[n][0], qreg[tt][0], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                s[tt][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[n][1], qreg[tt][1], s[tt][n], 0, 0, 0);
            }
        // causal diagonal: key <= token; any block: key < T
        const int64_t key0 = static_cast<int64_t>(j) * kTBs;
        if ((causal && key0 + kTBs - 1 > w_first) || key0 + kTBs > T) {  // wave-uniform
            const int lim_t = static_cast<int>(T - 1 - key0 < kTBs ? T - 1 - key0 : kTBs);
            const int d0 = static_cast<int>(t0 - key0);  // causal: at least -kWin + 1
#pragma unroll
            for (int tt = 0; tt < R; ++tt) {
                const int lim = causal && d0 + tok[tt] < lim_t ? d0 + tok[tt] : lim_t;
#pragma unroll
                for (int n = 0; n < 4; ++n)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (16 * n + 4 * grp + i > lim) s[tt][n][i] = -__builtin_inff();
            }
        }
    };

    const int keep = static_cast<int>(NB < kTKeep ? NB : kTKeep);
    const bool once = jmax < kTKeep;  // every block sum is kept: one walk
    float* ws = sums + static_cast<int64_t>(wave) * keep * kTSRow;
    // normalises and writes blocks [j0, j1) of the wavefront's rows from `ws` and
    // `lrow` (filled by this wavefront alone): lanes along the blocks of a token,
    // then its next tokens, so that few blocks do not leave lanes idle
    auto flush = [&](int j0, int j1) __attribute__((always_inline)) {
        __builtin_amdgcn_wave_barrier();
        const int nb = j1 - j0;
        int tk = lane / nb, jj = lane % nb;
        const int dt = kWave / nb, dj = kWave % nb;
        const int rows = static_cast<int>(T - w_first < 16 ? T - w_first : 16);
        const int ld = static_cast<int>(NB);
        float* out = mass + ((static_cast<int64_t>(b) * H + g) * T + w_first) * NB + j0;
        const float* lr = lrow[wave];
#pragma unroll 2
        for (int e = lane; e < 16 * nb; e += kWave) {
            float v = 0.0f;
#pragma unroll
            for (int hh = 0; hh < R; ++hh) v += ws[jj * kTSRow + R * tk + hh] / lr[R * tk + hh];
            if (tk < rows) out[tk * ld + jj] = v / static_cast<float>(R);
            tk += dt;
            jj += dj;
            if (jj >= nb) {
                jj -= nb;
                ++tk;
            }
        }
        __builtin_amdgcn_wave_barrier();
    };

    // this lane's part (16 keys) of the block sums of column col16 of each tile, from
    // the scores against m; returns the largest
    auto expsum = [&](const f32x4 (&s)[R][4], float (&part)[R]) __attribute__((always_inline)) {
        float top = 0.0f;
#pragma unroll
        for (int tt = 0; tt < R; ++tt) {
            float a[4];
#pragma unroll
            for (int n = 0; n < 4; ++n) {
                a[n] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[tt][n][0], scale_log2, -m[tt]));
#pragma unroll
                for (int i = 1; i < 4; ++i)
                    a[n] += __builtin_amdgcn_exp2f(__builtin_fmaf(s[tt][n][i], scale_log2, -m[tt]));
            }
            part[tt] = (a[0] + a[1]) + (a[2] + a[3]);
            top = __builtin_elementwise_maximum(top, part[tt]);
        }
        return top;
    };

    // one pass over the blocks: the block sums against m, added into l (count) and
    // kept, written when kTKeep of them are held (store). The first walk (refs) sets m
    // from block 0 and raises it where a lane's part of a later block's sum passes
    // the guard; what is held by then is scaled to the new reference.
    auto walk = [&](bool refs, bool count, bool store) __attribute__((always_inline)) {
        StageV nk{};
        fetch(0, nk);
        __syncthreads();  // the previous walk has read its last buffer
        stash(0, nk);
        if (jmax >= 1) fetch(1, nk);
        __syncthreads();
        if (refs) {
            f32x4 s[R][4];
            scores(0, 0, s);
#pragma unroll
            for (int tt = 0; tt < R; ++tt) {
                const float mx = pair32_max(pair16_max(max_acc(s[tt], -__builtin_inff()))) * scale_log2;
                m[tt] = mx == -__builtin_inff() ? -__FLT_MAX__ : mx;  // a block of -inf scores: any later one is above
            }
        }
        int j0 = 0;  // first block held in `ws`
        for (int j = 0; j <= jmax; ++j) {
            const int buf = j & 1;
            f32x4 s[R][4];
            scores(buf, j, s);
            float part[R];
            const float top = expsum(s, part);
            if (refs && __builtin_expect(__ballot(!(top <= kTGuard)) != 0ull, 0)) {  // wave-uniform
                // raise the references to this block's maxima (not to a NaN)
                float f = 1.0f;
#pragma unroll
                for (int tt = 0; tt < R; ++tt) {
                    const float mx = pair32_max(pair16_max(max_acc(s[tt], -__builtin_inff()))) * scale_log2;
                    const bool up = mx > m[tt];
                    const float ft = up ? __builtin_amdgcn_exp2f(m[tt] - mx) : 1.0f;
                    m[tt] = up ? mx : m[tt];
                    f = grp == tt ? ft : f;
                }
                l *= f;
                if (store && lane < 16 * R)
#pragma unroll 1
                    for (int r = 0; r < j - j0; ++r) ws[r * kTSRow + lane] *= f;
                expsum(s, part);
            }
            // the four lane groups' parts added: every row of the product is its column's sum, of that column alone
            float d = 0.0f;  // column col16 of tile grp
#pragma unroll
            for (int tt = 0; tt < R; ++tt) {
                const f32x4 c = __builtin_amdgcn_mfma_f32_16x16x4f32(1.0f, part[tt], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                d = tt == 0 || grp == tt ? c[0] : d;
            }
            if (count) l += d;
            if (store) {
                if (lane < 16 * R) ws[(j - j0) * kTSRow + lane] = d;
                if (!once && j - j0 == kTKeep - 1) {  // wave-uniform
                    flush(j0, j + 1);
                    j0 = j + 1;
                }
            }
            if (j + 1 <= jmax) {
                stash(buf ^ 1, nk);
                if (j + 2 <= jmax) fetch(j + 2, nk);
            }
            __syncthreads();
        }
        if (count && lane < 16 * R) lrow[wave][lane] = l;
        if (store && j0 <= jmax) flush(j0, jmax + 1);
    };
    walk(true, true, once);
    if (!once) walk(false, false, true);
    // blocks past the causal limit carry no probability
    if (jmax + 1 < NB) {
        for (int tk = 0; tk < 16; ++tk) {
            const int64_t t = w_first + tk;
            if (t >= T) break;
            float* row = mass + ((static_cast<int64_t>(b) * H + g) * T + t) * NB;
            for (int64_t j = jmax + 1 + lane; j < NB; j += kWave) row[j] = 0.0f;
        }
    }
}

int launch_teacher_mass(const void* q, int64_t q_sb, int64_t q_st, int64_t q_sh, const void* k, int64_t k_sb,
                        int64_t k_st, int64_t k_sh, int64_t B, int64_t T, int64_t Hq, int64_t Hkv, int causal,
                        float scale, float* mass, hipStream_t stream) {
    const int64_t NB = cdiv(T, kTBs);
    const float scale_log2 = scale * 1.4426950408889634f;
    const int R = static_cast<int>(Hq / Hkv);
    // windows of 64 tokens (K staged once for four wavefronts), of 32 where those
    // would leave the chip with fewer than two workgroups per CU, which is what
    // the LDS of a full window allows
    const int nw = B * Hkv * cdiv(T, 64) >= 2 * kTCus ? 4 : 2;
    const int64_t NBq = cdiv(T, 16 * nw);
    const size_t lds = static_cast<size_t>(nw) * (NB < kTKeep ? NB : kTKeep) * kTSRow * sizeof(float);
    dim3 grid(static_cast<unsigned>(B * Hkv * NBq));
#define SPARDA_TEACHER(R_, NW_)                                                                             \
    hipLaunchKernelGGL((teacher_mass_kernel<R_, NW_>), grid, dim3(NW_ * kWave), lds, stream,                \
                       static_cast<const uint16_t*>(q), q_sb, q_st, q_sh, static_cast<const uint16_t*>(k),  \
                       k_sb, k_st, k_sh, T, static_cast<int>(Hkv), NBq, NB, causal, scale_log2, mass)
#define SPARDA_TEACHER_W(R_)          \
    if (nw == 4) SPARDA_TEACHER(R_, 4); \
    else SPARDA_TEACHER(R_, 2);
    switch (R) {
        case 1: SPARDA_TEACHER_W(1); break;
        case 2: SPARDA_TEACHER_W(2); break;
        case 3: SPARDA_TEACHER_W(3); break;
        default: return set_error(SPARDA_ERR_SHAPE, "teacher_mass: Hq/Hkv = %d not in {1, 2, 3}", R);
    }
#undef SPARDA_TEACHER_W
#undef SPARDA_TEACHER
    return check_hip(hipGetLastError(), "teacher_mass_kernel");
}

}  // namespace sparda
