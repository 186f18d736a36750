// Producer of a layer's attention inputs: RMSNorm + the q / k / v / forecast
// projections + RoPE in one kernel (model/transformer.py:104-107 with
// model/norm.py:15-21, model/forecast.py:30-40, the projections of
// model/attention/base.py:38-52 and model/rope.py:34-65).
//
//   y[m, n] = (sum_c x[m, c] * W'[n, c]) / rms(x[m, :]),  W'[n, c] = W[n, c] * w_norm[c]
//
// W' stacks the q, k, v and forecast weights ([Hq*D; Hkv*D; Hkv*D; Hf*Df] rows,
// the RMSNorm weight folded into its columns by the caller), so the norm is a
// per-row scale applied after the product. rms is accumulated in fp32 from the
// A fragments the product streams anyway. q and k columns are rotated in the
// epilogue (pairs (i, i + D/2) of a head, fp32 cos / sin tables), and every
// region is written in its own [M, heads * D] layout.
//
// Tiling (D = 64): a 256-thread workgroup computes a BM x 128 tile of y
// (BM = 32 TM), each wavefront 16 TM x 64 = one head of one region, as the
// transposed product W' x^T in 4 x TM tiles of v_mfma_f32_16x16x32_bf16 (rows
// of W' are the A operand, rows of x the B operand). Both are staged per
// BK-wide step of c in LDS, the next step in flight in registers. W' rows are
// staged permuted (w_row), so that the tile pair (2p, 2p + 1) gives lane
// l the eight consecutive columns 32p + 8 (l / 16) + 0..7 of row l % 16: the
// outputs are 16-byte stores, and the rotation partner of a column (i + 32 or
// i - 32) sits in the same lane, one pair away. sum(x^2) is the diagonal of
// x x^T, formed on the matrix cores from the staged x fragments (each of the
// two wavefronts that share the rows takes every second row tile).
// Bound by the latency of a step's loads and LDS reads (the matrix cores are busy
// 40% of the time): 60 us = 647 TFLOP/s at M = 16384, N = 1536, C = 768, from
// 72 us with 128 x 128 tiles, the squares on the VALU and 2-byte stores (62 with
// padded rows staged before the products; M = 8192 37.9 then, 35.2 now).
#include "common.h"
#include "kernels.h"
#include "rows.h"

namespace sparda {

constexpr int kPBN = 128;          // columns of y per workgroup
constexpr int kPThreads = 256;
constexpr int64_t kPCus = 256;

template <int TM, int BK>
struct ProduceSmem {
    // rows of BK elements, their 16-byte chunks permuted by the row (swz)
    uint16_t a[2][32 * TM * BK];                 // x rows
    uint16_t b[2][kPBN * BK];                    // W' rows, permuted
    float inv_rms[32 * TM];
};

// Chunk c of LDS row r sits at chunk c ^ swz(r): any 8 consecutive lanes of an
// operand read (8 rows, one chunk) or of a staging write (one or two whole rows)
// then touch all 32 banks once. (Against rows padded by 16 bytes 2% faster at
// M = 16384 and 1 to 4% below.)
template <int BK>
__device__ __forceinline__ int swz(int r) { return BK == 32 ? (r >> 1) & 3 : r & 7; }

template <int ODT>
__device__ __forceinline__ void store_out(void* out, int64_t i, float v) {
    if constexpr (ODT == SPARDA_F32) {
        static_cast<float*>(out)[i] = v;
    } else {
        static_cast<__bf16*>(out)[i] = static_cast<__bf16>(v);
    }
}

// eight consecutive outputs; vec: the address is 16-byte aligned
template <int ODT>
__device__ __forceinline__ void store_out8(void* out, int64_t i, const float (&y)[8], bool vec) {
    if (vec) {
        if constexpr (ODT == SPARDA_F32) {
            float4* p = reinterpret_cast<float4*>(static_cast<float*>(out) + i);
            p[0] = make_float4(y[0], y[1], y[2], y[3]);
            p[1] = make_float4(y[4], y[5], y[6], y[7]);
        } else {
            bf16x8 w;
#pragma unroll
            for (int e = 0; e < 8; ++e) w[e] = static_cast<__bf16>(y[e]);
            *reinterpret_cast<bf16x8*>(static_cast<__bf16*>(out) + i) = w;
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) store_out<ODT>(out, i + e, y[e]);
    }
}

// eight consecutive table entries; vec: the address is 16-byte aligned
__device__ __forceinline__ void load_tab8(const float* __restrict__ p, float (&o)[8], bool vec) {
    if (vec) {
        const float4 u = reinterpret_cast<const float4*>(p)[0], w = reinterpret_cast<const float4*>(p)[1];
        o[0] = u.x; o[1] = u.y; o[2] = u.z; o[3] = u.w;
        o[4] = w.x; o[5] = w.y; o[6] = w.z; o[7] = w.w;
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = p[e];
    }
}

// LDS row r of a 64-column head holds W' row w_row(r) of the head: tile t = r / 16,
// row 4 g + i of it -> column 32 (t / 2) + 8 g + 4 (t % 2) + i
__device__ __forceinline__ int w_row(int r) {
    return (r & ~63) + 32 * ((r >> 5) & 1) + 8 * ((r >> 2) & 3) + 4 * ((r >> 4) & 1) + (r & 3);
}

template <int FDT, int TM, int BK>
__global__ void __launch_bounds__(kPThreads, 2)
produce_kernel(const uint16_t* __restrict__ x, int64_t x_st, const uint16_t* __restrict__ w,
               int64_t M, int C, int Nq, int Nk, int Nf, float eps,
               const float* __restrict__ cosv, const float* __restrict__ sinv, int64_t T, int64_t pos0,
               uint16_t* __restrict__ q, uint16_t* __restrict__ k, uint16_t* __restrict__ v,
               void* __restrict__ f, const int64_t* __restrict__ pos_dev, int64_t rope_len, int vec_out,
               int vec_tab) {
    using Smem = ProduceSmem<TM, BK>;
    constexpr int kBM = 32 * TM;
    constexpr int kCpr = BK / 8;                      // 16-byte chunks per row
    constexpr int kRps = kPThreads / kCpr;            // rows staged per round
    constexpr int kA = kBM / kRps, kB = kPBN / kRps;  // rounds
    __shared__ Smem sm;
    const int tid = threadIdx.x;
    const int lane = tid % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int col16 = lane % 16;
    const int grp = lane / 16;
    const int wm = wave / 2, wn = wave % 2;          // 2 x 2 wavefronts of 16 TM x 64
    const int64_t m0 = static_cast<int64_t>(blockIdx.x) * kBM;
    const int n0 = blockIdx.y * kPBN;

    // staging: thread -> 16-byte chunk tid % kCpr of rows tid / kCpr + i kRps
    const int sr = tid / kCpr, cc = (tid % kCpr) * 8;
    static_assert(kRps % 8 == 0, "swz is the same for every round of a thread");
    const int sc = (cc / 8 ^ swz<BK>(sr)) * 8;        // its place in the LDS row
    const int m_last = static_cast<int>(M - 1 - m0 < kBM - 1 ? M - 1 - m0 : kBM - 1);
    const uint16_t* xa[kA];
    const uint16_t* wb[kB];
#pragma unroll
    for (int i = 0; i < kA; ++i) {
        const int r = sr + i * kRps;
        xa[i] = x + (m0 + (r < m_last ? r : m_last)) * x_st + cc;  // rows past M repeat row M-1 (not stored)
    }
#pragma unroll
    for (int i = 0; i < kB; ++i) wb[i] = w + static_cast<int64_t>(n0 + w_row(sr + i * kRps)) * C + cc;
    typedef unsigned int StageA __attribute__((ext_vector_type(4 * kA)));
    typedef unsigned int StageB __attribute__((ext_vector_type(4 * kB)));
    StageA ra;
    StageB rb;
    auto fetch = [&](int c) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kA; ++i) {
            const uint4 t = *reinterpret_cast<const uint4*>(xa[i] + c);
            ra[4 * i] = t.x; ra[4 * i + 1] = t.y; ra[4 * i + 2] = t.z; ra[4 * i + 3] = t.w;
        }
#pragma unroll
        for (int i = 0; i < kB; ++i) {
            const uint4 t = *reinterpret_cast<const uint4*>(wb[i] + c);
            rb[4 * i] = t.x; rb[4 * i + 1] = t.y; rb[4 * i + 2] = t.z; rb[4 * i + 3] = t.w;
        }
    };
    auto stash = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kA; ++i)
            *reinterpret_cast<uint4*>(&sm.a[buf][(sr + i * kRps) * BK + sc]) =
                uint4{ra[4 * i], ra[4 * i + 1], ra[4 * i + 2], ra[4 * i + 3]};
#pragma unroll
        for (int i = 0; i < kB; ++i)
            *reinterpret_cast<uint4*>(&sm.b[buf][(sr + i * kRps) * BK + sc]) =
                uint4{rb[4 * i], rb[4 * i + 1], rb[4 * i + 2], rb[4 * i + 3]};
    };
    fetch(0);

    f32x4 acc[4][TM];  // [W' tile][x tile]: column 16 tn + 4 grp + i (permuted), row 16 tm + col16
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    f32x4 sq[TM / 2];  // x x^T of the row tiles 2 t + wn
#pragma unroll
    for (int j = 0; j < TM / 2; ++j) sq[j] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int steps = C / BK;
    stash(0);
    if (steps > 1) fetch(BK);
    __syncthreads();
    for (int st = 0; st < steps; ++st) {
        const int buf = st & 1;
#pragma unroll
        for (int kk = 0; kk < BK / 32; ++kk) {
            const int rc = ((4 * kk + grp) ^ swz<BK>(col16)) * 8;  // chunk of an operand row (row % 16 = col16)
            bf16x8 af[TM], bfr[4];
#pragma unroll
            for (int t = 0; t < 4; ++t)
                bfr[t] = lds_read8(&sm.b[buf][(64 * wn + 16 * t + col16) * BK + rc]);
#pragma unroll
            for (int t = 0; t < TM; ++t)
                af[t] = lds_read8(&sm.a[buf][(16 * TM * wm + 16 * t + col16) * BK + rc]);
#pragma unroll
            for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                for (int tn = 0; tn < 4; ++tn)
                    acc[tn][tm] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bfr[tn], af[tm], acc[tn][tm], 0, 0, 0);
            if (wn == 0) {  // wave-uniform
#pragma unroll
                for (int t = 0; t < TM / 2; ++t)
                    sq[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[2 * t], af[2 * t], sq[t], 0, 0, 0);
            } else {
#pragma unroll
                for (int t = 0; t < TM / 2; ++t)
                    sq[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[2 * t + 1], af[2 * t + 1], sq[t], 0, 0, 0);
            }
        }
        // the next step's rows go into LDS while the products drain (5% faster at
        // M = 4096 and 8192 than at the next step's start); their buffer was last
        // read before the previous step's barrier
        if (st + 1 < steps) {
            stash(buf ^ 1);
            if (st + 2 < steps) fetch((st + 2) * BK);
        }
        __syncthreads();
    }

    // 1/rms of the workgroup's rows: row r of a tile is element r % 4 of lane r + 16 (r / 4)
    if (col16 / 4 == grp) {
#pragma unroll
        for (int t = 0; t < TM / 2; ++t) {
            float s = sq[t][0];
#pragma unroll
            for (int e = 1; e < 4; ++e) s = col16 % 4 == e ? sq[t][e] : s;
            sm.inv_rms[16 * TM * wm + 16 * (2 * t + wn) + col16] = 1.0f / __builtin_sqrtf(s / static_cast<float>(C) + eps);
        }
    }
    __syncthreads();

    // epilogue: this wavefront's 64 columns are one head of one region
    const int nh = n0 + 64 * wn;                     // first column of the head
    const int Nv = Nk;
    int region, head;
    if (nh < Nq) { region = 0; head = nh / 64; }
    else if (nh < Nq + Nk) { region = 1; head = (nh - Nq) / 64; }
    else if (nh < Nq + Nk + Nv) { region = 2; head = (nh - Nq - Nk) / 64; }
    else { region = 3; head = (nh - Nq - Nk - Nv) / 64; }
    const int ld = region == 0 ? Nq : (region == 3 ? Nf : Nk);  // row stride of the output
    const int64_t t_first = m0 % T;                  // position of row m0 within its sequence
    // a device-held offset (a decode step at token *pos_dev): positions clamped into the tables
    const int64_t pos_base = pos0 + (pos_dev != nullptr ? *pos_dev : 0);
    const int64_t pos_hi = pos_dev != nullptr ? rope_len - 1 : INT64_MAX;
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) {
        const int rloc = 16 * (TM * wm + tm) + col16;
        const int64_t m = m0 + rloc;
        if (m >= M) continue;
        const float inv = sm.inv_rms[rloc];
        float y[2][8];                               // columns 32 p + 8 grp + 0..7
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int e = 0; e < 8; ++e) y[p][e] = acc[2 * p + e / 4][tm][e % 4] * inv;
        if (region <= 1) {
            int64_t t = t_first + rloc;
            while (t >= T) t -= T;
            int64_t pos = pos_base + t;
            pos = pos < 0 ? 0 : (pos > pos_hi ? pos_hi : pos);
            float cs[8], sn[8];
            load_tab8(cosv + pos * 32 + 8 * grp, cs, vec_tab != 0);
            load_tab8(sinv + pos * 32 + 8 * grp, sn, vec_tab != 0);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float x1 = y[0][e], x2 = y[1][e];
                y[0][e] = x1 * cs[e] - x2 * sn[e];
                y[1][e] = x2 * cs[e] + x1 * sn[e];
            }
        }
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const int64_t base = m * ld + 64 * head + 32 * p + 8 * grp;
            if (region == 0) store_out8<SPARDA_BF16>(q, base, y[p], vec_out != 0);
            else if (region == 1) store_out8<SPARDA_BF16>(k, base, y[p], vec_out != 0);
            else if (region == 2) store_out8<SPARDA_BF16>(v, base, y[p], vec_out != 0);
            else store_out8<FDT>(f, base, y[p], vec_out != 0);
        }
    }
}

// ---------------------------------------------------------------------------
// Decode shapes (M <= kRowsMaxM rows, a few tokens): the tiled kernel would
// run N/128 workgroups and stream all of W' through a dozen CUs. Here a
// workgroup owns 16 columns of one head (8 RoPE pairs: d0+p and d0+p+32,
// p < 8), so N/16 workgroups share the weight read; the 16 columns' rows of W'
// are the A operand of matrix-core products with the x rows (rows.h), which
// also yield sum(x^2) for 1/rms. Results go through LDS to the threads that
// rotate and store the pairs.
// ---------------------------------------------------------------------------
template <int FDT>
__global__ void __launch_bounds__(kPThreads)
produce_rows_kernel(const uint16_t* __restrict__ x, int64_t x_st, const uint16_t* __restrict__ w, int M, int C,
                    int Nq, int Nk, int Nf, float eps, const float* __restrict__ cosv,
                    const float* __restrict__ sinv, int64_t T, int64_t pos0, uint16_t* __restrict__ q,
                    uint16_t* __restrict__ k, uint16_t* __restrict__ v, void* __restrict__ f,
                    const int64_t* __restrict__ pos_dev, int64_t rope_len, uint16_t* __restrict__ kc,
                    uint16_t* __restrict__ vc, int64_t c_sb, int64_t c_st, int64_t c_sh, int64_t cap) {
    static_assert(kPThreads == kRowsWaves * kWave, "one rows_mfma workgroup");
    __shared__ RowsRed<1> red;
    __shared__ float ylds[1][kRowsMaxM][16];
    __shared__ float rs[16];
    const int tid = threadIdx.x;
    const int wave = tid / kWave;
    const int nh = (blockIdx.x / 4) * 64;            // first column of the head
    const int d0 = (blockIdx.x % 4) * 8;
    // local column lc = tile row: pair lc/2, half lc%2
    const int lr = tid % 16;
    const uint16_t* wrow[1] = {w + static_cast<int64_t>(nh + d0 + lr / 2 + 32 * (lr % 2)) * C};
    f32x4 acc[1];
    float ss;
    rows_mfma<1>(x, x_st, M, C, wrow, wave, acc, ss);
    rows_reduce<1>(red, acc, ss, wave, true, ylds, rs);
    if (tid < M * 16) {
        const int m = tid / 16, c = tid % 16;
        ylds[0][m][c] = ylds[0][m][c] / __builtin_sqrtf(rs[m] / static_cast<float>(C) + eps);
    }
    __syncthreads();

    const int Nv = Nk;
    int region, head;
    if (nh < Nq) { region = 0; head = nh / 64; }
    else if (nh < Nq + Nk) { region = 1; head = (nh - Nq) / 64; }
    else if (nh < Nq + Nk + Nv) { region = 2; head = (nh - Nq - Nk) / 64; }
    else { region = 3; head = (nh - Nq - Nk - Nv) / 64; }
    const int ld = region == 0 ? Nq : (region == 3 ? Nf : Nk);
    const int64_t pos_base = pos0 + (pos_dev != nullptr ? *pos_dev : 0);
    const int64_t pos_hi = pos_dev != nullptr ? rope_len - 1 : INT64_MAX;
    for (int t = tid; t < M * 8; t += kPThreads) {
        const int m = t / 8, p = t % 8;
        float y1 = ylds[0][m][2 * p], y2 = ylds[0][m][2 * p + 1];
        const int d = d0 + p;
        if (region <= 1) {
            int64_t pos = pos_base + m % T;
            pos = pos < 0 ? 0 : (pos > pos_hi ? pos_hi : pos);
            const float c = cosv[pos * 32 + d], sn = sinv[pos * 32 + d];
            const float r1 = y1 * c - y2 * sn;
            const float r2 = y2 * c + y1 * sn;
            y1 = r1;
            y2 = r2;
        }
        const int64_t base = static_cast<int64_t>(m) * ld + 64 * head + d;
        if (region == 0) { store_out<SPARDA_BF16>(q, base, y1); store_out<SPARDA_BF16>(q, base + 32, y2); }
        else if (region == 1) { store_out<SPARDA_BF16>(k, base, y1); store_out<SPARDA_BF16>(k, base + 32, y2); }
        else if (region == 2) { store_out<SPARDA_BF16>(v, base, y1); store_out<SPARDA_BF16>(v, base + 32, y2); }
        else { store_out<FDT>(f, base, y1); store_out<FDT>(f, base + 32, y2); }
        if (kc != nullptr && (region == 1 || region == 2)) {
            // the new key / value also as row p of sequence m / T in the caches
            int64_t p = pos_base + m % T;
            p = p < 0 ? 0 : (p > cap - 1 ? cap - 1 : p);
            const int64_t ci = (m / T) * c_sb + p * c_st + head * c_sh + d;
            uint16_t* dst = region == 1 ? kc : vc;
            store_out<SPARDA_BF16>(dst, ci, y1);
            store_out<SPARDA_BF16>(dst, ci + 32, y2);
        }
    }
}

int launch_produce(const void* x, int64_t x_st, const void* w, int64_t M, int64_t C, int64_t Nq, int64_t Nk,
                   int64_t Nf, float eps, const float* cosv, const float* sinv, int64_t T, int64_t pos0,
                   void* q, void* k, void* v, void* f, int f_dtype, hipStream_t stream,
                   const int64_t* pos_dev, int64_t rope_len, void* kc, void* vc, int64_t c_sb, int64_t c_st,
                   int64_t c_sh, int64_t cap) {
    const int64_t N = Nq + 2 * Nk + Nf;
    if (M <= kRowsMaxM && C % 128 == 0 && C / 128 <= kRowsWaves * kRowsMaxKB) {
        const size_t lds = 0;
#define SPARDA_PRODUCE_ROWS(FDT_)                                                                            \
    hipLaunchKernelGGL((produce_rows_kernel<FDT_>), dim3(static_cast<unsigned>(N / 16)), dim3(kPThreads), lds, \
                       stream, static_cast<const uint16_t*>(x), x_st, static_cast<const uint16_t*>(w),        \
                       static_cast<int>(M), static_cast<int>(C), static_cast<int>(Nq), static_cast<int>(Nk),  \
                       static_cast<int>(Nf), eps, cosv, sinv, T, pos0, static_cast<uint16_t*>(q),             \
                       static_cast<uint16_t*>(k), static_cast<uint16_t*>(v), f, pos_dev, rope_len,             \
                       static_cast<uint16_t*>(kc), static_cast<uint16_t*>(vc), c_sb, c_st, c_sh, cap)
        if (f_dtype == SPARDA_F32) SPARDA_PRODUCE_ROWS(SPARDA_F32);
        else SPARDA_PRODUCE_ROWS(SPARDA_BF16);
#undef SPARDA_PRODUCE_ROWS
        return check_hip(hipGetLastError(), "produce_rows_kernel");
    }
    if (kc != nullptr) return set_error(SPARDA_ERR_SHAPE, "produce: cache rows are written for M <= %d only",
                                        kRowsMaxM);
    auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    const int vec_out = al16(q) && al16(k) && al16(v) && al16(f);  // rows are multiples of 64 elements
    const int vec_tab = al16(cosv) && al16(sinv);
#define SPARDA_PRODUCE(FDT_, TM_, BK_)                                                                     \
    hipLaunchKernelGGL((produce_kernel<FDT_, TM_, BK_>),                                                   \
                       dim3(static_cast<unsigned>(cdiv(M, 32 * TM_)), static_cast<unsigned>(N / kPBN)),    \
                       dim3(kPThreads), 0, stream,                                                         \
                       static_cast<const uint16_t*>(x), x_st, static_cast<const uint16_t*>(w), M,        \
                       static_cast<int>(C), static_cast<int>(Nq), static_cast<int>(Nk),                   \
                       static_cast<int>(Nf), eps, cosv, sinv, T, pos0, static_cast<uint16_t*>(q),         \
                       static_cast<uint16_t*>(k), static_cast<uint16_t*>(v), f, pos_dev, rope_len,        \
                       vec_out, vec_tab)
#define SPARDA_PRODUCE_T(FDT_)                                  \
    switch (tile) {                                             \
        case 0: SPARDA_PRODUCE(FDT_, 8, 32); break;             \
        case 1: SPARDA_PRODUCE(FDT_, 4, 64); break;             \
        case 2: SPARDA_PRODUCE(FDT_, 2, 64); break;             \
        case 3: SPARDA_PRODUCE(FDT_, 4, 32); break;             \
        default: SPARDA_PRODUCE(FDT_, 2, 32); break;            \
    }
    // The widest tile that leaves the chip enough workgroups (N = 1536, C = 768):
    // 256 rows past two and a half workgroups per CU, two at a time (62 us against
    // 68 with 128 rows at M = 16384, 3 per CU; 69 against 58 at 12000, 2.2 per CU,
    // where a second round is nearly empty), 128 rows past one per CU (25.9 us
    // against 28.1 with 64 rows at 4096), 64 rows below (20.1 against 19.3 at 2048,
    // launch included). A width that is no multiple of 64 takes 32-wide steps.
    const int64_t cols = N / kPBN;
    const int tile = C % 64 != 0 ? (cdiv(M, 128) * cols > kPCus ? 3 : 4)
                                 : (2 * cdiv(M, 256) * cols > 5 * kPCus ? 0 : (cdiv(M, 128) * cols > kPCus ? 1 : 2));
    if (f_dtype == SPARDA_F32) { SPARDA_PRODUCE_T(SPARDA_F32) }
    else { SPARDA_PRODUCE_T(SPARDA_BF16) }
#undef SPARDA_PRODUCE_T
#undef SPARDA_PRODUCE
    return check_hip(hipGetLastError(), "produce_kernel");
}

}  // namespace sparda
