// Rows of (sequence, head) routed by a workgroup: forecast x prototype scores
// (the canonical fma chain, on the matrix cores) and the per-row top-k of route
// keys. Shared by the stand-alone router and the prefill kernel that routes
// its own query window, so both produce the same picks bit for bit.
#pragma once

#include "common.h"
#include "mfma.h"
#include "select.h"

namespace sparda {

constexpr int kRouteWaves = 4;
constexpr int kRouteThreads = kRouteWaves * kWave;

// top-k lists of lanes whose 16-lane rows differ in bit 0 (SWAP 16) or bit 1
// (32) of their row index, merged into both
template <int SWAP, int KMAX>
__device__ __forceinline__ void merge_rows(KeyTopK<KMAX>& best) {
    double a[KMAX], c[KMAX];
#pragma unroll
    for (int i = 0; i < KMAX; ++i) {
        const uint32_t lo = static_cast<uint32_t>(__double2loint(best.r[i]));
        const uint32_t hi = static_cast<uint32_t>(__double2hiint(best.r[i]));
        if constexpr (SWAP == 16) {
            const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
            const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
            a[i] = __hiloint2double(static_cast<int>(h[0]), static_cast<int>(l[0]));
            c[i] = __hiloint2double(static_cast<int>(h[1]), static_cast<int>(l[1]));
        } else {
            const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
            const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
            a[i] = __hiloint2double(static_cast<int>(h[0]), static_cast<int>(l[0]));
            c[i] = __hiloint2double(static_cast<int>(h[1]), static_cast<int>(l[1]));
        }
    }
#pragma unroll
    for (int i = 0; i < KMAX; ++i) best.r[i] = a[i];
    best.merge(c);
}

// Four consecutive forecast elements as fp32 (vec: 4-element aligned rows)
template <int FDT>
__device__ __forceinline__ float4 load_forecast4(const void* __restrict__ f, int64_t i, bool vec) {
    if (vec) {
        float o[4];
        load_vec<FDT, 4>(f, i, o);
        return make_float4(o[0], o[1], o[2], o[3]);
    }
    return make_float4(load_elem<FDT>(f, i), load_elem<FDT>(f, i + 1), load_elem<FDT>(f, i + 2),
                       load_elem<FDT>(f, i + 3));
}

// Shape of a routing workgroup: NW wavefronts, of which PG x BG form scores:
// row part p = w % PG takes RT tiles of 16 rows, block group w / PG every BG-th
// tile of 16 blocks of a chunk (all of a chunk's CB = 16 TB BG blocks are
// staged in LDS by the whole workgroup, the next chunk in flight).
template <int DF, int NW, int PG, int BG, int RT, int TB>
struct RouteShape {
    static_assert(PG * BG <= NW, "score waves");
    static constexpr int kRows = 16 * RT * PG;
    static constexpr int kCB = 16 * TB * BG;
    static constexpr int kRow = DF + 4;             // LDS row, floats: the 16 rows x 4 dims of an operand in 64 banks
    static constexpr int kThreads = NW * kWave;
    static constexpr int kFloats = kRows * kRow > 2 * kCB * kRow ? kRows * kRow : 2 * kCB * kRow;
};

// Routes rows row0 + r (r < nrows <= kRows) of (b, h). Scores are
// v_mfma_f32_16x16x4_f32 products, 16 blocks (A, from LDS) x 16 rows (B, in
// registers), the contraction walked in order: the instruction adds its four
// terms as a sequential fma chain, so a score is the canonical chain
// fma(f[d], p[d], acc), d ascending, bit for bit (checked for normal,
// denormal, cancelling and infinite values; only the payload of a NaN may
// differ, and a NaN score is formed again on the VALU). The matrix cores leave
// the VALU to the top-k: lane l of the result holds blocks 4 (l / 16) .. +3 of row
// l % 16, keeps that row's KMAX best route keys of its blocks, and the four
// lanes of a row merge their lists at the end. On return best[rt] of a score
// wavefront holds the list of row 16 (RT p + rt) + l % 16 over its block
// group's blocks (merged further by the caller where BG > 1), in lanes 0..15, and
// with ALL in the other lanes too. With scores
// non-null every score of the row (-inf where masked) is written to
// scores[row * NB]. Called by every wavefront of the workgroup (barriers
// inside; `lds` holds Shape::kFloats floats and is free again after the
// caller's next barrier).
template <int FDT, int DF, int KMAX, int NW, int PG, int BG, int RT, int TB, bool ALL>
__device__ __forceinline__ void route_tiles(const void* __restrict__ f, int64_t fsb, int64_t fst, int64_t fsh,
                                            const float* __restrict__ protos, int b, int h, int H, int64_t row0,
                                            int nrows, int64_t Tq, int64_t NB, int bs, int causal,
                                            int64_t score_pos0, float scale, float* __restrict__ scores,
                                            float* lds, KeyTopK<KMAX> (&best)[RT]) {
#pragma clang fp contract(off)
    using Shape = RouteShape<DF, NW, PG, BG, RT, TB>;
    constexpr int kRow = Shape::kRow;
    constexpr int kS = DF / 4;                      // products per score tile; 16-byte chunks per row
    const int tid = threadIdx.x;
    const int lane = tid % kWave;
    const int col16 = lane % 16;
    const int grp = lane / 16;
    const int w = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int p = w % PG, bg = w / PG;
    const bool scorer = bg < BG;                    // wave-uniform
    const float* __restrict__ pbh = protos + (static_cast<int64_t>(b) * NB * H + h) * DF;
    const int64_t pstride = static_cast<int64_t>(H) * DF;
    const int64_t t_last = (row0 + nrows < Tq ? row0 + nrows : Tq) - 1;
    int64_t jmax64 = causal ? (score_pos0 + t_last) / bs : NB - 1;
    if (jmax64 > NB - 1) jmax64 = NB - 1;
    const int jmax = __builtin_amdgcn_readfirstlane(static_cast<int>(jmax64));

    // chunk staging: thread -> 16-byte chunks e = tid + i kThreads of the chunk's rows (clamped to block jmax)
    constexpr int kChunks = Shape::kCB * kS;
    constexpr int kPer = (kChunks + Shape::kThreads - 1) / Shape::kThreads;
    typedef float StageV __attribute__((ext_vector_type(4 * kPer)));
    StageV pr;
    auto fetch = [&](int c0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int e = tid + i * Shape::kThreads;
            const int j = c0 + (e < kChunks ? e : 0) / kS;
            const float4 x = *reinterpret_cast<const float4*>(pbh + (j < jmax ? j : jmax) * pstride + 4 * (e % kS));
            pr[4 * i] = x.x; pr[4 * i + 1] = x.y; pr[4 * i + 2] = x.z; pr[4 * i + 3] = x.w;
        }
    };
    auto stash = [&](float* dst) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int e = tid + i * Shape::kThreads;
            if (kChunks % Shape::kThreads == 0 || e < kChunks)
                *reinterpret_cast<float4*>(dst + (e / kS) * kRow + 4 * (e % kS)) =
                    make_float4(pr[4 * i], pr[4 * i + 1], pr[4 * i + 2], pr[4 * i + 3]);
        }
    };

    // the forecast rows through LDS into the B operands (step s: element 4 s + grp of row col16)
    const int64_t V = 4;
    const bool vec = (reinterpret_cast<uintptr_t>(f) & (FDT == SPARDA_F32 ? 15u : 7u)) == 0 && fsb % V == 0 &&
                     fst % V == 0 && fsh % V == 0;
    const int64_t fbase = b * fsb + h * fsh;
    fetch(0);  // under the forecast's way through LDS
    for (int e = tid; e < Shape::kRows * kS; e += Shape::kThreads) {
        int64_t t = row0 + e / kS;
        t = t < t_last ? t : t_last;
        *reinterpret_cast<float4*>(lds + (e / kS) * kRow + 4 * (e % kS)) =
            load_forecast4<FDT>(f, fbase + t * fst + 4 * (e % kS), vec);
    }
    __syncthreads();
    float fr[RT][kS];
    int limit[RT];
    float* srow[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int r = 16 * (RT * p + rt) + col16;
#pragma unroll
        for (int s = 0; s < kS; ++s) fr[rt][s] = lds[r * kRow + 4 * s + grp];
        const int64_t t = row0 + r < t_last ? row0 + r : t_last;
        const int64_t lim = causal ? (score_pos0 + t) / bs : NB - 1;
        limit[rt] = static_cast<int>(lim < jmax ? lim : jmax);
        srow[rt] = (scores != nullptr && scorer && row0 + r <= t_last)
                       ? scores + ((static_cast<int64_t>(b) * H + h) * Tq + row0 + r) * NB
                       : nullptr;
        best[rt].init();
    }
    __syncthreads();  // the forecast's bytes are free

    int cb = 0;
    for (int c0 = 0; c0 <= jmax; c0 += Shape::kCB) {  // workgroup-uniform
        float* buf = lds + cb * Shape::kCB * kRow;
        stash(buf);
        __syncthreads();
        if (c0 + Shape::kCB <= jmax) fetch(c0 + Shape::kCB);
        const int j0 = c0 + 16 * TB * bg;             // this wavefront's blocks of the chunk
        if (scorer && j0 <= jmax) {
            f32x4 acc[TB][RT];
#pragma unroll
            for (int tb = 0; tb < TB; ++tb)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) acc[tb][rt] = f32x4{0.f, 0.f, 0.f, 0.f};
            const float* pa = buf + (16 * TB * bg + col16) * kRow + grp;
#pragma unroll
            for (int s = 0; s < kS; ++s)
#pragma unroll
                for (int tb = 0; tb < TB; ++tb) {
                    const float a = pa[16 * tb * kRow + 4 * s];
#pragma unroll
                    for (int rt = 0; rt < RT; ++rt)
                        acc[tb][rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, fr[rt][s], acc[tb][rt], 0, 0, 0);
                }
#pragma unroll
            for (int tb = 0; tb < TB; ++tb)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    f32x4 v = acc[tb][rt];
                    if (__ballot(__builtin_isunordered(v[0], v[1]) || __builtin_isunordered(v[2], v[3])) != 0ull) {
                        // a NaN: the chain itself, for its payload
                        const int64_t t = row0 + 16 * (RT * p + rt) + col16;
                        const int64_t fi = fbase + (t < t_last ? t : t_last) * fst;
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const int j = j0 + 16 * tb + 4 * grp + i;
                            if (j > limit[rt] || v[i] == v[i]) continue;
                            float x = 0.0f;
                            for (int d = 0; d < DF; ++d)
                                x = __builtin_fmaf(pbh[j * pstride + d], load_elem<FDT>(f, fi + d), x);
                            v[i] = x;
                        }
                    }
                    double key[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int j = j0 + 16 * tb + 4 * grp + i;
                        const bool ok = j <= limit[rt];
                        const float sc = v[i] * scale;
                        if (srow[rt] != nullptr && ok) srow[rt][j] = sc;
                        key[i] = ok ? route_key(sc, j) : 0.0;
                    }
                    if (c0 == 0 && tb == 0) best[rt].init4(key);
                    else best[rt].push4(key);
                }
        }
        cb ^= 1;
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        if (srow[rt] != nullptr && bg == 0)
            for (int64_t j = limit[rt] + 1 + grp; j < NB; j += 4) srow[rt][j] = -__builtin_inff();
        if (scorer && 16 * TB * bg <= jmax) {  // wave-uniform: the others' lists are empty
            if (ALL || jmax >= 4) merge_rows<16>(best[rt]);  // fewer blocks sit in the first lanes alone
            if (ALL || jmax >= 8) merge_rows<32>(best[rt]);
        }
    }
}

// the row's picks (slots i >= ke: -1; slots no candidate filled: block i, the
// masked blocks in ascending order)
template <int KMAX>
__device__ __forceinline__ void route_picks(const KeyTopK<KMAX>& best, int ke, int32_t (&picks)[KMAX]) {
#pragma unroll
    for (int i = 0; i < KMAX; ++i) picks[i] = (i < ke) ? (best.r[i] == 0.0 ? i : route_key_index(best.r[i])) : -1;
}

}  // namespace sparda
