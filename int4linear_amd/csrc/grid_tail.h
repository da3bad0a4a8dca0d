// What the two small-grid kernels (int8: kernels_grid.hip, FP6: kernels_fp6_grid.hip) have in
// common: the order of tiles, and everything after the last MFMA.  In both, KG waves share a tile of
// FM x FN MFMA fragments and split K between them.
#pragma once
#include "kernels.h"

#include <numeric>
#include <type_traits>
#include <utility>

namespace int4linear {

constexpr int kGridFrag = 32;    // rows of an MFMA operand
constexpr int kGridMaxSlices = 8; // of K, over workgroups

#if defined(__HIPCC__)
// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>)
template <int N, class F>
__device__ __forceinline__ void static_for(F &&f)
{
    [&]<int... I>(std::integer_sequence<int, I...>) {
        (f(std::integral_constant<int, I>{}), ...);
    }(std::make_integer_sequence<int, N>{});
}

// A wave-uniform value that the compiler may hold on the vector side, in scalar registers.
__device__ __forceinline__ unsigned uniform(unsigned v) { return (unsigned)__builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ const uint8_t *uniform(const uint8_t *p)
{
    const unsigned long long v = (unsigned long long)p;
    return (const uint8_t *)((unsigned long long)uniform((unsigned)v) | ((unsigned long long)uniform((unsigned)(v >> 32)) << 32));
}

// XCD-aware tile order, as in kernels_mfma.hip.
__device__ __forceinline__ void grid_tile_coords(int v, int total, int tiles_m, int tiles_n, int &tm, int &tn)
{
    constexpr int kXcd = 8, kGroup = 8;
    const int x = v % kXcd, j = v / kXcd;
    const int cnt = total / kXcd, rem = total % kXcd;
    const int q = x * cnt + (x < rem ? x : rem) + j;
    const int per_group = kGroup * tiles_n;
    const int group = q / per_group;
    const int first_m = group * kGroup;
    const int gsz = (tiles_m - first_m < kGroup) ? (tiles_m - first_m) : kGroup;
    const int in_group = q % per_group;
    tm = first_m + in_group % gsz;
    tn = in_group / gsz;
}

// The end of a workgroup.  Accumulator t of fragment (i, j) (X is the MFMA A operand) is row
// 32 j + 8 (t / 4) + 4 (lane / 32) + t % 4, column 32 i + lane % 32 of the tile and has the linear
// index (j * FN + i) * 16 + t; wave w collects, adds up and stores the sums with indices
// [w * KEEP, (w + 1) * KEEP).
template <int FM, int FN, int KG, bool HALF_OUT>
struct GridTail {
    static constexpr int KEEP = FM * FN * 16 / KG;
    static constexpr int RUN = std::gcd(KEEP, 16);  // sums in a row that are in one fragment
    static constexpr int FRAGS = KEEP / RUN;        // such runs
    static constexpr int BM = FM * kGridFrag, BN = FN * kGridFrag;
    static constexpr int LDS_BYTES = KG * (KG - 1) * KEEP * 256;
    static_assert(KEEP % 2 == 0, "exchange() sends pairs");

    int lane, wave, m0, n0, M, N;
    int bias[FRAGS];
    float col_scale[FRAGS], row_scale[KEEP];
    int kept[KEEP];

    __device__ __forceinline__ int row_of(int q) const
    {
        const int r = wave * KEEP + q, t = r % 16;
        return r / 16 / FN * kGridFrag + 8 * (t / 4) + 4 * (lane >> 5) + t % 4;
    }
    __device__ __forceinline__ int col_of(int f) const { return (wave * KEEP + f * RUN) / 16 % FN * kGridFrag + (lane & 31); }

    // The epilogue's operands (clamped inside the matrix).  Called early, behind the first loads
    // of the main loop, so that nothing waits for them at the end.
    __device__ __forceinline__ void fetch(const Epilogue &ep)
    {
#pragma unroll
        for (int f = 0; f < FRAGS; ++f) {
            bias[f] = 0;
            col_scale[f] = 1.f;
        }
#pragma unroll
        for (int q = 0; q < KEEP; ++q)
            row_scale[q] = 1.f;
        if (ep.bias) {
#pragma unroll
            for (int f = 0; f < FRAGS; ++f)
                bias[f] = ep.bias[min(n0 + col_of(f), N - 1)];
        }
        if (ep.col_scale) {
#pragma unroll
            for (int f = 0; f < FRAGS; ++f)
                col_scale[f] = ep.col_scale[min(n0 + col_of(f), N - 1)];
        }
        if (ep.row_scale) {
#pragma unroll
            for (int q = 0; q < KEEP; ++q)
                row_scale[q] = ep.row_scale[min(m0 + row_of(q), M - 1)];
        }
    }

    // The sums meet in LDS (LDS_BYTES, no longer read for anything else by any wave):
    // [collecting wave][sending wave][KEEP] x 64 lanes.  sum(i, j, t) is this wave's share.
    template <class F>
    __device__ __forceinline__ void collect(uint8_t *lds, F &&sum)
    {
        int *const area = (int *)lds + lane;
        static_for<KG>([&](auto me_tag) {
            constexpr int me = decltype(me_tag)::value;
            if (wave == me) {
                static_for<KG>([&](auto to_tag) {
                    constexpr int to = decltype(to_tag)::value;
                    static_for<KEEP>([&](auto q) {
                        constexpr int r = to * KEEP + decltype(q)::value;
                        const int v = sum(std::integral_constant<int, r / 16 % FN>{}, std::integral_constant<int, r / 16 / FN>{},
                                          std::integral_constant<int, r % 16>{});
                        if constexpr (to == me)
                            kept[q()] = v;
                        else
                            area[((to * (KG - 1) + (me < to ? me : me - 1)) * KEEP + q()) * 64] = v;
                    });
                });
            }
        });
        __syncthreads();
#pragma unroll
        for (int q = 0; q < KEEP; ++q)
#pragma unroll
            for (int g = 0; g < KG - 1; ++g)
                kept[q] += area[((wave * (KG - 1) + g) * KEEP + q) * 64];
    }

    // Slices of K: every wave leaves its sums in the slab of (tile, slice), waits until they have
    // been acknowledged and counts itself in at the counter of (tile, wave).  The waves with
    // one number hold the same sums in every slice's workgroup, so the last of them to arrive adds
    // the others' up, stores (true is returned), and puts the counter back to zero.  Nobody
    // waits for anybody, and integer sums do not depend on who arrives when.  (Relaxed atomic
    // operations at device scope go through to the level all workgroups share; fences at that
    // scope would write back and invalidate the XCD's whole L2 instead.)
    __device__ __forceinline__ bool exchange(int *partial, unsigned *arrivals, int tile, int slice, int slices)
    {
        typedef unsigned long long u64;
        constexpr int kWords = KEEP / 2, kSlab = KG * kWords * 64;
        u64 *const slabs = (u64 *)partial + (size_t)tile * slices * kSlab + (size_t)wave * kWords * 64 + lane;
#pragma unroll
        for (int q = 0; q < kWords; ++q)
            __hip_atomic_store(slabs + slice * kSlab + q * 64, (u64)(unsigned)kept[2 * q] | ((u64)(unsigned)kept[2 * q + 1] << 32),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        unsigned *const counter = arrivals + tile * KG + wave;
        unsigned before = 0;
        if (lane == 0)
            before = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        before = uniform(before);
        if (before != (unsigned)(slices - 1))
            return false;
        if (lane == 0)
            __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        u64 got[kGridMaxSlices - 1][kWords];  // all loads go out together
#pragma unroll
        for (int p = 0; p < kGridMaxSlices - 1; ++p)
#pragma unroll
            for (int q = 0; q < kWords; ++q)
                got[p][q] = p < slices - 1 ? __hip_atomic_load(slabs + (p < slice ? p : p + 1) * kSlab + q * 64, __ATOMIC_RELAXED,
                                                               __HIP_MEMORY_SCOPE_AGENT)
                                           : 0ull;
#pragma unroll
        for (int p = 0; p < kGridMaxSlices - 1; ++p)
#pragma unroll
            for (int q = 0; q < kWords; ++q) {
                kept[2 * q] += (int)(unsigned)got[p][q];
                kept[2 * q + 1] += (int)(unsigned)(got[p][q] >> 32);
            }
        return true;
    }

    // 32 lanes store 32 consecutive columns, through a descriptor over the tile's rows: a lane
    // outside the matrix gets an offset beyond it and the hardware drops the store.
    __device__ __forceinline__ void store(const Epilogue &ep, void *y)
    {
        constexpr unsigned kElem = HALF_OUT ? 2u : 4u;
        const bool plain = !ep.bias && !ep.out;
        const int rows_left = M - m0, cols_left = N - n0;
        const size_t extent = ((size_t)(min(rows_left, BM) - 1) * N + min(cols_left, BN)) * kElem;
        __amdgpu_buffer_rsrc_t rsrc =
            __builtin_amdgcn_make_buffer_rsrc((uint8_t *)y + ((size_t)m0 * N + n0) * kElem, 0, (int)extent, 0x00020000);
        unsigned col_off[FRAGS];
#pragma unroll
        for (int f = 0; f < FRAGS; ++f)
            col_off[f] = col_of(f) < cols_left ? (unsigned)col_of(f) * kElem : 0x40000000u;
#pragma unroll
        for (int q = 0; q < KEEP; ++q) {
            const unsigned off = (row_of(q) < rows_left ? (unsigned)row_of(q) * (unsigned)N * kElem : 0x80000000u) + col_off[q / RUN];
            if constexpr (HALF_OUT)
                __builtin_amdgcn_raw_buffer_store_b16(
                    (unsigned short)epilogue_value16(ep, kept[q], bias[q / RUN], row_scale[q], col_scale[q / RUN]), rsrc, off, 0, 0);
            else
                __builtin_amdgcn_raw_buffer_store_b32(
                    (unsigned)(plain ? kept[q] : epilogue_value32(ep, kept[q], bias[q / RUN], row_scale[q], col_scale[q / RUN])), rsrc,
                    off, 0, 0);
        }
    }
};
#endif

inline long grid_tiles(int m, int n, int bm, int bn) { return (long)((m + bm - 1) / bm) * ((n + bn - 1) / bn); }

// Where a launch that is split over K keeps its partial sums and counts its arrivals.
struct GridSplit {
    int slices = 1;
    void *partial = nullptr;
    unsigned *arrivals = nullptr;
};

// What exchange() assumes of a split into equal slices of `parts` parts of K over tiles of `kg` waves.
inline bool grid_split_valid(const GridSplit &split, long tiles, int kg, int parts)
{
    return split.slices == 1 || (split.slices > 1 && split.slices <= kGridMaxSlices && parts % split.slices == 0 && split.partial &&
                                 split.arrivals && tiles * kg <= kSkinnyArrivalWords);
}

}  // namespace int4linear
