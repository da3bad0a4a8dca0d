// Small-grid form of the int8-MFMA GEMM: shapes whose 128 x 128 tiles would leave half of the CUs
// idle or more.  Same arithmetic as kernels_mfma.hip (packed s4 through LDS, nibbles widened to
// 16 times their value in int8 lanes, C = acc >> 8).
//
// What bounds such a grid is the time to get a CU's operands to it and the length of one
// wave's chain of instructions: with a tile per CU nothing else runs there.  Hence
//   * all waves of a workgroup share one tile of C and split every stage's K between them.  A wave
//     then owns a block of C large enough (64 x 64 or 64 x 32) that a widened fragment feeds
//     several MFMAs: 6 vector operations per MFMA instead of the 12 of 32 x 32 quadrants, where
//     the vector unit, not the matrix unit, sets the pace.  The sums meet in LDS at the end: each
//     wave collects one part of the tile and stores it.
//   * a stage is 256 or 512 of K: whole 128-byte lines of every row, one barrier.
//   * one set of packed and of widened operands is a pipeline: the even-nibble MFMAs of a unit run
//     while its odd nibbles are masked, its odd-nibble MFMAs while the next unit's even nibbles
//     are shifted and masked.  No registers for a second set, so three waves fit a SIMD.
//   * the epilogue's operands are fetched behind the first stage's loads, not after the last MFMA.
//   * neighbouring columns of tiles start at different stages of K (the order of K does not
//     matter to the sums), so that the CUs do not all miss on the same lines at the same time.
// Measured against the 64 x 64 tile of four quadrants by two halves of K that it replaces, launches
// from a graph: 65 x 4096 x 4096 9.5 -> 6.5 us, 333 x 1111 x 4096 9.6 -> 6.6, 256 x 4096 x 4096
// 10.0 -> 9.1, 128 x 14336 x 4096 14.9 -> 13.0, 300 x 520 x 640 4.15 -> 3.7.
//
// With few tiles and long K a tile's K is split over workgroups as well; they exchange partial sums
// through memory inside the same launch (see the kernel's end).
#include "kernels.h"

#include <type_traits>
#include <utility>

namespace int4linear {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef unsigned long long u64;

#define I4L_LDS(p) ((__attribute__((address_space(3))) void *)(p))
// s_waitcnt immediate: vmcnt only, the other counters left at "no wait"; and lgkmcnt(0) only
#define I4L_VMCNT(n) ((0x0F70) | ((n) & 0xF) | ((((n) >> 4) & 0x3) << 14))
#define I4L_LGKM0 0xC07F

// 16 bytes per lane from global memory (wave-uniform base + per-lane offset) straight into LDS
// at lds_addr + 16 * lane.
__device__ __forceinline__ void dma16(const void *sbase, unsigned voff, unsigned lds_addr)
{
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(voff), "s"(sbase), "s"(lds_addr)
                 : "memory");
}

template <int N>
__device__ __forceinline__ void wait_vm()
{
    static_assert(N >= 0 && N <= 63, "vmcnt is six bits");
    __builtin_amdgcn_s_waitcnt(I4L_VMCNT(N));
}

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
    const u64 v = (u64)p;
    return (const uint8_t *)((u64)uniform((unsigned)v) | ((u64)uniform((unsigned)(v >> 32)) << 32));
}

constexpr int kPieceK = 128;  // K comes in pieces of 128: 64 bytes of a row
constexpr int kFrag = 32;     // rows of an MFMA 32x32x32 operand
constexpr int kMaxSlices = 8; // of K, over workgroups

// KG waves share a tile of FM x FN fragments; each takes 1 / KG of every stage's K.  A stage is
// PIECES pieces of every row, NSTAGE of them ring in LDS.
template <int FM_, int FN_, int KG_, int PIECES_, int NSTAGE_, int WAVES_PER_SIMD_>
struct GridTile {
    static constexpr int FM = FM_, FN = FN_, KG = KG_, PIECES = PIECES_, NSTAGE = NSTAGE_, OCC = WAVES_PER_SIMD_;
    static constexpr int THREADS = KG * 64;
    static constexpr int BM = FM * kFrag, BN = FN * kFrag;
    static constexpr int ROW_BYTES = 64 * PIECES;       // of a row in a stage
    static constexpr int CHUNKS = ROW_BYTES / 16;
    static constexpr int LOAD_ROWS = 1024 / ROW_BYTES;  // rows one load instruction of a wave moves
    static constexpr int STAGE_BYTES = (BM + BN) * ROW_BYTES;
    static constexpr int LDS_BYTES = STAGE_BYTES * NSTAGE;
    static constexpr int CH = (BM + BN) / LOAD_ROWS / KG;  // loads per wave and stage
    static constexpr int STEPS = 2 * PIECES / KG;          // units of 64 k per wave and stage
    static constexpr int KEEP = FM * FN * 16 / KG;         // sums per lane that a wave collects in the end
    static_assert(PIECES == 2 || PIECES == 4, "rows of 128 or 256 bytes");
    static_assert((BM + BN) / LOAD_ROWS % KG == 0, "loads split evenly");
    static_assert(STEPS == 1 || STEPS == 2, "");
    static_assert(KEEP % 2 == 0 && (KEEP <= 16 ? 16 % KEEP == 0 : KEEP % 16 == 0), "parts of fragments or whole ones");
    static_assert(KG * (KG - 1) * KEEP * 256 <= LDS_BYTES, "the sums meet in the ring's LDS");
    static_assert((NSTAGE - 1) * CH <= 63, "vmcnt is six bits");
    // LDS slot of 16-byte chunk c of row r is c ^ swizzle(r): sixteen lanes that read one chunk of
    // sixteen consecutive rows hit sixteen different 16-byte groups of the banks (no conflicts
    // counted).
    __device__ static int swizzle(int r) { return PIECES == 2 ? (r >> 1) & 7 : r & 15; }
};

// XCD-aware tile order, as in kernels_mfma.hip.
__device__ __forceinline__ void tile_coords(int v, int total, int tiles_m, int tiles_n, int &tm, int &tn)
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

// One argument instead of eleven: the host's cost of a launch grows with their number.
struct GridArgs {
    const uint8_t *x, *w;
    void *y;
    int m, n, k, tiles_m, tiles_n, slices;
    int *partial;
    unsigned *arrivals;
    Epilogue ep;
};

// HALF_OUT: the build for the two output kinds of 16-bit elements.
// Workgroup v computes slice v / tiles of K of tile v % tiles; slices > 1 meet in `partial` and
// `arrivals` (kernels.h: launch_grid).
template <class C, bool HALF_OUT>
__global__ __launch_bounds__(C::THREADS, C::OCC) void mfma_grid_kernel(GridArgs args)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const uint8_t *const X = args.x, *const W = args.w;
    const int M = args.m, N = args.n, K = args.k, tiles_m = args.tiles_m, tiles_n = args.tiles_n, slices = args.slices;
    const Epilogue &ep = args.ep;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rowbytes = K >> 1;
    const int tiles = tiles_m * tiles_n;
    const int slice = blockIdx.x / tiles;
    const int tile = blockIdx.x - slice * tiles;
    const int pieces = K / kPieceK / slices;  // of this workgroup's slice of a row
    const int KT = (pieces + C::PIECES - 1) / C::PIECES;
    const int last_pieces = pieces - (KT - 1) * C::PIECES;  // in the last stage
    const bool ragged = last_pieces != C::PIECES;
    int tm, tn;
    tile_coords(tile, tiles, tiles_m, tiles_n, tm, tn);
    const int m0 = tm * C::BM, n0 = tn * C::BN;

    // ---- loads.  A stage is the tile's rows of X, then those of W; lane p of a load lands at byte
    //      16 p: row p / CHUNKS, slot p % CHUNKS.  Rows past the matrix re-read its last row,
    //      pieces past the end of K the last valid piece.
    const uint8_t *base[C::CH];
    unsigned voff[C::CH];
    const unsigned place = (unsigned)(size_t)I4L_LDS(lds) + wave * C::CH * 1024;
    auto chunk_of = [&](int c) {  // the chunk this lane fetches in load c (BM is a multiple of the swizzle's period)
        const int r = (wave * C::CH + c) * C::LOAD_ROWS + lane / C::CHUNKS;
        return (lane & (C::CHUNKS - 1)) ^ C::swizzle(r);
    };
#pragma unroll
    for (int c = 0; c < C::CH; ++c) {
        const int i = wave * C::CH + c;
        const bool is_x = i < C::BM / C::LOAD_ROWS;
        const int r = (is_x ? i : i - C::BM / C::LOAD_ROWS) * C::LOAD_ROWS + lane / C::CHUNKS;
        const int row = is_x ? min(r, M - 1 - m0) : min(r, N - 1 - n0);
        base[c] = uniform((is_x ? X + (size_t)m0 * rowbytes : W + (size_t)n0 * rowbytes) + (size_t)slice * pieces * 64);
        voff[c] = (unsigned)row * (unsigned)rowbytes + (unsigned)chunk_of(c) * 16u;
    }
    const int whole = KT - (ragged ? 1 : 0);  // stages in full
    const int first = whole > 0 ? (int)((unsigned)tn % (unsigned)whole) : 0;  // the one taken first
    auto issue = [&](int st, unsigned ring) {
        if (ragged && st == KT - 1) {
#pragma unroll
            for (int c = 0; c < C::CH; ++c) {
                const int beyond = (chunk_of(c) >> 2) - (last_pieces - 1);
                dma16(base[c] + (size_t)st * C::ROW_BYTES, voff[c] - (unsigned)max(beyond, 0) * 64u, place + c * 1024 + ring);
            }
        } else {
            const int from = st + first < whole ? st + first : st + first - whole;
#pragma unroll
            for (int c = 0; c < C::CH; ++c)
                dma16(base[c] + (size_t)from * C::ROW_BYTES, voff[c], place + c * 1024 + ring);
        }
    };
    issue(0, 0);

    // ---- The sums this wave collects in the end are those with linear index (j * FN + i) * 16 + t
    //      in [wave * KEEP, (wave + 1) * KEEP), accumulator t of fragment (i, j) being row
    //      32 j + 8 (t / 4) + 4 (lane / 32) + t % 4, column 32 i + lane % 32 of the tile (X is the
    //      MFMA A operand).  Their epilogue operands are fetched now.
    const int fr = lane & 31;
    const int fg = lane >> 5;
    constexpr int kCols = C::KEEP > 16 ? C::KEEP / 16 : 1;  // fragments they come from
    auto row_of = [&](int q) {
        const int r = wave * C::KEEP + q, t = r % 16;
        return r / 16 / C::FN * kFrag + 8 * (t / 4) + 4 * fg + t % 4;
    };
    auto col_of = [&](int i) { return (wave * C::KEEP / 16 + i) % C::FN * kFrag + fr; };
    int bias_v[kCols];
    float cs_v[kCols], rs_v[C::KEEP];
#pragma unroll
    for (int i = 0; i < kCols; ++i) {
        bias_v[i] = 0;
        cs_v[i] = 1.f;
    }
#pragma unroll
    for (int q = 0; q < C::KEEP; ++q)
        rs_v[q] = 1.f;
    if (ep.bias) {
#pragma unroll
        for (int i = 0; i < kCols; ++i)
            bias_v[i] = ep.bias[min(n0 + col_of(i), N - 1)];
    }
    if (ep.col_scale) {
#pragma unroll
        for (int i = 0; i < kCols; ++i)
            cs_v[i] = ep.col_scale[min(n0 + col_of(i), N - 1)];
    }
    if (ep.row_scale) {
#pragma unroll
        for (int q = 0; q < C::KEEP; ++q)
            rs_v[q] = ep.row_scale[min(m0 + row_of(q), M - 1)];
    }
#pragma unroll
    for (int st = 1; st < C::NSTAGE; ++st)
        if (st < KT)
            issue(st, st * C::STAGE_BYTES);

    // ---- math.  A unit is 64 k: two 16-byte chunks of a row, one per half of the wave; the even
    //      nibbles of a chunk feed one MFMA, the odd ones another.  This wave's units of a stage
    //      are wave * STEPS, ...
    unsigned rd[C::STEPS];
#pragma unroll
    for (int s = 0; s < C::STEPS; ++s)
        rd[s] = (unsigned)(fr * C::ROW_BYTES + ((2 * (C::STEPS * wave + s) + fg) ^ C::swizzle(fr)) * 16);
    const int himask = (int)0xF0F0F0F0u;
    v16i acc[C::FN][C::FM];
#pragma unroll
    for (int i = 0; i < C::FN; ++i)
#pragma unroll
        for (int j = 0; j < C::FM; ++j)
#pragma unroll
            for (int t = 0; t < 16; ++t)
                acc[i][j][t] = 0;
    v4i px[C::FM], pw[C::FN], xlo[C::FM], xhi[C::FM], wlo[C::FN], whi[C::FN];
    constexpr int kSlots = C::FM * C::FN;                            // MFMAs per half unit
    constexpr int kHiOps = 4 * (C::FM + C::FN), kLoOps = 2 * kHiOps; // vector operations to widen one
    constexpr int kHiSlots = (kSlots + 1) / 2;                       // slots the odd nibbles are masked in
    auto read_unit = [&](unsigned ring, int s) {
        const uint8_t *stage = lds + ring + rd[s];
#pragma unroll
        for (int j = 0; j < C::FM; ++j)
            px[j] = *(const v4i *)(stage + j * kFrag * C::ROW_BYTES);
#pragma unroll
        for (int i = 0; i < C::FN; ++i)
            pw[i] = *(const v4i *)(stage + (C::BM + i * kFrag) * C::ROW_BYTES);
    };
    auto hi_op = [&](int op) {
        const int f = op / 4, d = op % 4;
        if (f < C::FM)
            xhi[f][d] = px[f][d] & himask;
        else
            whi[f - C::FM][d] = pw[f - C::FM][d] & himask;
    };
    auto lo_op = [&](int op) {
        const int f = op / 8, d = op % 4;
        const bool shift = (op & 4) == 0;
        if (f < C::FM)
            xlo[f][d] = shift ? px[f][d] << 4 : xlo[f][d] & himask;
        else
            wlo[f - C::FM][d] = shift ? pw[f - C::FM][d] << 4 : wlo[f - C::FM][d] & himask;
    };
    // The even-nibble MFMAs of the current unit, its odd nibbles masked behind the first of them;
    // then its packed registers are free: `between` reads the next unit into them.
    auto lo_phase = [&](auto &&between) {
        static_for<kSlots>([&](auto slot_tag) {
            constexpr int slot = decltype(slot_tag)::value, j = slot / C::FN, i = slot % C::FN;
            acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(xlo[j], wlo[i], acc[i][j], 0, 0, 0);
            if constexpr (slot < kHiSlots) {
#pragma unroll
                for (int op = slot * kHiOps / kHiSlots; op < (slot + 1) * kHiOps / kHiSlots; ++op)
                    hi_op(op);
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (slot == kHiSlots - 1) {
                between();
                __builtin_amdgcn_sched_barrier(0);
            }
        });
    };
    // The odd-nibble MFMAs; the next unit's even nibbles are widened behind them.
    auto hi_phase = [&](auto widen_next) {
        static_for<kSlots>([&](auto slot_tag) {
            constexpr int slot = decltype(slot_tag)::value, j = slot / C::FN, i = slot % C::FN;
            acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(xhi[j], whi[i], acc[i][j], 0, 0, 0);
            if constexpr (decltype(widen_next)::value) {
#pragma unroll
                for (int op = slot * kLoOps / kSlots; op < (slot + 1) * kLoOps / kSlots; ++op)
                    lo_op(op);
            }
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    // Waits until all but `younger` of the stages issued so far have landed, for every wave; by
    // then every wave has also finished reading the stage before (lgkmcnt), whose buffer may be
    // refilled.
    auto arrive = [&](int younger) {
        switch (younger) {
        case 0: wait_vm<0>(); break;
        case 1: wait_vm<C::CH>(); break;
        case 2: wait_vm<(C::NSTAGE > 2 ? 2 : 0) * C::CH>(); break;
        default: wait_vm<(C::NSTAGE > 3 ? 3 : 0) * C::CH>(); break;
        }
        __builtin_amdgcn_s_waitcnt(I4L_LGKM0);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    static_assert(C::NSTAGE <= 4, "arrive() knows up to three younger stages");
    arrive(min(KT, C::NSTAGE) - 1);
    read_unit(0, 0);
#pragma unroll
    for (int op = 0; op < kLoOps; ++op)
        lo_op(op);
    unsigned ring = 0;  // of the current stage
#pragma unroll 1
    for (int st = 0; st + 1 < KT; ++st) {
        const unsigned next = ring + C::STAGE_BYTES == C::LDS_BYTES ? 0u : ring + C::STAGE_BYTES;
        if constexpr (C::STEPS == 2) {
            lo_phase([&] { read_unit(ring, 1); });
            hi_phase(std::true_type{});
        }
        arrive(min(KT - 2 - st, C::NSTAGE - 2));  // stage st + 1
        lo_phase([&] {
            read_unit(next, 0);
            if (st + C::NSTAGE < KT)
                issue(st + C::NSTAGE, ring);
        });
        hi_phase(std::true_type{});
        ring = next;
    }
    if (wave * C::STEPS / 2 < last_pieces) {  // the last stage holds something of this wave's
        if constexpr (C::STEPS == 2) {
            lo_phase([&] { read_unit(ring, 1); });
            hi_phase(std::true_type{});
        }
        lo_phase([] {});
        hi_phase(std::false_type{});
    }

    // ---- the sums meet in LDS: [collecting wave][sending wave][KEEP] x 64 lanes
    __builtin_amdgcn_s_waitcnt(I4L_LGKM0);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    int kept[C::KEEP];
    int *const area = (int *)lds + lane;
    static_for<C::KG>([&](auto me_tag) {
        constexpr int me = decltype(me_tag)::value;
        if (wave == me) {
            static_for<C::KG>([&](auto to_tag) {
                constexpr int to = decltype(to_tag)::value;
                static_for<C::KEEP>([&](auto q) {
                    constexpr int r = to * C::KEEP + decltype(q)::value;
                    const int sum = acc[r / 16 % C::FN][r / 16 / C::FN][r % 16];
                    if constexpr (to == me)
                        kept[q()] = sum;
                    else
                        area[((to * (C::KG - 1) + (me < to ? me : me - 1)) * C::KEEP + q()) * 64] = sum;
                });
            });
        }
    });
    __syncthreads();
#pragma unroll
    for (int q = 0; q < C::KEEP; ++q) {
#pragma unroll
        for (int g = 0; g < C::KG - 1; ++g)
            kept[q] += area[((wave * (C::KG - 1) + g) * C::KEEP + q) * 64];
        kept[q] >>= 8;  // both operands carried a factor 16 (exact for every slice of K: each product is a multiple of 256)
    }

    // ---- slices of K: every wave leaves its sums in the slab of (tile, slice), waits until they
    //      have been acknowledged and counts itself in at the counter of (tile, wave).  The waves
    //      with one number hold the same sums in every slice's workgroup, so the last of them to
    //      arrive adds the others' up, stores, and puts the counter back to zero.  Nobody waits for
    //      anybody, and integer sums do not depend on who arrives when.  (Relaxed atomic operations
    //      at device scope go through to the level all workgroups share; fences at that scope
    //      would write back and invalidate the XCD's whole L2 instead.)
    if (slices > 1) {
        constexpr int kWords = C::KEEP / 2;
        u64 *const slabs = (u64 *)args.partial + (size_t)tile * slices * C::KG * kWords * 64 + (size_t)wave * kWords * 64 + lane;
        constexpr int kSlab = C::KG * kWords * 64;
#pragma unroll
        for (int q = 0; q < kWords; ++q)
            __hip_atomic_store(slabs + slice * kSlab + q * 64, (u64)(unsigned)kept[2 * q] | ((u64)(unsigned)kept[2 * q + 1] << 32),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        unsigned *const counter = args.arrivals + tile * C::KG + wave;
        unsigned before = 0;
        if (lane == 0)
            before = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        before = uniform(before);
        if (before != (unsigned)(slices - 1))
            return;
        if (lane == 0)
            __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        u64 got[kMaxSlices - 1][kWords];  // all loads go out together
#pragma unroll
        for (int p = 0; p < kMaxSlices - 1; ++p)
#pragma unroll
            for (int q = 0; q < kWords; ++q)
                got[p][q] = p < slices - 1 ? __hip_atomic_load(slabs + (p < slice ? p : p + 1) * kSlab + q * 64, __ATOMIC_RELAXED,
                                                               __HIP_MEMORY_SCOPE_AGENT)
                                           : 0ull;
#pragma unroll
        for (int p = 0; p < kMaxSlices - 1; ++p)
#pragma unroll
            for (int q = 0; q < kWords; ++q) {
                kept[2 * q] += (int)(unsigned)got[p][q];
                kept[2 * q + 1] += (int)(unsigned)(got[p][q] >> 32);
            }
    }

    // ---- store: 32 lanes write 32 consecutive columns.  Through a descriptor over the tile's
    //      rows: a lane outside the matrix gets an offset beyond it and the hardware drops the
    //      store.
    constexpr unsigned kElem = HALF_OUT ? 2u : 4u;
    const bool plain = !ep.bias && !ep.out;
    const int rows_left = M - m0, cols_left = N - n0;
    const size_t extent = ((size_t)(min(rows_left, C::BM) - 1) * N + min(cols_left, C::BN)) * kElem;
    __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc((uint8_t *)args.y + ((size_t)m0 * N + n0) * kElem, 0, (int)extent, 0x00020000);
    unsigned col_off[kCols];
#pragma unroll
    for (int i = 0; i < kCols; ++i)
        col_off[i] = col_of(i) < cols_left ? (unsigned)col_of(i) * kElem : 0x40000000u;
#pragma unroll
    for (int q = 0; q < C::KEEP; ++q) {
        const unsigned off = (row_of(q) < rows_left ? (unsigned)row_of(q) * (unsigned)N * kElem : 0x80000000u) + col_off[q / 16];
        if constexpr (HALF_OUT)
            __builtin_amdgcn_raw_buffer_store_b16(
                (unsigned short)epilogue_value16(ep, kept[q], bias_v[q / 16], rs_v[q], cs_v[q / 16]), rsrc, off, 0, 0);
        else
            __builtin_amdgcn_raw_buffer_store_b32(
                (unsigned)(plain ? kept[q] : epilogue_value32(ep, kept[q], bias_v[q / 16], rs_v[q], cs_v[q / 16])), rsrc, off, 0, 0);
    }
}

// The tiles, smallest grids first.
using Tile32x32 = GridTile<1, 1, 8, 4, 4, 2>;        // 64 KiB of LDS
using Tile64x32Short = GridTile<2, 1, 4, 4, 3, 2>;   // 72 KiB; four waves: less to bring together at the end
using Tile64x32Long = GridTile<2, 1, 8, 4, 3, 4>;    // 72 KiB; eight waves
using Tile64x64 = GridTile<2, 2, 4, 4, 2, 2>;        // 64 KiB

long tiles_of(int m, int n, int bm, int bn) { return (long)((m + bm - 1) / bm) * ((n + bn - 1) / bn); }

enum class Tile { k32x32, k64x32Short, k64x32Long, k64x64 };

// The smallest tile of which there is at most one per CU: more of the device works, and every
// CU pulls less.  Measured (us; 32 x 32 / 64 x 32 / 64 x 64): 100 x 1000 x 2048, 128 tiles of the
// first, 4.2 / 4.8 / 5.8; 333 x 1111 x 4096, 385 and 210: 7.4 / 6.6 / 8.2; 128 x 8192 x 4096, 512
// and 256: 13.0 / 9.9 / 9.4.  Eight waves on a 64 x 32 tile pay from K = 2048 on (100 x 1000 x
// 2048 4.83 / 4.82 with four / eight; 200 x 2000 x 512 3.5 / 3.9; 65 x 4096 x 4096 7.1 / 6.5).
Tile choose_tile(int m, int n, int k, const DeviceInfo &dev)
{
    if (tiles_of(m, n, 32, 32) <= dev.cu_count)
        return Tile::k32x32;
    if (tiles_of(m, n, 64, 32) <= dev.cu_count)
        return k > 2048 ? Tile::k64x32Long : Tile::k64x32Short;
    return Tile::k64x64;
}

// The split of K over workgroups: for 64 pieces of K and more, where one slice per tile leaves
// CUs without work (32 x 32 and 64 x 32 tiles) or, with 64 x 64 tiles, a second workgroup fits every
// CU.  The exchange costs some 2 us.  Measured, unsplit -> split: 200 x 136 x 16384 12.6 -> 7.9 us,
// 300 x 520 x 12288 10.6 -> 10.0, 100 x 2000 x 16384 12.7 -> 11.6, 128 x 4096 x 28672 25.2 -> 22.3,
// 128 x 4096 x 14336 14.8 -> 15.2 (nothing gained, nothing lost).
struct SplitPlan {
    Tile tile = Tile::k64x64;
    int slices = 1;
    size_t bytes = 0;  // of partial sums
};

SplitPlan plan_split(int m, int n, int k, const DeviceInfo &dev)
{
    constexpr int kMinPieces = 64, kMinPiecesPerSlice = 8;
    SplitPlan p;
    const int pieces = k / kPieceK;
    if (pieces < kMinPieces)
        return p;
    long tiles, most, waves, area;
    if (tiles_of(m, n, 32, 32) * 4 <= dev.cu_count) {
        p.tile = Tile::k32x32;
        tiles = tiles_of(m, n, 32, 32), most = dev.cu_count, waves = Tile32x32::KG, area = 32 * 32;
    } else if (tiles_of(m, n, 64, 32) * 2 <= dev.cu_count) {
        p.tile = Tile::k64x32Long;
        tiles = tiles_of(m, n, 64, 32), most = dev.cu_count, waves = Tile64x32Long::KG, area = 64 * 32;
    } else {
        tiles = tiles_of(m, n, 64, 64), most = 2l * dev.cu_count, waves = Tile64x64::KG, area = 64 * 64;
    }
    if (tiles * waves > kSkinnyArrivalWords)
        return p;
    for (int d = 2; d <= kMaxSlices && tiles * d <= most; ++d)
        if (pieces % d == 0 && pieces / d >= kMinPiecesPerSlice)
            p.slices = d;
    if (p.slices > 1)
        p.bytes = (size_t)tiles * p.slices * area * 4;
    return p;
}

template <class C>
hipError_t init_tile()
{
    hipError_t e = hipFuncSetAttribute((const void *)mfma_grid_kernel<C, false>, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS_BYTES);
    if (e == hipSuccess)
        e = hipFuncSetAttribute((const void *)mfma_grid_kernel<C, true>, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS_BYTES);
    return e;
}

struct Split {
    int slices = 1;
    void *partial = nullptr;
    unsigned *arrivals = nullptr;
};

template <class C>
hipError_t launch_tile(const void *a, const void *b, void *c, int m, int n, int k, const Split &split, const Epilogue &ep,
                       hipStream_t stream)
{
    const int tiles_m = (m + C::BM - 1) / C::BM, tiles_n = (n + C::BN - 1) / C::BN;
    // what the kernel assumes of a split: slices of whole pieces, a counter for every (tile, wave)
    if (split.slices > 1 &&
        (split.slices > kMaxSlices || k / kPieceK % split.slices != 0 || !split.partial || !split.arrivals ||
         (long)tiles_m * tiles_n * C::KG > kSkinnyArrivalWords))
        return hipErrorInvalidValue;
    auto *kern = ep.out >= kOutF16 ? mfma_grid_kernel<C, true> : mfma_grid_kernel<C, false>;
    kern<<<(unsigned)(tiles_m * tiles_n * split.slices), C::THREADS, C::LDS_BYTES, stream>>>(
        GridArgs{(const uint8_t *)a, (const uint8_t *)b, c, m, n, k, tiles_m, tiles_n, split.slices, (int *)split.partial, split.arrivals, ep});
    return hipGetLastError();
}

hipError_t launch(Tile tile, const void *a, const void *b, void *c, int m, int n, int k, const Split &split, const Epilogue &ep,
                  hipStream_t stream)
{
    switch (tile) {
    case Tile::k32x32:
        return launch_tile<Tile32x32>(a, b, c, m, n, k, split, ep, stream);
    case Tile::k64x32Short:
        return launch_tile<Tile64x32Short>(a, b, c, m, n, k, split, ep, stream);
    case Tile::k64x32Long:
        return launch_tile<Tile64x32Long>(a, b, c, m, n, k, split, ep, stream);
    default:
        return launch_tile<Tile64x64>(a, b, c, m, n, k, split, ep, stream);
    }
}

}  // namespace

hipError_t grid_init(const DeviceInfo &)
{
    hipError_t e = init_tile<Tile32x32>();
    if (e == hipSuccess)
        e = init_tile<Tile64x32Short>();
    if (e == hipSuccess)
        e = init_tile<Tile64x32Long>();
    if (e == hipSuccess)
        e = init_tile<Tile64x64>();
    return e;
}

bool grid_preferred(int m, int n, const DeviceInfo &dev) { return tiles_of(m, n, 128, 128) * 2 <= dev.cu_count; }

hipError_t launch_grid(const void *a, const void *b, void *c, int m, int n, int k, const Epilogue &ep, const DeviceInfo &dev,
                       hipStream_t stream)
{
    return launch(choose_tile(m, n, k, dev), a, b, c, m, n, k, Split{}, ep, stream);
}

size_t grid_split_bytes(int m, int n, int k, const DeviceInfo &dev)
{
    return grid_preferred(m, n, dev) ? plan_split(m, n, k, dev).bytes : 0;
}

hipError_t launch_grid_split(const void *a, const void *b, void *c, int m, int n, int k, void *workspace, unsigned *arrivals,
                             const Epilogue &ep, const DeviceInfo &dev, hipStream_t stream)
{
    const SplitPlan p = plan_split(m, n, k, dev);
    return launch(p.tile, a, b, c, m, n, k, Split{p.slices, workspace, arrivals}, ep, stream);
}

}  // namespace int4linear
