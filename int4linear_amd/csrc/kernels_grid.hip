// Small-grid form of the int8-MFMA GEMM: shapes whose 128 x 128 tiles would leave half of the CUs
// idle or more, or whose 64 x 96 tiles fit the device two to a CU, with K long enough for the larger
// tiles.  Same arithmetic as kernels_mfma.hip (packed s4 through LDS, nibbles widened to 16 times
// their value in int8 lanes, C = acc >> 8).
//
// What bounds such a grid is the time to get a CU's operands to it and the length of one
// wave's chain of instructions: with a tile per CU nothing else runs there.  Hence
//   * all waves of a workgroup share one tile of C and split every stage's K between them.  A wave
//     then owns a block of C large enough (64 x 96 to 64 x 32) that a widened fragment feeds
//     several MFMAs: 6 vector operations per MFMA instead of the 12 of 32 x 32 quadrants, where
//     the vector unit, not the matrix unit, sets the pace.  The sums meet in LDS at the end: each
//     wave collects one part of the tile and stores it.
//   * a stage is 512 of K: whole 128-byte lines of every row, one barrier.  (256 of K in a ring twice as
//     deep is slower: 128 x 14336 x 4096 13.6 instead of 12.4 us, 1000 x 3000 x 4096 20.1 instead of 18.7.)
//   * one set of packed and of widened operands is a pipeline: the even-nibble MFMAs of a unit run
//     while its odd nibbles are masked, its odd-nibble MFMAs while the next unit's even nibbles
//     are shifted and masked.  No registers for a second set, so three waves fit a SIMD.
//   * the epilogue's operands are fetched behind the first stage's loads, not after the last MFMA.
//   * neighbouring columns of tiles start at different stages of K (the order of K does not
//     matter to the sums), so that the CUs do not all miss on the same lines at the same time.  (All at
//     the first: 120 shapes on the larger tiles within 5 % either way, 0.2 % on average.)
// Measured against the 64 x 64 tile of four quadrants by two halves of K (mfma_pair64_kernel), back to back
// on operands that stay in the caches: 65 x 4096 x 4096 9.3 -> 6.6 us, 333 x 1111 x 4096 9.3 -> 6.7, 256 x
// 4096 x 4096 9.7 -> 8.5, 128 x 14336 x 4096 13.9 -> 12.2, 300 x 520 x 640 4.1 -> 3.7.  (Figures beside one
// another are from one run; another machine, or a profiler, moves them by up to a third together.)
//
// With few tiles and long K a tile's K is split over workgroups as well; they exchange partial sums
// through memory inside the same launch (see the kernel's end).
#include "grid_tail.h"

namespace int4linear {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

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

constexpr int kPieceK = 128;  // K comes in pieces of 128: 64 bytes of a row
constexpr int kFrag = kGridFrag;

// KG waves share a tile of FM x FN fragments; each takes 1 / KG of every stage's K.  NSTAGE stages
// ring in LDS.
template <int FM_, int FN_, int KG_, int NSTAGE_, int WAVES_PER_SIMD_>
struct GridTile {
    static constexpr int FM = FM_, FN = FN_, KG = KG_, NSTAGE = NSTAGE_, OCC = WAVES_PER_SIMD_;
    static constexpr int PIECES = 4;                    // of every row in a stage
    static constexpr int THREADS = KG * 64;
    static constexpr int BM = FM * kFrag, BN = FN * kFrag;
    static constexpr int ROW_BYTES = 64 * PIECES;       // of a row in a stage
    static constexpr int CHUNKS = ROW_BYTES / 16;
    static constexpr int LOAD_ROWS = 1024 / ROW_BYTES;  // rows one load instruction of a wave moves
    static constexpr int STAGE_BYTES = (BM + BN) * ROW_BYTES;
    static constexpr int LDS_BYTES = STAGE_BYTES * NSTAGE;
    static constexpr int CH = (BM + BN) / LOAD_ROWS / KG;  // loads per wave and stage
    static constexpr int STEPS = 2 * PIECES / KG;          // units of 64 k per wave and stage
    template <bool HALF_OUT>
    using Tail = GridTail<FM, FN, KG, HALF_OUT>;
    static_assert((BM + BN) / LOAD_ROWS % KG == 0, "loads split evenly");
    static_assert(STEPS == 1 || STEPS == 2, "");
    static_assert(Tail<false>::LDS_BYTES <= LDS_BYTES, "the sums meet in the ring's LDS");
    static_assert((NSTAGE - 1) * CH <= 63, "vmcnt is six bits");
    // LDS slot of 16-byte chunk c of row r is c ^ swizzle(r): sixteen lanes that read one chunk of
    // sixteen consecutive rows hit sixteen different 16-byte groups of the banks (no conflicts
    // counted).
    __device__ static int swizzle(int r) { return r & 15; }
};

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
    grid_tile_coords(tile, tiles, tiles_m, tiles_n, tm, tn);
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

    typename C::template Tail<HALF_OUT> tail;
    tail.lane = lane;
    tail.wave = wave;
    tail.m0 = m0;
    tail.n0 = n0;
    tail.M = M;
    tail.N = N;
    tail.fetch(ep);
#pragma unroll
    for (int st = 1; st < C::NSTAGE; ++st)
        if (st < KT)
            issue(st, st * C::STAGE_BYTES);

    // ---- math.  A unit is 64 k: two 16-byte chunks of a row, one per half of the wave; the even
    //      nibbles of a chunk feed one MFMA, the odd ones another.  This wave's units of a stage
    //      are wave * STEPS, ...
    const int fr = lane & 31;
    const int fg = lane >> 5;
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

    __builtin_amdgcn_s_waitcnt(I4L_LGKM0);  // every wave is done with the ring
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    // (both operands carried a factor 16: every product, and with it every wave's share, is a
    // multiple of 256)
    tail.collect(lds, [&](auto i, auto j, auto t) { return acc[i()][j()][t()] >> 8; });
    if (slices > 1 && !tail.exchange(args.partial, args.arrivals, tile, slice, slices))
        return;
    tail.store(ep, args.y);
}

// The tiles, smallest grids first.
using Tile32x32 = GridTile<1, 1, 8, 4, 2>;        // 64 KiB of LDS
using Tile64x32Short = GridTile<2, 1, 4, 3, 2>;   // 72 KiB; four waves: less to bring together at the end
using Tile64x32Long = GridTile<2, 1, 8, 3, 4>;    // 72 KiB; eight waves
using Tile64x64 = GridTile<2, 2, 4, 2, 2>;        // 64 KiB
using Tile64x96 = GridTile<2, 3, 4, 2, 2>;        // 80 KiB

enum class Tile { k32x32, k64x32Short, k64x32Long, k64x64, k64x96 };

// 128 x 128 tiles on half of the CUs at most.
bool few_tiles(int m, int n, const DeviceInfo &dev) { return grid_tiles(m, n, 128, 128) * 2 <= dev.cu_count; }

// The smallest tile of which there is at most one per CU: more of the device works, and every
// CU pulls less.  Measured (us; 32 x 32 / 64 x 32 / 64 x 64): 100 x 1000 x 2048, 128 tiles of the
// first, 4.2 / 4.8 / 5.8; 333 x 1111 x 4096, 385 and 210: 7.4 / 6.6 / 8.2; 128 x 8192 x 4096, 512
// and 256: 13.0 / 9.9 / 9.4.  Eight waves on a 64 x 32 tile pay from K = 2048 on (100 x 1000 x
// 2048 4.83 / 4.82 with four / eight; 200 x 2000 x 512 3.5 / 3.9; 65 x 4096 x 4096 7.1 / 6.5).
// Above that, 64 x 64 or 64 x 96, whichever leaves the busiest CU fewer columns; 64 x 96 if they are
// equal (five fragments are read and widened for six MFMAs, not four for four).  64 x 64 / 64 x 96 in us:
// 128 x 11008 x 4096, 344 and 230 tiles, 12.5 / 11.8; 1000 x 1500 x 2048, 376 and 256, 8.6 / 8.4; 128 x
// 14336 x 4096, 448 and 300, 13.5 / 16.2; 64 x 32768 x 1024, 512 and 342, 8.0 / 9.7.
Tile choose_tile(int m, int n, int k, const DeviceInfo &dev)
{
    if (grid_tiles(m, n, 32, 32) <= dev.cu_count)
        return Tile::k32x32;
    if (grid_fits_narrow_tiles(m, n, dev))
        return k > 2048 ? Tile::k64x32Long : Tile::k64x32Short;
    const auto columns = [&](int bn) { return (grid_tiles(m, n, 64, bn) + dev.cu_count - 1) / dev.cu_count * bn; };
    return columns(64) < columns(96) ? Tile::k64x64 : Tile::k64x96;
}

// K from which the 64 x 64 and 64 x 96 tiles pay: `from`, or 1024 if every stage is full (a last stage of one
// piece takes the time of four).  int32, us, the other form / this one, up to 128 tiles of 128 x 128:
// 1024 x 1024 x 512 4.35 / 4.5, x 1024 5.15 / 5.15, x 1152 5.4 / 5.7, x 1408 5.8 / 5.75, x 1920 6.5 / 6.3; 1000 x 1500 x
// 640 6.1 / 6.6, x 1024 7.0 / 6.7, x 1152 7.2 / 7.4, x 1408 7.8 / 7.5; beyond: 1000 x 3000 x 512 7.9 / 7.9, x 1024 9.4 / 9.0,
// x 1152 9.5 / 10.6, x 2176 12.6 / 14.3, x 2560 14.1 / 13.8, x 2688 14.2 / 15.0, x 3200 15.8 / 16.3, x 3328 16.3 / 16.2,
// x 4096 18.6 / 18.0; 2048 x 1280 x 1664 10.6 / 12.1, x 2048 11.9 / 11.6, x 2304 12.7 / 13.0, x 2816 14.0 / 14.0.
bool long_enough(int k, int from)
{
    constexpr int kStageK = Tile64x96::PIECES * kPieceK;
    return k >= from || (k >= 1024 && k % kStageK == 0);
}

// The split of K over workgroups: for 64 pieces of K and more, where one slice per tile leaves
// CUs without work (32 x 32 and 64 x 32 tiles) or, with 64 x 64 tiles, a second workgroup fits every
// CU.  The exchange costs some 2 us.  Measured, unsplit -> split: 200 x 136 x 16384 12.6 -> 7.9 us,
// 300 x 520 x 12288 10.6 -> 10.0, 100 x 2000 x 16384 12.7 -> 11.6, 128 x 4096 x 28672 25.2 -> 22.3,
// 128 x 4096 x 14336 14.8 -> 15.2 (nothing gained, nothing lost).  K that the few slices of the smaller
// tiles do not divide goes to four and more slices of a larger one if it is long and they fit the CUs: 112 pieces
// and more (us, unsplit / in five or seven slices: 242 x 133 x 17024 13.3 / 8.9, 229 x 329 x 15232 12.4 / 10.5, 299 x 553 x
// 16000 12.85 / 11.85; more workgroups than CUs 104 x 1907 x 14720 12.6 / 13.1, three slices 119 x 1387 x 14976 12.5 /
// 12.6 and with weights from HBM 12.5 / 16.1, shorter K 557 x 289 x 8832 8.65 / 10.2).
struct SplitPlan {
    Tile tile = Tile::k64x64;
    int slices = 1;
    size_t bytes = 0;  // of partial sums
};

SplitPlan plan_split(int m, int n, int k, const DeviceInfo &dev)
{
    constexpr int kMinPieces = 64, kLongPieces = 112, kMinPiecesPerSlice = 8;
    SplitPlan p;
    const int pieces = k / kPieceK;
    if (pieces < kMinPieces)
        return p;
    // (`least`, `most`: slices and workgroups)
    const auto split = [&](Tile tile, int bm, int bn, int waves, int least, long most) {
        const long tiles = grid_tiles(m, n, bm, bn);
        if (tiles * waves > kSkinnyArrivalWords)
            return;
        for (int d = least; d <= kGridMaxSlices && tiles * d <= most; ++d)
            if (pieces % d == 0 && pieces / d >= kMinPiecesPerSlice) {
                p.tile = tile;
                p.slices = d;
                p.bytes = (size_t)tiles * d * bm * bn * 4;
            }
    };
    const int cus = dev.cu_count;
    const bool tiles32 = grid_tiles(m, n, 32, 32) * 4 <= cus, tiles64x32 = grid_tiles(m, n, 64, 32) * 2 <= cus;
    if (tiles32)
        split(Tile::k32x32, 32, 32, Tile32x32::KG, 2, cus);
    else if (tiles64x32)
        split(Tile::k64x32Long, 64, 32, Tile64x32Long::KG, 2, cus);
    else
        split(Tile::k64x64, 64, 64, Tile64x64::KG, 2, 2l * cus);
    if (p.slices == 1 && pieces >= kLongPieces && tiles32)
        split(Tile::k64x32Long, 64, 32, Tile64x32Long::KG, 4, cus);
    if (p.slices == 1 && pieces >= kLongPieces && tiles64x32)
        split(Tile::k64x64, 64, 64, Tile64x64::KG, 4, cus);
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

template <class C>
hipError_t launch_tile(const void *a, const void *b, void *c, int m, int n, int k, const GridSplit &split, const Epilogue &ep,
                       hipStream_t stream)
{
    const int tiles_m = (m + C::BM - 1) / C::BM, tiles_n = (n + C::BN - 1) / C::BN;
    if (!grid_split_valid(split, (long)tiles_m * tiles_n, C::KG, k / kPieceK))
        return hipErrorInvalidValue;
    auto *kern = ep.out >= kOutF16 ? mfma_grid_kernel<C, true> : mfma_grid_kernel<C, false>;
    kern<<<(unsigned)(tiles_m * tiles_n * split.slices), C::THREADS, C::LDS_BYTES, stream>>>(
        GridArgs{(const uint8_t *)a, (const uint8_t *)b, c, m, n, k, tiles_m, tiles_n, split.slices, (int *)split.partial, split.arrivals, ep});
    return hipGetLastError();
}

hipError_t launch(Tile tile, const void *a, const void *b, void *c, int m, int n, int k, const GridSplit &split, const Epilogue &ep,
                  hipStream_t stream)
{
    switch (tile) {
    case Tile::k32x32:
        return launch_tile<Tile32x32>(a, b, c, m, n, k, split, ep, stream);
    case Tile::k64x32Short:
        return launch_tile<Tile64x32Short>(a, b, c, m, n, k, split, ep, stream);
    case Tile::k64x32Long:
        return launch_tile<Tile64x32Long>(a, b, c, m, n, k, split, ep, stream);
    case Tile::k64x96:
        return launch_tile<Tile64x96>(a, b, c, m, n, k, split, ep, stream);
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
    if (e == hipSuccess)
        e = init_tile<Tile64x96>();
    return e;
}

// Up to 128 tiles of 128 x 128, where mfma_pair64_kernel is the other choice: 64 x 32 and 32 x 32 tiles
// always, the larger ones once K is long enough.  Beyond, where it is mfma_pair_kernel: always up to
// 64 rows, half of what its tiles hold, and where 64 x 64 tiles fit the device two to a CU (int32, us, that
// kernel / this one: 700 x 2712, 473 of them, x 256 6.8 / 6.0, x 1152 8.9 / 7.7; 257 x 5464, 430, x 1920 10.5 / 8.2), so
// that they are the ones chosen; with 64 x 96 tiles once K is long enough (580 x 3500 x 640 7.5 / 8.5), which is
// sooner where C is written in 32 bits and has a bias or scales, which end that kernel's tiles later
// (with a bias: 386 x 6470 x 512 9.4 / 8.4, 418 x 4705 x 896 9.3 / 8.4, 1161 x 2474 x 640 9.7 / 9.3, 2009 x 1444 x 384 9.0 /
// 8.5, x 1152 equal, 429 x 5383 x 1792 12.7 / 11.6; float output: 924 x 2594 x 640 9.35 / 9.8, 424 x 5377 x 1152 equal, 410 x
// 5392 x 1280 11.05 / 10.6, 807 x 2734 x 2432 15.0 / 13.5, whole stages 619 x 4252 x 512 9.3 / 8.85; without either, and in 16 bits,
// that line stays: 309 x 9099 x 1280 10.1 / 10.4).
bool grid_preferred(int m, int n, int k, const Epilogue &ep, const DeviceInfo &dev)
{
    if (few_tiles(m, n, dev)) {
        const Tile tile = choose_tile(m, n, k, dev);
        return (tile != Tile::k64x64 && tile != Tile::k64x96) || long_enough(k, 1408);
    }
    if (grid_tiles(m, n, 64, 96) > 2l * dev.cu_count)
        return false;
    if (m <= 64 || grid_tiles(m, n, 64, 64) <= 2l * dev.cu_count)
        return true;
    if (ep.out == kOutF32)
        return k >= 1152 || k % 512 == 0;
    if (ep.out == kOutS32 && ep.bias)
        return k >= 384;
    return long_enough(k, k % 512 == 128 ? 3328 : 2816);
}

bool grid_fits_narrow_tiles(int m, int n, const DeviceInfo &dev) { return grid_tiles(m, n, 64, 32) <= dev.cu_count; }

hipError_t launch_grid(const void *a, const void *b, void *c, int m, int n, int k, const Epilogue &ep, const DeviceInfo &dev,
                       hipStream_t stream)
{
    return launch(choose_tile(m, n, k, dev), a, b, c, m, n, k, GridSplit{}, ep, stream);
}

size_t grid_split_bytes(int m, int n, int k, const DeviceInfo &dev)
{
    return few_tiles(m, n, dev) ? plan_split(m, n, k, dev).bytes : 0;
}

int grid_split_slices(int m, int n, int k, const DeviceInfo &dev)
{
    return few_tiles(m, n, dev) ? plan_split(m, n, k, dev).slices : 1;
}

hipError_t launch_grid_split(const void *a, const void *b, void *c, int m, int n, int k, void *workspace, unsigned *arrivals,
                             const Epilogue &ep, const DeviceInfo &dev, hipStream_t stream)
{
    const SplitPlan p = plan_split(m, n, k, dev);
    return launch(p.tile, a, b, c, m, n, k, GridSplit{p.slices, workspace, arrivals}, ep, stream);
}

}  // namespace int4linear
