// FP6-MFMA GEMM over signed-int4 operands for gfx950 (CDNA4), exact in int32.
//
// CDNA4's matrix cores run the 6-bit float format E2M3 at twice the int8 rate
// (v_mfma_scale_f32_32x32x64_f8f6f4: 32x32x64 per instruction in the time the int8
// instruction does 32x32x32), and E2M3 holds every signed 4-bit integer exactly:
// sign, two exponent bits and three mantissa bits encode n/8 for n = -15..15 as the plain
// sign-magnitude integer |n| with the sign in bit 5 (subnormals 0..7 are |n| itself, 8 is
// exponent 1 with mantissa 0).  The instruction is used without block scales (both scale
// arguments zero select the unscaled opcode, one instruction where the scaled one is a
// pair), so a product is n*m/64, the fp32 accumulator holds multiples of 1/64, which fp32
// represents exactly while |sum of n*m| < 2^24, i.e. for K * 64 < 2^24, and the store
// multiplies by 64 (exact) before the conversion to int32.  The launcher refuses larger K;
// the result is bit-identical to integer arithmetic (the tests compare it against the CPU
// oracle).
//
// Two kernels:
//   * fp6_convert_kernel rewrites packed s4 operands (rows x K/2 bytes) into FP6
//     "fragment-major" form in a workspace: for every block of 32 rows x 64 k the 24
//     bytes each of the 64 MFMA lanes feeds to the instruction, stored as 64 x 16 B
//     followed by 64 x 8 B.  Rows are padded with zeros to a multiple of the 256-row
//     tile.  One launch converts both operands.  HBM-bound: 0.5 B read and 0.75 B
//     written per element.
//   * fp6_gemm_kernel is a persistent, LDS-pipelined GEMM over those fragments.  Because
//     the workspace is already in the order lanes consume it, global->LDS is a linear
//     direct-to-LDS copy, LDS->VGPR is one 16-byte and one 8-byte read per lane per
//     fragment at consecutive addresses (no swizzle, no bank conflicts), and the main loop
//     contains no VALU work at all.  Grids of few tiles run on kernels_fp6_grid.hip, or here as
//     slices of K whose partial sums a second kernel adds up (plan_gemm).
//
// Order of k inside a fragment is whatever the converter produces; it only has to be the
// same for both operands, which it is because both go through the same converter.
#include "kernels.h"
#include "fp6_format.h"
#include "grid_tail.h"

#include <type_traits>
#include <utility>

namespace int4linear {

namespace {

typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

#define I4L_LDS(p) ((__attribute__((address_space(3))) void *)(p))
// s_waitcnt immediate for gfx9: vmcnt[3:0] bits 3:0, vmcnt[5:4] bits 15:14, expcnt bits
// 6:4, lgkmcnt bits 11:8.  VM only leaves the others at "no wait".
#define I4L_WAIT_VM(n) ((0x0F70) | ((n) & 0xF) | ((((n) >> 4) & 0x3) << 14))
#define I4L_WAIT_LGKM0 0xC07F

constexpr int kStageBytes = 2 * kOperandStageBytes;                    // 48 KiB
constexpr int kStages = 3;
constexpr int kLdsBytes = kStages * kStageBytes;                       // 144 KiB
constexpr int kStaggerGroups = 8;                     // start groups within an XCD (power of two)
constexpr int kStaggerTicks = 120;                    // delay between groups, in 10-ns ticks of the constant clock
constexpr int kStaggerMinRounds = 2;                  // tiles per workgroup from which the start is staggered

// ---- converter --------------------------------------------------------------------------

// Four nibble values (one per byte of x, 0..15 meaning 0..7,-8..-1) -> four E2M3 codes
// (sign << 5 | magnitude), one per byte.
__device__ __forceinline__ unsigned fp6_codes(unsigned x)
{
    const unsigned s = x & 0x08080808u;   // sign bits
    const unsigned t = s >> 3;            // 1 in negative bytes
    const unsigned m = t * 15u;           // 0x0F in negative bytes
    const unsigned mag = (x ^ m) + t;     // 16 - x for negatives, x otherwise
    return mag | (s << 2);
}

// Four 6-bit codes, one per byte -> 24 contiguous bits.
__device__ __forceinline__ unsigned pack_codes(unsigned c)
{
    const unsigned t = (c & 0x003F003Fu) | ((c >> 2) & 0x0FC00FC0u);  // 12 bits per half
    return (t & 0x00000FFFu) | ((t >> 4) & 0x00FFF000u);
}

// One packed dword (8 nibbles) -> 48 bits of FP6 codes.
__device__ __forceinline__ unsigned long long fp6_from_dword(unsigned w)
{
    const unsigned even = pack_codes(fp6_codes(w & 0x0F0F0F0Fu));
    const unsigned odd = pack_codes(fp6_codes((w >> 4) & 0x0F0F0F0Fu));
    return (unsigned long long)even | ((unsigned long long)odd << 24);
}

// Workspace index of the fragment (tile, stage, k-fragment, row-fragment).
__device__ __forceinline__ size_t frag_offset(int tile, int stage, int kf, int rf, int stages)
{
    return ((((size_t)tile * stages + stage) * kFragsK + kf) * kFragsRows + rf) * (size_t)kFragBytes;
}

// One operand of a conversion launch.
struct ConvertJob {
    const uint8_t *src;   // packed s4, rows x k/2 bytes
    uint8_t *dst;         // fragment-major FP6
    int rows;             // real rows; rows up to the next multiple of 256 are written as zeros
    int row_blocks;       // 32-row blocks including the padding
};

typedef v4i v4i_dword_aligned __attribute__((aligned(4)));

constexpr int kConvK = 512;                          // k per converter workgroup
constexpr int kConvFrags = kConvK / kFragK;          // 8 fragments out
constexpr int kConvChunks = kConvK / 32;             // 16-byte input chunks per row
// LDS stride of a fragment being assembled: 64 bytes more than its size, so that the eight
// lanes of a wave that write the same lane slot of different fragments hit different banks.
constexpr int kConvFragLds = kFragBytes + 64;

// One workgroup converts 32 rows x 512 k of one operand: thread t reads the 16-byte chunks
// t%8 and t%8 + 8 of row t/8 (eight neighbouring lanes fetch a whole 128-byte line), the
// FP6 fragments are assembled in LDS, and the eight finished fragments (1536 contiguous
// bytes each) leave with full-line 16-byte stores.  blockIdx.y selects the operand and the
// 32-row block, so one launch converts both A and B.
// k is the operand's real K (a multiple of 8; the row stride is k/2 bytes), k_pad the next
// multiple of 128: k positions from k up to k_pad are written as zeros.  ALIGNED16: k is a
// multiple of 32, so every 16-byte chunk of a row is aligned and entirely inside the row.
template <bool ALIGNED16>
__global__ __launch_bounds__(256) void fp6_convert_kernel(ConvertJob ja, ConvertJob jb, int k, int k_pad)
{
    __shared__ __attribute__((aligned(16))) uint8_t out[kConvFrags * kConvFragLds];
    const bool second = (int)blockIdx.y >= ja.row_blocks;
    const ConvertJob job = second ? jb : ja;
    const int rb = second ? blockIdx.y - ja.row_blocks : blockIdx.y;
    const int r = threadIdx.x >> 3;
    const int c = threadIdx.x & 7;
    const int row = rb * kFragRows + r;
    const int stages = k_pad / kStageK;
    const int kchunk0 = blockIdx.x * kConvChunks;
    const int chunks_here = min(kConvChunks, (k_pad >> 5) - kchunk0);   // k_pad % 512 may be 128..384

    v4i w[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int kc = c + 8 * h;
        w[h] = (v4i){0, 0, 0, 0};
        const int k0 = (kchunk0 + kc) * 32;  // first k of the chunk
        const uint8_t *src = job.src + (size_t)row * (k >> 1) + (size_t)(kchunk0 + kc) * 16;
        if (ALIGNED16) {
            if (row < job.rows && k0 < k)
                w[h] = __builtin_nontemporal_load((const v4i *)src);
        } else if (row < job.rows) {
            if (k0 + 32 <= k) {
                w[h] = *(const v4i_dword_aligned *)src;
            } else {
#pragma unroll
                for (int d = 0; d < 3; ++d)
                    if (k0 + 8 * d < k)
                        w[h][d] = *(const int *)(src + 4 * d);
            }
        }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const unsigned long long q0 = fp6_from_dword((unsigned)w[h][0]);
        const unsigned long long q1 = fp6_from_dword((unsigned)w[h][1]);
        const unsigned long long q2 = fp6_from_dword((unsigned)w[h][2]);
        const unsigned long long q3 = fp6_from_dword((unsigned)w[h][3]);
        const unsigned long long o0 = q0 | (q1 << 48);
        const unsigned long long o1 = (q1 >> 16) | (q2 << 32);
        const unsigned long long o2 = (q2 >> 32) | (q3 << 16);
        const int kc = c + 8 * h;
        const int lane = (kc & 1) * 32 + r;
        uint8_t *frag = out + (kc >> 1) * kConvFragLds;
        *(v4i *)(frag + lane * 16) = (v4i){(int)o0, (int)(o0 >> 32), (int)o1, (int)(o1 >> 32)};
        *(v2i *)(frag + kFragLoBytes + lane * 8) = (v2i){(int)o2, (int)(o2 >> 32)};
    }
    __syncthreads();

    // Fragment f of this workgroup is k-fragment kfrag0 + f of the row block.
    const int tile = row / kTileRows;                 // uniform in the workgroup
    const int rf = rb % kFragsRows;
    const int kfrag0 = kchunk0 >> 1;
    const int frags_here = chunks_here >> 1;
    constexpr int kVecPerFrag = kFragBytes / 16;      // 96
    for (int i = threadIdx.x; i < frags_here * kVecPerFrag; i += 256) {
        const int f = i / kVecPerFrag, v = i % kVecPerFrag;
        const int kfrag = kfrag0 + f;
        uint8_t *dst = job.dst + frag_offset(tile, kfrag / kFragsK, kfrag % kFragsK, rf, stages);
        *(v4i *)(dst + v * 16) = *(const v4i *)(out + f * kConvFragLds + v * 16);
    }
}

// ---- GEMM ---------------------------------------------------------------------------------

// 16 bytes per lane from sbase + voff + IMM straight into LDS at place + ring + IMM + 16 * lane
// (the hardware adds the instruction's constant on both sides, which is what a linear copy
// wants; the two scalar summands of the LDS address are added on the way into M0).
template <int IMM>
__device__ __forceinline__ void dma16(const void *sbase, unsigned voff, unsigned place, unsigned ring)
{
    static_assert(IMM >= 0 && IMM < 4096, "13-bit signed immediate");
    asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 offset:%4"
                 :
                 : "v"(voff), "s"(sbase), "s"(place), "s"(ring), "n"(IMM)
                 : "memory", "scc");
}

// Marks a value as used at this point of the program without generating code.
__device__ __forceinline__ void pin(const v16f &v) { asm volatile("" ::"v"(v)); }

__device__ __forceinline__ int opaque(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// Same XCD-aware grouped tile order as the int8 kernel: workgroup ids go round-robin
// over 8 XCDs; ids congruent mod 8 get consecutive positions of an 8-tile-row-tall,
// column-major grouped order so that concurrent tiles of one XCD share operand rows in L2.
__device__ __forceinline__ void tile_coords(int v, int total, int tiles_m, int tiles_n,
                                            int &tm, int &tn)
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

// WAVES_M x WAVES_N wavefronts per workgroup; each owns FM x FN MFMA tiles of 32x32.
template <int WAVES_M_, int WAVES_N_, int OCC_>
struct Fp6Config {
    static constexpr int WAVES_M = WAVES_M_, WAVES_N = WAVES_N_, OCC = OCC_;
    static constexpr int NWAVES = WAVES_M * WAVES_N;
    static constexpr int THREADS = NWAVES * 64;
    static constexpr int FM = kTileRows / kFragRows / WAVES_M;
    static constexpr int FN = kTileRows / kFragRows / WAVES_N;
    static constexpr int CHUNKS = kStageBytes / 1024;  // 1-KiB direct-to-LDS loads per stage
    static constexpr int CH = CHUNKS / NWAVES;         // per wave
    static constexpr int STORES = FM * FN * 16;        // dword stores per lane per tile
    static constexpr int SLOTS = FM * FN;              // MFMAs per unit (one k-fragment)
    static_assert(CHUNKS % NWAVES == 0 && CH % 2 == 0 && CH <= 63, "loads must split evenly");
};

// What the GEMM kernel is put together from.  The library builds WholeKernel and nothing else;
// ablation/fp6_ablation.cpp, which compiles this file again, passes variations of its own
// (derived from this one, with single members changed) to time what each part costs.
struct WholeKernel {
    static constexpr bool kStores = true;    // a finished tile is stored
    static constexpr bool kLoads = true;     // global -> LDS loads go on after the prologue
    static constexpr bool kLdsReads = true;  // LDS -> register reads go on after the prologue
    static constexpr bool kOwnTile = true;   // a tile reads its own operands (false: those of tile (0, 0), L2-resident)
    static constexpr bool kStagger = true;   // workgroups of an XCD start in groups (see the kernel)
    static constexpr bool kFences = true;    // every MFMA and its share of the housekeeping are fenced off from the scheduler
    // Called by lane 0 of wave 0 when the workgroup starts and after its last tile.
    __device__ static void stamp(const Epilogue &, int /* workgroup */, int /* 0: start, 1: end */) {}
};

// HALF_OUT: the build for the two output kinds of 16-bit elements (its own build, so that the
// one for 32-bit elements carries none of its code).
template <class C, bool HALF_OUT = false, class Parts = WholeKernel>
__global__ __launch_bounds__(C::THREADS, C::OCC) void fp6_gemm_kernel(
    const uint8_t *__restrict__ XW, const uint8_t *__restrict__ WW, int32_t *__restrict__ Y,
    int M, int N, int K, int tiles_m, int tiles_n, Epilogue ep)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / C::WAVES_N;
    const int wn = wave % C::WAVES_N;
    // gridDim.y > 1: few tiles and long K.  Slice y covers KT of the KT_all stages and stores its plain
    // partial sums into slab y of Y (M * N int32 each), which a second kernel adds up.
    const int KT_all = K / kStageK;
    const int KT = KT_all / (int)gridDim.y;
    const int slice = blockIdx.y;
    const int total_tiles = tiles_m * tiles_n;
    const int nblk = gridDim.x;
    const int bid = blockIdx.x;
    const bool ep_plain = !HALF_OUT && !ep.bias && !ep.row_scale && !ep.col_scale && !ep.out;
    if (bid >= total_tiles)
        return;
    const int my_tiles = (total_tiles - bid + nblk - 1) / nblk;
    // ---- load side: stage = 24 KiB of X fragments then 24 KiB of W fragments, copied
    //      linearly; wave w moves CH/2 consecutive 1-KiB chunks of either half, so that the
    //      chunks of a half differ only in the instruction's constant.
    const uint8_t *xptr = XW, *wptr = WW;  // wave-uniform: this tile's current stage
    int ld_it = 0, ld_k = 0;
    const unsigned lds_base = (unsigned)(size_t)I4L_LDS(lds);
    const unsigned lane16 = (unsigned)lane * 16u;
    constexpr int kHalfChunks = C::CH / 2;
    static_assert(kHalfChunks * 1024 <= 4096, "a wave's chunks of one half must be within reach of the constant");
    const unsigned ld_voff = lane16 + (unsigned)(wave * kHalfChunks * 1024);
    const unsigned place_x = lds_base + (unsigned)(wave * kHalfChunks * 1024);
    const unsigned place_w = place_x + (unsigned)kOperandStageBytes;
    unsigned wr_ring = 0;  // the prologue's: offset of the stage buffer being filled

    auto ld_setup_tile = [&](int it) {
        int tm, tn;
        tile_coords(bid + it * nblk, total_tiles, tiles_m, tiles_n, tm, tn);
        if constexpr (!Parts::kOwnTile)
            tm = tn = 0;
        xptr = XW + ((size_t)tm * KT_all + (size_t)slice * KT) * kOperandStageBytes;
        wptr = WW + ((size_t)tn * KT_all + (size_t)slice * KT) * kOperandStageBytes;
    };
    auto ld_chunk = [&](auto c, unsigned ring) {  // c < CH/2: X half, else W half; ring: the buffer's offset
        constexpr int cc = decltype(c)::value;
        if constexpr (cc < kHalfChunks)
            dma16<cc * 1024>(xptr, ld_voff, place_x, ring);
        else
            dma16<(cc - kHalfChunks) * 1024>(wptr, ld_voff, place_w, ring);
    };
    auto ld_advance = [&]() {
        wr_ring = wr_ring + kStageBytes == kLdsBytes ? 0u : wr_ring + kStageBytes;
        ++ld_k;
        xptr += kOperandStageBytes;
        wptr += kOperandStageBytes;
        if (ld_k == KT) {
            if (ld_it + 1 < my_tiles) {
                ld_k = 0;
                ++ld_it;
                ld_setup_tile(ld_it);
            } else {
                // Past the last stage the cursor stays on it: the loop keeps issuing loads
                // unconditionally, and these re-read valid data into buffers nobody reads.
                ld_k = KT - 1;
                xptr -= kOperandStageBytes;
                wptr -= kOperandStageBytes;
            }
        }
    };

    // Prologue: stages 0 and 1 in full and the first half of stage 2's loads.  From then on
    // every iteration gs finishes stage gs+2 in its first unit and begins stage gs+3 in its
    // second, so the loop body needs no branch around a load.
    ld_setup_tile(0);
    auto ld_chunks = [&]<int... CC>(std::integer_sequence<int, CC...>) {
        (ld_chunk(std::integral_constant<int, CC>{}, wr_ring), ...);
    };
#pragma unroll
    for (int s = 0; s < kStages - 1; ++s) {
        ld_chunks(std::make_integer_sequence<int, C::CH>{});
        ld_advance();
    }
    ld_chunks(std::make_integer_sequence<int, C::CH / 2>{});

    // ---- math side.  Unit u = (stage, k-fragment kf); its operands are FM X fragments
    //      and FN W fragments, each 6 VGPRs read as 16 + 8 bytes.  While the MFMAs of unit
    //      u run, the fragments of unit u+1 are read into the other register set.
    const unsigned x_rd = (unsigned)(wm * C::FM * kFragBytes) + lane16;
    const unsigned w_rd = (unsigned)(kOperandStageBytes + wn * C::FN * kFragBytes) + lane16;
    const unsigned hi_delta = (unsigned)kFragLoBytes - (unsigned)lane * 8u;  // from the 16-B to the 8-B part

    v16f acc[C::FN][C::FM];
    v4i xlo[2][C::FM], wlo[2][C::FN];  // first 128 bits of each fragment's 192
    v2i xhi[2][C::FM], whi[2][C::FN];  // last 64 bits
    int cur_it = 0, kk = 0;

    // Read instruction r (0 .. 2*(FM+FN)-1) of unit (st, kf) into register set p:
    // fragment r/2, 16-byte part for even r, 8-byte part for odd r; X fragments first.
    auto read_op = [&](unsigned ring, int kf, int p, int r) {  // ring: offset of the stage's buffer
        const uint8_t *base = lds + ring + kf * kFragsRows * kFragBytes;
        const int f = r >> 1;
        const bool is_x = f < C::FM;
        const int idx = is_x ? f : f - C::FM;
        const uint8_t *a = base + (is_x ? x_rd : w_rd) + idx * kFragBytes;
        if ((r & 1) == 0)
            (is_x ? xlo[p][idx] : wlo[p][idx]) = *(const v4i *)a;
        else
            (is_x ? xhi[p][idx] : whi[p][idx]) = *(const v2i *)(a + hi_delta);
    };
    auto frag = [](const v4i &lo, const v2i &hi) {
        return (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], 0, 0};
    };
    constexpr int kReads = 2 * (C::FM + C::FN);

    // The MFMAs of the unit held in register set p; `hook(slot)` is housekeeping placed
    // behind the MFMA of that slot.
    auto unit = [&](auto p_tag, auto &&hook) {
        constexpr int p = decltype(p_tag)::value;
        [&]<int... SLOT>(std::integer_sequence<int, SLOT...>) {
            ([&] {
                constexpr int j = SLOT / C::FN, i = SLOT % C::FN;
                acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
                    frag(xlo[p][j], xhi[p][j]), frag(wlo[p][i], whi[p][i]), acc[i][j], 2, 2, 0, 0, 0,
                    0);
                // An MFMA has no side effect, so nothing stops the optimiser from moving it
                // down to its next use, past the housekeeping meant to run in its shadow;
                // this empty statement "uses" the result here and keeps the MFMA in place.
                pin(acc[i][j]);
                if constexpr (Parts::kFences)
                    __builtin_amdgcn_sched_barrier(0);
                hook(std::integral_constant<int, SLOT>{});
                if constexpr (Parts::kFences)
                    __builtin_amdgcn_sched_barrier(0);
            }(), ...);
        }(std::make_integer_sequence<int, C::SLOTS>{});
    };

    // Housekeeping positions inside a unit of SLOTS slots: the kReads LDS reads of the
    // next unit go two per slot from slot 0 (so they have landed well before the unit
    // ends), the CH/2 direct-to-LDS loads one per slot from slot SLOTS/2.
    constexpr int kReadsPerSlot = 2;
    constexpr int kDmaFirstSlot = C::SLOTS / 2;
    static_assert(kReads <= kReadsPerSlot * C::SLOTS, "not enough slots for the LDS reads");
    static_assert(kDmaFirstSlot + C::CH / 2 <= C::SLOTS, "not enough slots for the loads");
    auto spread = [&](auto slot_tag, unsigned read_ring, int read_kf, int read_p, auto half_pos, unsigned load_ring) {
        constexpr int slot = decltype(slot_tag)::value;
        if constexpr (Parts::kLdsReads) {
#pragma unroll
            for (int r = slot * kReadsPerSlot; r < (slot + 1) * kReadsPerSlot && r < kReads; ++r)
                read_op(read_ring, read_kf, read_p, r);
        }
        if constexpr (Parts::kLoads && slot >= kDmaFirstSlot && slot < kDmaFirstSlot + C::CH / 2) {
            ld_chunk(std::integral_constant<int, decltype(half_pos)::value * (C::CH / 2) + slot - kDmaFirstSlot>{}, load_ring);
        }
    };

    // Workgroups that start together reach every tile end together, and the stores of all
    // tiles then queue for the same path to memory while no CU computes.  With two or
    // more tiles per workgroup the 32 workgroups of an XCD (ids congruent mod 8) therefore
    // start in eight groups about a microsecond apart: their tile ends stay that
    // far apart for the rest of the launch, which costs the spread once at the end and
    // saves most of the wait at every tile end before.  (The wait sits behind the first loads,
    // which travel meanwhile.)
    if (threadIdx.x == 0)
        Parts::stamp(ep, bid, 0);
    if (Parts::kStagger && total_tiles >= kStaggerMinRounds * nblk) {
        const int grp = (bid >> 3) & (kStaggerGroups - 1);
        const unsigned long long until = wall_clock64() + (unsigned long long)(grp * kStaggerTicks);
        while (wall_clock64() < until)
            __builtin_amdgcn_s_sleep(2);
    }

    // Stage 0 must have landed before the first read; stage 1 and half of stage 2 are
    // in flight behind it.
    __builtin_amdgcn_s_waitcnt(I4L_WAIT_VM(C::CH + C::CH / 2));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int r = 0; r < kReads; ++r)
        read_op(0u, 0, 0, r);
    if constexpr (!Parts::kLdsReads) {
#pragma unroll
        for (int r = 0; r < kReads; ++r)
            read_op(0u, 1, 1, r);
    }

    int stores_behind = 0;  // a tile has just been stored: its stores sit behind the loads waited for next
    // One iteration of the stage loop, for the stage whose buffer is ring position RING.  The
    // loop below is unrolled over the three positions, so that every LDS address is a
    // loop-invariant register plus a constant and every buffer offset a constant.
    auto clear_acc = [&]() {
#pragma unroll
        for (int i = 0; i < C::FN; ++i)
#pragma unroll
            for (int j = 0; j < C::FM; ++j)
#pragma unroll
                for (int t = 0; t < 16; ++t)
                    acc[i][j][t] = 0.f;
    };
    clear_acc();
    // Returns true after the block's last tile.  Whatever a stage does only at a tile's end
    // (store, clear the accumulators, test for the end) sits behind the one branch on kk.
    auto iteration = [&](auto ring_tag) -> bool {
        constexpr unsigned rd_cur = decltype(ring_tag)::value * kStageBytes;              // stage gs
        constexpr unsigned rd_next = (decltype(ring_tag)::value + 1) % kStages * kStageBytes;  // stage gs+1
        constexpr unsigned wr_first = (decltype(ring_tag)::value + 2) % kStages * kStageBytes; // stage gs+2
        constexpr unsigned wr_second = rd_cur;                                            // stage gs+3
        // ---- unit (gs, 0): reads unit (gs, 1); finishes the loads of stage gs+2
        unit(std::integral_constant<int, 0>{}, [&](auto slot_tag) {
            spread(slot_tag, rd_cur, 1, 1, std::integral_constant<int, 1>{}, wr_first);
            if constexpr (decltype(slot_tag)::value == C::SLOTS - 1)
                ld_advance();
        });

        // ---- between the units: every LDS read of stage gs has been issued; once they
        //      have returned (lgkmcnt 0) and every wave is here, the buffer of stage gs is
        //      free for stage gs+3.  Stage gs+1 must have landed: memory operations complete
        //      in order and normally one younger stage (gs+2) is in flight behind it.  In
        //      the first stage after a tile end that tile's C stores sit behind it as well:
        //      they are more than the counter can hold (63), so their issue has already
        //      waited for everything older, and no wait is wanted (one for CH would stall
        //      until the stores have drained).  The common case falls through the branch.
        {
            static_assert(C::STORES >= 64, "the stores of a tile must saturate the counter");
            asm volatile("s_cmp_lg_u32 %0, 0\n\t"
                         "s_cbranch_scc1 1f\n\t"
                         "s_waitcnt vmcnt(%1)\n"
                         "1:"
                         :
                         : "s"(stores_behind), "n"(C::CH)
                         : "scc", "memory");
            stores_behind = 0;
            __builtin_amdgcn_s_waitcnt(I4L_WAIT_LGKM0);
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        }

        // ---- unit (gs, 1): reads unit (gs+1, 0) (a stale buffer past the last stage, never
        //      multiplied into a stored tile); begins the loads of stage gs+3 into the
        //      buffer of stage gs
        unit(std::integral_constant<int, 1>{}, [&](auto slot_tag) {
            spread(slot_tag, rd_next, 0, 0, std::integral_constant<int, 0>{}, wr_second);
        });
        ++kk;
        if (kk != KT)
            return false;
        {
            // ---- store the tile.  X is the MFMA A operand: accumulator t of tile (i, j) is
            //   m = 32*j + 8*(t/4) + 4*(lane/32) + t%4,  n = 32*i + lane%32,
            // so one dword store writes two rows of 32 consecutive n (128 B each).
            int tm, tn;
            tile_coords(bid + cur_it * nblk, total_tiles, tiles_m, tiles_n, tm, tn);
            const int m0 = tm * kTileRows, n0 = tn * kTileRows;
            const int rows_left = M - m0;  // > 0
            const int cols_left = N - n0;  // > 0
            int32_t *ybase = Y + (size_t)slice * (size_t)M * (size_t)N + (size_t)m0 * N + n0;
            const size_t slab_rows = rows_left < kTileRows ? rows_left : kTileRows;
            const size_t extent = ((slab_rows - 1) * (size_t)N + (size_t)(cols_left < kTileRows ? cols_left : kTileRows)) * 4u;
            __amdgpu_buffer_rsrc_t rsrc =
                __builtin_amdgcn_make_buffer_rsrc(ybase, 0, (int)extent, 0x00020000);
            // A lane outside the matrix gets an offset part so large that the sum falls
            // outside the descriptor's range and the hardware drops the store.
            const int lm = opaque(wm * C::FM * kFragRows + (lane >> 5) * 4);
            const int ln = opaque(wn * C::FN * kFragRows + (lane & 31));
            const unsigned lm_off = (unsigned)lm * (unsigned)N * 4u;
            unsigned col_off[C::FN];
#pragma unroll
            for (int i = 0; i < C::FN; ++i) {
                const int ncol = ln + i * kFragRows;
                col_off[i] = ncol < cols_left ? (unsigned)ncol * 4u : 0x40000000u;
            }
            if constexpr (!Parts::kStores) {
                pin(acc[0][0]);
            } else if (ep_plain) {
#pragma unroll
                for (int j = 0; j < C::FM; ++j) {
#pragma unroll
                    for (int t = 0; t < 16; ++t) {
                        const int dm = j * kFragRows + 8 * (t / 4) + (t % 4);  // uniform
                        const unsigned row_off = lm + dm < rows_left ? lm_off + (unsigned)dm * (unsigned)N * 4u : 0x80000000u;
#pragma unroll
                        for (int i = 0; i < C::FN; ++i) {
                            const int v = (int)(acc[i][j][t] * kUnscale);
                            __builtin_amdgcn_raw_buffer_store_b32((unsigned)v, rsrc, row_off + col_off[i], 0, 2 /* nt */);
                        }
                    }
                }
            } else {
                // Epilogue operands of this lane's columns and rows (clamped inside the
                // matrix).  These ordinary loads make the compiler wait for everything in
                // flight, prefetched stages included: the price of an epilogue, kept out of
                // the plain path above.
                int bias_v[C::FN];
                float cs_v[C::FN];
#pragma unroll
                for (int i = 0; i < C::FN; ++i) {
                    const int ncol = ln + i * kFragRows;
                    const int nn = n0 + (ncol < cols_left ? ncol : cols_left - 1);
                    bias_v[i] = ep.bias ? ep.bias[nn] : 0;
                    cs_v[i] = ep.col_scale ? ep.col_scale[nn] : 1.f;
                }
                if constexpr (!HALF_OUT) {
#pragma unroll
                    for (int j = 0; j < C::FM; ++j) {
                        float rs[16];
#pragma unroll
                        for (int t = 0; t < 16; ++t) {
                            const int dm = j * kFragRows + 8 * (t / 4) + (t % 4);
                            rs[t] = ep.row_scale ? ep.row_scale[m0 + (lm + dm < rows_left ? lm + dm : rows_left - 1)] : 1.f;
                        }
#pragma unroll
                        for (int t = 0; t < 16; ++t) {
                            const int dm = j * kFragRows + 8 * (t / 4) + (t % 4);  // uniform
                            const unsigned row_off = lm + dm < rows_left ? lm_off + (unsigned)dm * (unsigned)N * 4u : 0x80000000u;
#pragma unroll
                            for (int i = 0; i < C::FN; ++i) {
                                const int v = epilogue_value32(ep, (int)(acc[i][j][t] * kUnscale), bias_v[i], rs[t], cs_v[i]);
                                __builtin_amdgcn_raw_buffer_store_b32((unsigned)v, rsrc, row_off + col_off[i], 0, 2 /* nt */);
                            }
                        }
                    }
                } else {
                    // The half-width kinds: a descriptor over the same tile of an output of
                    // two-byte elements, every offset halved (slices of K are int32 always).
                    __amdgpu_buffer_rsrc_t rsrc16 = __builtin_amdgcn_make_buffer_rsrc(
                        (uint8_t *)Y + ((size_t)m0 * N + n0) * 2u, 0, (int)(extent / 2u), 0x00020000);
#pragma unroll
                    for (int j = 0; j < C::FM; ++j) {
                        float rs[16];
#pragma unroll
                        for (int t = 0; t < 16; ++t) {
                            const int dm = j * kFragRows + 8 * (t / 4) + (t % 4);
                            rs[t] = ep.row_scale ? ep.row_scale[m0 + (lm + dm < rows_left ? lm + dm : rows_left - 1)] : 1.f;
                        }
#pragma unroll
                        for (int t = 0; t < 16; ++t) {
                            const int dm = j * kFragRows + 8 * (t / 4) + (t % 4);  // uniform
                            const unsigned row_off = lm + dm < rows_left ? (lm_off + (unsigned)dm * (unsigned)N * 4u) / 2u : 0x80000000u;
#pragma unroll
                            for (int i = 0; i < C::FN; ++i) {
                                const int v = epilogue_value16(ep, (int)(acc[i][j][t] * kUnscale), bias_v[i], rs[t], cs_v[i]);
                                __builtin_amdgcn_raw_buffer_store_b16((unsigned short)v, rsrc16,
                                                                      row_off + (col_off[i] == 0x40000000u ? col_off[i] : col_off[i] / 2u), 0, 2 /* nt */);
                            }
                        }
                    }
                }
            }
            kk = 0;
            ++cur_it;
            stores_behind = 1;
            clear_acc();
        }
        return cur_it == my_tiles;
    };
    for (;;) {
        if (iteration(std::integral_constant<int, 0>{}))
            break;
        if (iteration(std::integral_constant<int, 1>{}))
            break;
        if (iteration(std::integral_constant<int, 2>{}))
            break;
    }
    if (threadIdx.x == 0)
        Parts::stamp(ep, bid, 1);
}

// Eight wavefronts of 64 (m) x 128 (n), two per SIMD, one workgroup per CU.  (With four
// fragments along n a wave's stores of one accumulator row cover 512 contiguous bytes of a
// row of C; measured 0-2 % faster than 128 (m) x 64 (n) on every large shape tried.)
using Fp6Cfg = Fp6Config<4, 2, 1>;

size_t operand_ws_bytes(int rows, int k)
{
    const size_t tiles = (size_t)(rows + kTileRows - 1) / kTileRows;
    return tiles * (size_t)((k + kStageK - 1) / kStageK) * (size_t)kOperandStageBytes;
}

}  // namespace

bool fp6_supports(int m, int n, int k)
{
    // fp32 accumulation of products bounded by 64 stays exact while K * 64 < 2^24.  The
    // converter pads K to a multiple of 128 with zeros, so any K % 8 == 0 is fine.
    // Rows: the converter's grid (one y block per 32 rows of either operand) ends at 65535
    // and the store addresses a tile's 256 rows of C with byte offsets below 2^30.
    constexpr int kMaxRows = (1 << 20) - kTileRows;
    return m >= 1 && n >= 1 && m <= kMaxRows && n <= kMaxRows && k >= 8 && k % 8 == 0 && k <= (1 << 18) - kStageK;
}

namespace {

// How a GEMM of converted operands runs.
struct GemmPlan {
    bool grid = false;   // on kernels_fp6_grid.hip
    int slices = 1;      // of K
    size_t partial = 0;  // bytes of their partial sums
};

// The most slices of K of the large kernel that leave a workgroup per CU, 2048 k per slice and equal slices.
int large_slices(long tiles, int stages, const DeviceInfo &dev)
{
    if (tiles * 4 > dev.cu_count)  // (two slices of 128 tiles gain nothing over 128 unsplit ones)
        return 1;
    for (int d = kGridMaxSlices; d > 1; --d)
        if (tiles * d <= dev.cu_count && stages % d == 0 && stages / d >= 16)
            return d;
    return 1;
}

// `room`: the most bytes the large kernel's partial sums may take.  Grids of up to one 64 x 64 tile per CU run on those
// tiles.  Beyond, they read every operand four times as often as 256 x 256 tiles do, and what the larger
// ones lose is idle CUs, or the partial sums' way to memory and back: the least of the three
// estimates below, in us, without the converter.  us, 64 x 64 / 256 x 256 in slices of K (their number) / unsplit:
// 1024 x 4096 x 8192 54 / 65 (4) / -; x 12296 74 / - / 70; x 16384 98 / 85 (4) / -; x 20488 115 / - / 109; x
// 28672 161 / 116 (4) / -; 768 x 3072 x 16376 72 / 55 (4) / -; 1000 x 3000 x 12296 58 / - / 67; 512 x 4096 x 16384
// 60 / 73 (8) / -, x 28680 98 / 80 (5) / -; 600 x 3300 x 28680 121 / 89 (5) / -.  Unsplit 256 x 256 tiles fall behind
// again once the operands outgrow the memory-side cache (512 x 8192 x 24584, 160 MB: 158 / - / 161; x 32776 252 / - / 281).
// Rows of C that are no multiple of 4 long are stored and added up a dword at a time: 64 x 64 / slices, 2026 x 1819 x 10728
// 68 / 87 (4), 256 x 13066 x 10232 80 / 95 (4), 2692 x 1086 x 14240 68 / 82 (4), though 482 x 6845 x 14888 96 / 84 (3); a
// multiple of 4: 4743 x 704 x 13016 82 / 69 (3), 1482 x 2220 x 12256 75 / 70 (4).  (The converter is in these times.)
GemmPlan plan_gemm(int m, int n, int k, const DeviceInfo &dev, size_t room)
{
    constexpr size_t kCachedOperands = 140u << 20;
    const long tiles64 = grid_tiles(m, n, 64, 64), tiles = grid_tiles(m, n, kTileRows, kTileRows);
    const int stages = (k + kStageK - 1) / kStageK;
    GemmPlan p;
    p.grid = fp6_grid_preferred(m, n, dev);
    if (!p.grid)
        return p;
    if (tiles64 > dev.cu_count) {
        const double per_k = 3.7e-3 * k;
        const double small = 8 + 0.98e-3 * k * (double)((tiles64 + dev.cu_count - 1) / dev.cu_count);
        const bool cached = operand_ws_bytes(m, k) + operand_ws_bytes(n, k) <= kCachedOperands;
        const double whole = cached ? 10 + per_k : small;
        const int d = large_slices(tiles, stages, dev);
        const size_t slabs = (size_t)d * (size_t)m * (size_t)n * 4u;
        const double slab_rate = n % 4 == 0 ? 4.2e6 : 2.8e6;  // bytes per us
        const double split = d > 1 && slabs <= room ? 10 + per_k / d + (2 * d + 1) * 4. * m * n / slab_rate : small;
        if (split < small && split <= whole)
            return GemmPlan{false, d, slabs};
        if (whole < small)
            return GemmPlan{};
    }
    p.slices = fp6_grid_slices(m, n, k, dev, &p.partial);
    return p;
}

}  // namespace

size_t fp6_workspace_bytes(int m, int n, int k, const DeviceInfo &dev, size_t limit)
{
    const size_t operands = operand_ws_bytes(m, k) + operand_ws_bytes(n, k);
    if (dev.cu_count <= 0)
        return operands;
    // (partial sums: whole multiples of the output's size)
    const size_t out = (size_t)m * (size_t)n * 4u;
    const size_t partial = plan_gemm(m, n, k, dev, limit > operands ? limit - operands : 0).partial;
    return operands + (partial + out - 1) / out * out;
}

hipError_t fp6_init(const DeviceInfo &dev)
{
    if (dev.lds_per_cu < kLdsBytes)
        return hipErrorInvalidConfiguration;
    hipError_t e = fp6_grid_init(dev);
    if (e != hipSuccess)
        return e;
    e = hipFuncSetAttribute((const void *)fp6_gemm_kernel<Fp6Cfg>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes);
    if (e != hipSuccess)
        return e;
    return hipFuncSetAttribute((const void *)fp6_gemm_kernel<Fp6Cfg, true>,
                               hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes);
}

size_t fp6_operand_bytes(int rows, int k) { return operand_ws_bytes(rows, k); }

namespace {

// whole_tiles: rows of zeros up to the next multiple of 256 are written as well (the large GEMM
// kernel reads them, the small-grid one reads 64-row pairs at most).
ConvertJob make_job(const void *src, void *dst, int rows, bool whole_tiles = true)
{
    const int unit = whole_tiles ? kTileRows : 2 * kFragRows;
    return ConvertJob{(const uint8_t *)src, (uint8_t *)dst, rows, (rows + unit - 1) / unit * (unit / kFragRows)};
}

int padded_k(int k) { return (k + kStageK - 1) / kStageK * kStageK; }

hipError_t launch_convert_jobs(const ConvertJob &ja, const ConvertJob &jb, int k, hipStream_t stream)
{
    const int yblocks = ja.row_blocks + jb.row_blocks;
    if (yblocks > 65535)
        return hipErrorInvalidValue;
    if (yblocks == 0)
        return hipSuccess;
    const int k_pad = padded_k(k);
    const dim3 grid((k_pad + kConvK - 1) / kConvK, yblocks);
    if (k % 32 == 0)
        fp6_convert_kernel<true><<<grid, 256, 0, stream>>>(ja, jb, k, k_pad);
    else
        fp6_convert_kernel<false><<<grid, 256, 0, stream>>>(ja, jb, k, k_pad);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_fp6_convert(const void *src, void *dst, int rows, int k, hipStream_t stream)
{
    return launch_convert_jobs(make_job(src, dst, rows), ConvertJob{nullptr, nullptr, 0, 0}, k, stream);
}

namespace {

// slices > 1: `c` is as many slabs of m * n partial sums and `ep` must be empty.
hipError_t launch_tiles(const void *a_conv, const void *b_conv, void *c, int m, int n, int k, int slices, const Epilogue &ep,
                        const DeviceInfo &dev, hipStream_t stream)
{
    using C = Fp6Cfg;
    const int tiles_m = (m + kTileRows - 1) / kTileRows;
    const int tiles_n = (n + kTileRows - 1) / kTileRows;
    const long total = (long)tiles_m * tiles_n;
    if (total > 0x7fffffffL || (size_t)kTileRows * (size_t)n * 4u > 0x40000000ull || (slices > 1 && ep.out >= kOutF16))
        return hipErrorInvalidValue;
    long grid = (long)dev.cu_count * C::OCC;
    if (grid > total)
        grid = total;
    auto *kern = ep.out >= kOutF16 ? fp6_gemm_kernel<C, true> : fp6_gemm_kernel<C>;
    kern<<<dim3((unsigned)grid, (unsigned)slices), C::THREADS, kLdsBytes, stream>>>(
        (const uint8_t *)a_conv, (const uint8_t *)b_conv, (int32_t *)c, m, n, padded_k(k), tiles_m, tiles_n, ep);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_fp6_gemm(const void *a_conv, const void *b_conv, void *c, int m, int n, int k,
                           const Epilogue &ep, const DeviceInfo &dev, hipStream_t stream)
{
    if (plan_gemm(m, n, k, dev, 0).grid)
        return launch_fp6_grid(a_conv, b_conv, c, m, n, k, 1, nullptr, nullptr, ep, dev, stream);
    return launch_tiles(a_conv, b_conv, c, m, n, k, 1, ep, dev, stream);
}

hipError_t launch_fp6(const void *a, const void *b, void *c, int m, int n, int k, void *workspace, size_t workspace_bytes,
                      unsigned *arrivals, const Epilogue &ep, const DeviceInfo &dev, hipStream_t stream)
{
    uint8_t *xws = (uint8_t *)workspace;
    uint8_t *wws = xws + operand_ws_bytes(m, k);
    uint8_t *partial = wws + operand_ws_bytes(n, k);
    const GemmPlan p = plan_gemm(m, n, k, dev, workspace_bytes - (size_t)(partial - xws));
    hipError_t e = launch_convert_jobs(make_job(a, xws, m, !p.grid), make_job(b, wws, n, !p.grid), k, stream);
    if (e != hipSuccess)
        return e;
    if (p.grid)
        return launch_fp6_grid(xws, wws, c, m, n, k, p.slices, partial, arrivals, ep, dev, stream);
    if (p.slices == 1)
        return launch_tiles(xws, wws, c, m, n, k, 1, ep, dev, stream);
    e = launch_tiles(xws, wws, partial, m, n, k, p.slices, Epilogue{}, dev, stream);
    return e == hipSuccess ? launch_splitk_reduce(partial, c, (size_t)m * (size_t)n, p.slices, n, ep, stream) : e;
}

}  // namespace int4linear
