// Small-grid form of the FP6 GEMM: converted operands whose 256 x 256 tiles are few.
//
// The waves of a workgroup share one tile of C and split K between them.  The converted form lies
// in the order MFMA lanes consume it, and a wave's k-fragments are nobody else's, so
// operands go from memory straight into registers at consecutive addresses: no LDS, no barrier
// before the sums meet, several fragments in flight per wave.  What bounds it is the rate at
// which a CU pulls operands through its L1 (about 100 bytes per ns): 64 x 64 tiles read every operand
// four times as often as 256 x 256 ones, which pays while those leave most of the device idle.
// Measured against the large kernel (us, converter included): 333 x 1111 x 4104, 10 tiles of 256 x 256,
// 32.9 -> 12.6; 256 x 1024 x 4104, 4 tiles, 28.7 -> 10.3; 512 x 4096 x 4104, 32 tiles, 33.5 -> 25.1; 2048 x 2048 x
// 2056, 64 tiles, 24.2 -> 23.3; 1024 x 4096 x 4104, 64 tiles, 32.3 -> 32.0; longer K: plan_gemm in kernels_fp6.hip.
#include "fp6_format.h"
#include "grid_tail.h"

namespace int4linear {

namespace {

typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

// KG waves, a tile of FM x FN fragments, DEPTH k-fragments in flight per wave.
template <int FM_, int FN_, int KG_, int DEPTH_, int WAVES_PER_SIMD_>
struct Fp6GridTile {
    static constexpr int FM = FM_, FN = FN_, KG = KG_, DEPTH = DEPTH_, OCC = WAVES_PER_SIMD_;
    static constexpr int THREADS = KG * 64;
    static constexpr int BM = FM * kFragRows, BN = FN * kFragRows;
    template <bool HALF_OUT>
    using Tail = GridTail<FM, FN, KG, HALF_OUT>;
    static constexpr int LDS_BYTES = Tail<false>::LDS_BYTES;
    static_assert(kTileRows % BM == 0 && kTileRows % BN == 0, "a tile lies inside one 256-row tile of the operand");
};

struct Fp6GridArgs {
    const uint8_t *x, *w;
    void *y;
    int m, n, units, tiles_m, tiles_n, slices;  // units: k-fragments in a row
    int *partial;
    unsigned *arrivals;
    Epilogue ep;
};

// Workgroup v computes slice v / tiles of K of tile v % tiles.
template <class C, bool HALF_OUT>
__global__ __launch_bounds__(C::THREADS, C::OCC) void fp6_grid_kernel(Fp6GridArgs args)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int slices = args.slices;
    const Epilogue &ep = args.ep;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tiles = args.tiles_m * args.tiles_n;
    const int slice = blockIdx.x / tiles;
    const int tile = blockIdx.x - slice * tiles;
    int tm, tn;
    grid_tile_coords(tile, tiles, args.tiles_m, args.tiles_n, tm, tn);
    const int m0 = tm * C::BM, n0 = tn * C::BN;

    // This wave's k-fragments: slice * units + wave, + KG, ...
    const int units = args.units / slices;
    const int mine = (units - wave + C::KG - 1) / C::KG;
    const size_t first = (size_t)(slice * units + wave) * kUnitBytes;
    const size_t tile_bytes = (size_t)args.units * kUnitBytes;
    const uint8_t *const xbase = args.x + (m0 / kTileRows) * tile_bytes + first + m0 % kTileRows / kFragRows * kFragBytes;
    const uint8_t *const wbase = args.w + (n0 / kTileRows) * tile_bytes + first + n0 % kTileRows / kFragRows * kFragBytes;
    const unsigned lo = lane * 16u, hi = kFragLoBytes + lane * 8u;
    v4i xlo[C::DEPTH][C::FM], wlo[C::DEPTH][C::FN];
    v2i xhi[C::DEPTH][C::FM], whi[C::DEPTH][C::FN];
    auto load = [&](auto d_tag, int i) {
        constexpr int d = decltype(d_tag)::value;
        const size_t at = (size_t)i * ((size_t)C::KG * kUnitBytes);
#pragma unroll
        for (int j = 0; j < C::FM; ++j) {
            xlo[d][j] = *(const v4i *)(xbase + at + j * kFragBytes + lo);
            xhi[d][j] = *(const v2i *)(xbase + at + j * kFragBytes + hi);
        }
#pragma unroll
        for (int j = 0; j < C::FN; ++j) {
            wlo[d][j] = *(const v4i *)(wbase + at + j * kFragBytes + lo);
            whi[d][j] = *(const v2i *)(wbase + at + j * kFragBytes + hi);
        }
    };
    static_for<C::DEPTH>([&](auto d) {
        if (d() < mine)
            load(d, d());
    });

    typename C::template Tail<HALF_OUT> tail;
    tail.lane = lane;
    tail.wave = wave;
    tail.m0 = m0;
    tail.n0 = n0;
    tail.M = args.m;
    tail.N = args.n;
    tail.fetch(ep);

    v16f acc[C::FN][C::FM];
#pragma unroll
    for (int i = 0; i < C::FN; ++i)
#pragma unroll
        for (int j = 0; j < C::FM; ++j)
#pragma unroll
            for (int t = 0; t < 16; ++t)
                acc[i][j][t] = 0.f;
    auto frag = [](const v4i &l, const v2i &h) { return (v8i){l[0], l[1], l[2], l[3], h[0], h[1], 0, 0}; };
#pragma unroll 1
    for (int u = 0; u < mine; u += C::DEPTH) {
        static_for<C::DEPTH>([&](auto d_tag) {
            constexpr int d = decltype(d_tag)::value;
            if (u + d < mine) {
#pragma unroll
                for (int j = 0; j < C::FM; ++j)
#pragma unroll
                    for (int i = 0; i < C::FN; ++i)
                        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(frag(xlo[d][j], xhi[d][j]), frag(wlo[d][i], whi[d][i]),
                                                                                    acc[i][j], 2, 2, 0, 0, 0, 0);
                if (u + d + C::DEPTH < mine)
                    load(d_tag, u + d + C::DEPTH);
            }
        });
    }

    // (every wave's share is exact in float, and so is the product with 64)
    tail.collect(lds, [&](auto i, auto j, auto t) { return (int)(acc[i()][j()][t()] * kUnscale); });
    if (slices > 1 && !tail.exchange(args.partial, args.arrivals, tile, slice, slices))
        return;
    tail.store(ep, args.y);
}

using Tile32x32 = Fp6GridTile<1, 1, 8, 4, 2>;
using Tile64x32 = Fp6GridTile<2, 1, 8, 4, 2>;
using Tile64x64 = Fp6GridTile<2, 2, 4, 3, 3>;

enum class Tile { k32x32, k64x32, k64x64 };

// The smallest tile of which there is at most one per CU (us, 32 x 32 / 64 x 32 / 64 x 64, converter
// included): 256 x 1024 x 4096, 256 tiles of the first, 8.7 / 10.1 / 12.1 (graph); 333 x 1111 x 4104,
// 385 and 210, 14.3 / 12.6 / 14.9; 512 x 4096 x 4096, 2048, 1024 and 512, 22.1 / 18.9 / 15.9.
Tile choose_tile(int m, int n, const DeviceInfo &dev)
{
    if (grid_tiles(m, n, 32, 32) <= dev.cu_count)
        return Tile::k32x32;
    return grid_tiles(m, n, 64, 32) <= dev.cu_count ? Tile::k64x32 : Tile::k64x64;
}

template <class C>
hipError_t init_tile()
{
    hipError_t e = hipFuncSetAttribute((const void *)fp6_grid_kernel<C, false>, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS_BYTES);
    if (e == hipSuccess)
        e = hipFuncSetAttribute((const void *)fp6_grid_kernel<C, true>, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS_BYTES);
    return e;
}

template <class C>
hipError_t launch_tile(const void *a, const void *b, void *c, int m, int n, int k, const GridSplit &split, const Epilogue &ep,
                       hipStream_t stream)
{
    const int tiles_m = (m + C::BM - 1) / C::BM, tiles_n = (n + C::BN - 1) / C::BN;
    const int stages = (k + kStageK - 1) / kStageK;
    if (!grid_split_valid(split, (long)tiles_m * tiles_n, C::KG, stages))
        return hipErrorInvalidValue;
    auto *kern = ep.out >= kOutF16 ? fp6_grid_kernel<C, true> : fp6_grid_kernel<C, false>;
    kern<<<(unsigned)(tiles_m * tiles_n * split.slices), C::THREADS, C::LDS_BYTES, stream>>>(
        Fp6GridArgs{(const uint8_t *)a, (const uint8_t *)b, c, m, n, stages * kFragsK, tiles_m, tiles_n, split.slices, (int *)split.partial,
                    split.arrivals, ep});
    return hipGetLastError();
}

}  // namespace

hipError_t fp6_grid_init(const DeviceInfo &)
{
    hipError_t e = init_tile<Tile32x32>();
    if (e == hipSuccess)
        e = init_tile<Tile64x32>();
    if (e == hipSuccess)
        e = init_tile<Tile64x64>();
    return e;
}

// Up to four 64 x 64 tiles per CU, i.e. 256 x 256 tiles on a quarter of the CUs when they are whole; long
// K decides between the two in plan_gemm (kernels_fp6.hip).
bool fp6_grid_preferred(int m, int n, const DeviceInfo &dev) { return grid_tiles(m, n, 64, 64) <= 4l * dev.cu_count; }

// Slices of K across workgroups: the most that leave at most two workgroups per CU (they fit), 4096 k
// per slice (the exchange takes about as long as 2000 k) and equal slices.
int fp6_grid_slices(int m, int n, int k, const DeviceInfo &dev, size_t *bytes)
{
    const Tile tile = choose_tile(m, n, dev);
    const int bm = tile == Tile::k32x32 ? 32 : 64, bn = tile == Tile::k64x64 ? 64 : 32;
    const int kg = tile == Tile::k64x64 ? Tile64x64::KG : Tile64x32::KG;
    const long tiles = grid_tiles(m, n, bm, bn), most = 2l * dev.cu_count;
    const int stages = (k + kStageK - 1) / kStageK;
    int slices = 1;
    if (fp6_grid_preferred(m, n, dev) && tiles * kg <= kSkinnyArrivalWords)
        for (int d = 2; d <= kGridMaxSlices && tiles * d <= most; ++d)
            if (stages % d == 0 && stages / d >= 32)
                slices = d;
    *bytes = slices > 1 ? (size_t)tiles * slices * bm * bn * 4 : 0;
    return slices;
}

hipError_t launch_fp6_grid(const void *a_conv, const void *b_conv, void *c, int m, int n, int k, int slices, void *partial,
                           unsigned *arrivals, const Epilogue &ep, const DeviceInfo &dev, hipStream_t stream)
{
    const GridSplit split{slices, partial, arrivals};
    switch (choose_tile(m, n, dev)) {
    case Tile::k32x32:
        return launch_tile<Tile32x32>(a_conv, b_conv, c, m, n, k, split, ep, stream);
    case Tile::k64x32:
        return launch_tile<Tile64x32>(a_conv, b_conv, c, m, n, k, split, ep, stream);
    default:
        return launch_tile<Tile64x64>(a_conv, b_conv, c, m, n, k, split, ep, stream);
    }
}

}  // namespace int4linear
