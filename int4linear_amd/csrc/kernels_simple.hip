// Simple kernels: the scalar cross-check GEMM (written to be obviously right and to accept
// every shape the packed layout allows), the memory-bound device packer and unpacker, a zero
// fill and the sum over split-K slabs.
#include "kernels.h"

namespace int4linear {

namespace {

constexpr int kTile = 16;       // outputs per block edge
constexpr int kChunkWords = 16; // 32-bit words (128 nibbles) of K staged per step

// Signed value of nibble `slot` (0..7) of a packed word: utils/packer.cpp:27.
__device__ __forceinline__ int nibble_s4(uint32_t word, int slot)
{
    int v = (int)((word >> (4 * slot)) & 0xFu);
    return (v & 8) ? v - 16 : v;
}

// C[i][j] = sum_l A[i][l] * B[j][l]; one thread per output, operands staged through
// LDS one 128-nibble chunk at a time.  test/test_correctness.cu:12-19 semantics.
__global__ __launch_bounds__(kTile *kTile) void simple_gemm_kernel(
    const uint32_t *__restrict__ a, const uint32_t *__restrict__ b, int32_t *__restrict__ c,
    int m, int n, int k_words, unsigned tile_row0, Epilogue ep)
{
    __shared__ uint32_t a_lds[kTile][kChunkWords + 1];
    __shared__ uint32_t b_lds[kTile][kChunkWords + 1];

    const int tx = threadIdx.x % kTile;  // column of C inside the tile
    const int ty = threadIdx.x / kTile;  // row of C inside the tile
    const long tile_row = (long)tile_row0 + blockIdx.y;  // a launch covers at most 65535 tile rows
    const long row = tile_row * kTile + ty;
    const long col = (long)blockIdx.x * kTile + tx;

    int acc = 0;
    for (int w0 = 0; w0 < k_words; w0 += kChunkWords) {
        // Thread (ty, tx) stages word tx of row ty of each operand tile.
        const int w = w0 + tx;
        const long a_row = tile_row * kTile + ty;
        const long b_row = (long)blockIdx.x * kTile + ty;
        a_lds[ty][tx] = (a_row < m && w < k_words) ? a[a_row * k_words + w] : 0u;
        b_lds[ty][tx] = (b_row < n && w < k_words) ? b[b_row * k_words + w] : 0u;
        __syncthreads();
        for (int ww = 0; ww < kChunkWords; ++ww) {
            const uint32_t aw = a_lds[ty][ww];
            const uint32_t bw = b_lds[tx][ww];
            for (int s = 0; s < 8; ++s)
                acc += nibble_s4(aw, s) * nibble_s4(bw, s);
        }
        __syncthreads();
    }
    if (row < m && col < n)
        store_out(ep, c, (size_t)(row * n + col),
                  epilogue_value(ep, acc, ep.bias ? ep.bias[col] : 0, ep.row_scale ? ep.row_scale[row] : 1.f,
                                 ep.col_scale ? ep.col_scale[col] : 1.f));
}

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef v4i v4i_dword_aligned __attribute__((aligned(4)));  // rows of any length start on a dword only

// Packer and unpacker are bound by memory: four bytes per element on the unpacked side, half a
// byte on the other.  Every lane moves 16 bytes per access, and rows are found without a
// 64-bit division per lane: a workgroup finds the row and column of its first item once
// (wave-uniform), and its lanes divide 32-bit distances from there.  One item per lane: two or
// four, which would have more loads in flight, measured the same on large arrays and slower on
// small ones (pack 16 x 4096 1.9 -> 2.3 us).
constexpr int kCodecThreads = 256;

// Row of a wave-uniform position (hardly any array needs the 64-bit division).
__device__ __forceinline__ long row_of(long position, int per_row)
{
    return position >> 32 ? position / per_row : (long)((unsigned)position / (unsigned)per_row);
}

// Row and column `distance` items after item `col0` of row `row0`, in rows of `per_row` items.
__device__ __forceinline__ void locate(unsigned distance, long row0, unsigned col0, unsigned per_row, long &row, unsigned &col)
{
    const unsigned c = col0 + distance;
    const unsigned down = c / per_row;
    row = row0 + down;
    col = c - down * per_row;
}

// utils/packer.cpp:3-18 on device arrays: one thread per destination word, its eight values
// read as two 16-byte loads.  FLAT: n is a multiple of 8, so words and groups of eight values
// correspond without regard to rows.  2048 x 4096, 37.7 MB moved: 19.3 -> 6.7 us (5.6 TB/s);
// 1999 x 4095 the same.
template <bool FLAT>
__global__ __launch_bounds__(kCodecThreads) void pack_kernel(const int *__restrict__ src, int *__restrict__ dst, long total,
                                                             int n, int words)
{
    const long first = (long)blockIdx.x * kCodecThreads;
    const long i = first + threadIdx.x;
    if (i >= total)
        return;
    v4i v[2] = {};
    if constexpr (FLAT) {
        v[0] = ((const v4i_dword_aligned *)(src + i * 8))[0];
        v[1] = ((const v4i_dword_aligned *)(src + i * 8))[1];
    } else {
        const long row0 = row_of(first, words);
        long row;
        unsigned w;
        locate(threadIdx.x, row0, (unsigned)(first - row0 * words), (unsigned)words, row, w);
        const int *from = src + row * n + (long)w * 8;
        const int left = n - (int)w * 8;  // values from here to the end of the row
        if (left >= 8) {
            v[0] = ((const v4i_dword_aligned *)from)[0];
            v[1] = ((const v4i_dword_aligned *)from)[1];
        } else {
#pragma unroll
            for (int s = 0; s < 7; ++s)
                if (s < left)
                    v[s / 4][s % 4] = from[s];
        }
    }
    unsigned word = 0;
#pragma unroll
    for (int s = 0; s < 8; ++s)
        word |= ((unsigned)v[s / 4][s % 4] & 0xFu) << (4 * s);
    dst[i] = (int)word;
}

// utils/packer.cpp:20-31 on device arrays: one thread per four consecutive destination
// elements, which go out as one 16-byte store.  FLAT: n is a multiple of 8, the four are half a
// source word.  Otherwise they may lie in two words of a row, or in several rows.
// 4096 x 4096, 75.5 MB moved: 26.6 -> 12.3 us (6.1 TB/s); 4097 x 4093: 26.9 -> 13.1 us,
// 40000 x 133 (in a graph): 10.5 -> 6.5 us.
template <bool FLAT>
__global__ __launch_bounds__(kCodecThreads) void unpack_kernel(const uint32_t *__restrict__ src, int *__restrict__ dst,
                                                               long count, int n, int words)
{
    const long first = (long)blockIdx.x * kCodecThreads * 4;
    const long i = first + threadIdx.x * 4;
    if (i >= count)
        return;
    unsigned nibbles = 0;
    if constexpr (FLAT) {
        nibbles = ((const unsigned short *)src)[i >> 2];
    } else {
        const long row0 = row_of(first, n);
        long row;
        unsigned col;
        locate(threadIdx.x * 4, row0, (unsigned)(first - row0 * n), (unsigned)n, row, col);
        const uint32_t *from = src + row * words;
        if (n >= 3) {
            // at most two rows: what is left of this one lies in one or two words, the rest in
            // the first word of the next
            const unsigned left = (unsigned)n - col;
            const uint32_t low = from[col >> 3], high = from[(left < 4 ? (unsigned)n - 1 : col + 3) >> 3];
            nibbles = (unsigned)((((unsigned long long)high << 32) | low) >> (4 * (col & 7)));
            if (left < 4 && i + left < count)
                nibbles = (nibbles & ((1u << (4 * left)) - 1)) | (from[words] << (4 * left));
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (i + q < count)
                    nibbles |= ((from[col >> 3] >> (4 * (col & 7))) & 0xFu) << (4 * q);
                if (++col == (unsigned)n) {
                    col = 0;
                    from += words;
                }
            }
        }
    }
    v4i v;
#pragma unroll
    for (int q = 0; q < 4; ++q)
        v[q] = (int)(nibbles << (28 - 4 * q)) >> 28;
    if (i + 3 < count) {
        *(v4i_dword_aligned *)(dst + i) = v;
    } else {
#pragma unroll
        for (int q = 0; q < 3; ++q)
            if (i + q < count)
                dst[i + q] = v[q];
    }
}

__global__ void zero_i32_kernel(int4 *__restrict__ dst4, int *__restrict__ dst, size_t vec_count,
                                size_t count)
{
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (size_t v = i; v < vec_count; v += stride)
        dst4[v] = make_int4(0, 0, 0, 0);
    for (size_t t = vec_count * 4 + i; t < count; t += stride)
        dst[t] = 0;
}

// Second kernel of the split-K forms: Y = epilogue(sum of the ksplit slabs), four outputs of
// one row per thread (VEC: n % 4 == 0) or one.
template <bool VEC>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const int32_t *__restrict__ partial,
                                                                int32_t *__restrict__ Y, size_t count, int ksplit,
                                                                int N, Epilogue ep)
{
    constexpr int kPer = VEC ? 4 : 1;
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * kPer;
    if (i >= count)
        return;
    int sum[kPer] = {};
    for (int s = 0; s < ksplit; ++s) {
        const int32_t *src = partial + (size_t)s * count + i;
        if constexpr (VEC) {
            const v4i v = __builtin_nontemporal_load((const v4i *)src);
#pragma unroll
            for (int q = 0; q < 4; ++q)
                sum[q] += v[q];
        } else {
            sum[0] += *src;
        }
    }
    const size_t row = i / (size_t)N;
    const int col = (int)(i - row * (size_t)N);
    const float rs = ep.row_scale ? ep.row_scale[row] : 1.f;
    by_output_width(ep, [&](auto half) {
#pragma unroll
        for (int q = 0; q < kPer; ++q)
            sum[q] = epilogue_value_of<half()>(ep, sum[q], ep.bias ? ep.bias[col + q] : 0, rs,
                                               ep.col_scale ? ep.col_scale[col + q] : 1.f);
        if constexpr (half() && VEC)  // i % 4 == 0: four half-width outputs are eight aligned bytes
            *(v2i *)((unsigned short *)Y + i) = (v2i){sum[0] | (sum[1] << 16), sum[2] | (sum[3] << 16)};
        else if constexpr (half())
            ((unsigned short *)Y)[i] = (unsigned short)sum[0];
        else if constexpr (VEC)
            *(v4i *)(Y + i) = (v4i){sum[0], sum[1], sum[2], sum[3]};
        else
            Y[i] = sum[0];
    });
}

}  // namespace

hipError_t launch_simple(const void *a, const void *b, void *c, int m, int n, int k,
                         const Epilogue &ep, hipStream_t stream)
{
    // The grid's y extent ends at 65535: more tile rows than that go out as several launches.
    const unsigned tile_rows = (unsigned)((m + kTile - 1) / kTile);
    for (unsigned row0 = 0; row0 < tile_rows; row0 += 65535u) {
        const unsigned rows = tile_rows - row0 < 65535u ? tile_rows - row0 : 65535u;
        const dim3 grid((n + kTile - 1) / kTile, rows);
        simple_gemm_kernel<<<grid, kTile * kTile, 0, stream>>>(
            (const uint32_t *)a, (const uint32_t *)b, (int32_t *)c, m, n, k / 8, row0, ep);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess)
            return e;
    }
    return hipSuccess;
}

hipError_t launch_pack(const int *src, int *dst, int m, int n, hipStream_t stream)
{
    const int words = n / 8 + (n % 8 != 0);
    const long total = (long)m * words;
    if (total == 0)
        return hipSuccess;
    constexpr int per_block = kCodecThreads;
    const unsigned grid = (unsigned)((total + per_block - 1) / per_block);
    if (n % 8 == 0)
        pack_kernel<true><<<grid, kCodecThreads, 0, stream>>>(src, dst, total, n, words);
    else
        pack_kernel<false><<<grid, kCodecThreads, 0, stream>>>(src, dst, total, n, words);
    return hipGetLastError();
}

hipError_t launch_unpack(const int *src, int *dst, int m, int n, hipStream_t stream)
{
    const int words = n / 8 + (n % 8 != 0);
    const long count = (long)m * n;
    if (count == 0)
        return hipSuccess;
    constexpr int per_block = kCodecThreads * 4;
    const unsigned grid = (unsigned)((count + per_block - 1) / per_block);
    if (n % 8 == 0)
        unpack_kernel<true><<<grid, kCodecThreads, 0, stream>>>((const uint32_t *)src, dst, count, n, words);
    else
        unpack_kernel<false><<<grid, kCodecThreads, 0, stream>>>((const uint32_t *)src, dst, count, n, words);
    return hipGetLastError();
}

hipError_t launch_zero_i32(int *dst, size_t count, hipStream_t stream)
{
    if (count == 0)
        return hipSuccess;
    // dst is 16-byte aligned (checked by the API layer), so the bulk goes out as int4.
    const size_t vec_count = count / 4;
    const int block = 256;
    size_t want = (vec_count + block - 1) / block;
    unsigned grid = (unsigned)(want < 1 ? 1 : (want > 8192 ? 8192 : want));
    zero_i32_kernel<<<grid, block, 0, stream>>>((int4 *)dst, dst, vec_count, count);
    return hipGetLastError();
}

hipError_t launch_splitk_reduce(const void *slabs, void *c, size_t count, int ksplit, int n, const Epilogue &ep,
                                hipStream_t stream)
{
    if (count == 0)
        return hipSuccess;
    if (n % 4 == 0)
        splitk_reduce_kernel<true><<<(unsigned)((count / 4 + 255) / 256), 256, 0, stream>>>(
            (const int32_t *)slabs, (int32_t *)c, count, ksplit, n, ep);
    else
        splitk_reduce_kernel<false><<<(unsigned)((count + 255) / 256), 256, 0, stream>>>(
            (const int32_t *)slabs, (int32_t *)c, count, ksplit, n, ep);
    return hipGetLastError();
}

}  // namespace int4linear
