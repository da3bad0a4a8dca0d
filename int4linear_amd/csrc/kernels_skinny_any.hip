// Weight streaming for up to 64 rows of X and any K that is a multiple of 8: the shapes whose rows
// of W do not split into whole 128-byte tiles (kernels_skinny.hip).  Packed operands are multiplied
// as they lie, in one launch without scratch memory; arithmetic as in kernels_skinny.hip
// (v_mfma_i32_16x16x64_i8 on nibbles widened to 16 times their value, C = acc >> 8).
//
// What bounds it is W's way from HBM, so the loads are chosen for their shape.  A row starts at
// any multiple of 4 bytes, which rules out direct-to-LDS loads of 16 bytes per lane but not plain
// ones: every quad of lanes reads 64 contiguous bytes of a row, four loads cover 256 bytes of 16
// rows, and a transposition inside the quads turns them into MFMA fragments.  The waves of a workgroup
// split K in units of 512; where the registers allow it each asks for its next unit before it
// multiplies the one it has.
// At the end of a row a chunk of 16 bytes that would run past it is read as the row's last 16 bytes,
// of X and of W alike, and the dwords of W that an earlier chunk has had already are zeroed:
// nothing is read outside a row, and no padded copy is made.
// Measured against converting both operands for the FP6 kernel: 16 x 4096 x 4104 16.6 -> 5 us, 16 x
// 14336 x 4160 30.2 -> 11.0, 64 x 14336 x 4160 29.9 -> 20.7, 16 x 28672 x 8200 96 -> 30.0 (3.9 TB/s), and against
// skinny_basic_kernel's fragment-form loads: see skinny_any_preferred_to_basic.
#include "kernels.h"
#include "quad_transpose.h"

namespace int4linear {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v4i_dword_aligned __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kUnitBytes = 256;  // of a row: 512 of K
constexpr int kAnyMaxK = 131071 - 127;  // |sum| <= 64 K, times 256, fits 32 bits

// FMX: 16-row groups of X.  R: 16-row groups of W per workgroup.  MAX_WAVES: the most waves it is
// launched with, which sets the registers a lane may have.
template <int FMX, int R, int MAX_WAVES>
__global__ __launch_bounds__(MAX_WAVES * 64) void skinny_any_kernel(const uint8_t *X, const uint8_t *W, void *Y, int M, int N, int K, Epilogue ep)
{
    constexpr bool kAskAhead = R + FMX <= (MAX_WAVES == 16 ? 2 : 4);  // two units of 16 (R + FMX) registers fit a lane
    extern __shared__ v4i partial[];  // [waves][R * FMX][64]
    const int waves = blockDim.x >> 6;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rowbytes = K >> 1;
    const int units = (rowbytes + kUnitBytes - 1) / kUnitBytes;
    const int n0 = blockIdx.x * 16 * R;
    const uint8_t *const w0 = W + (size_t)n0 * (unsigned)rowbytes;
    const int rows_here = N - n0;

    // Load t of a unit: this lane's quad q = lane / 4 reads row 4 * (q % 4) + t, bytes 64 * (q / 4) .. + 64.
    const int lrow = (lane >> 2 & 3) * 4;
    const int lbyte = (lane >> 4) * 64 + (lane & 3) * 16;
    unsigned w_off[R][4], x_off[FMX][4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
#pragma unroll
        for (int r = 0; r < R; ++r)
            w_off[r][t] = (unsigned)min(16 * r + lrow + t, rows_here - 1) * (unsigned)rowbytes;
#pragma unroll
        for (int f = 0; f < FMX; ++f)
            x_off[f][t] = (unsigned)min(16 * f + lrow + t, M - 1) * (unsigned)rowbytes;
    }
    struct Unit {
        v4i w[R][4], x[FMX][4];
    };
    auto load = [&](Unit &d, int u) {
        const unsigned at = (unsigned)min(u * kUnitBytes + lbyte, rowbytes - 16);
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int t = 0; t < 4; ++t)
                d.w[r][t] = __builtin_nontemporal_load((const v4i_dword_aligned *)(w0 + (w_off[r][t] + at)));
#pragma unroll
        for (int f = 0; f < FMX; ++f)
#pragma unroll
            for (int t = 0; t < 4; ++t)
                d.x[f][t] = *(const v4i_dword_aligned *)(X + (x_off[f][t] + at));
    };
    const int himask = (int)0xF0F0F0F0u;
    v4i acc[R][FMX];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int f = 0; f < FMX; ++f)
            acc[r][f] = (v4i){0, 0, 0, 0};
    // Afterwards register t holds chunk 4 * (lane / 16) + t of row lane % 16: the same chunks, hence
    // the same k, for W and X.
    auto multiply = [&](Unit &d, int u) {
#pragma unroll
        for (int r = 0; r < R; ++r)
            quad_transpose(d.w[r][0], d.w[r][1], d.w[r][2], d.w[r][3], lane);
#pragma unroll
        for (int f = 0; f < FMX; ++f)
            quad_transpose(d.x[f][0], d.x[f][1], d.x[f][2], d.x[f][3], lane);
        if ((u + 1) * kUnitBytes > rowbytes) {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int again = u * kUnitBytes + (lane >> 4) * 64 + t * 16 - (rowbytes - 16);  // bytes read before
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        d.w[r][t][q] = again > 4 * q ? 0 : d.w[r][t][q];
            }
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            v4i xlo[FMX], xhi[FMX];
#pragma unroll
            for (int f = 0; f < FMX; ++f) {
                xlo[f] = (d.x[f][t] << 4) & himask;
                xhi[f] = d.x[f][t] & himask;
            }
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const v4i wlo = (d.w[r][t] << 4) & himask, whi = d.w[r][t] & himask;
#pragma unroll
                for (int f = 0; f < FMX; ++f) {
                    acc[r][f] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wlo, xlo[f], acc[r][f], 0, 0, 0);
                    acc[r][f] = __builtin_amdgcn_mfma_i32_16x16x64_i8(whi, xhi[f], acc[r][f], 0, 0, 0);
                }
            }
        }
    };
    if constexpr (!kAskAhead) {
        for (int u = wave; u < units; u += waves) {
            Unit a;
            load(a, u);
            multiply(a, u);
        }
    } else if (wave < units) {
        Unit a, b;
        int u = wave;
        load(a, u);
        while (true) {
            if (u + waves < units)
                load(b, u + waves);
            multiply(a, u);
            u += waves;
            if (u >= units)
                break;
            if (u + waves < units)
                load(a, u + waves);
            multiply(b, u);
            u += waves;
            if (u >= units)
                break;
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int f = 0; f < FMX; ++f)
            partial[(wave * R * FMX + r * FMX + f) * 64 + lane] = acc[r][f];
    __syncthreads();
    for (int e = threadIdx.x; e < R * FMX * 64; e += waves * 64) {
        const int block = e >> 6, l = e & 63;
        v4i s = partial[e];
        for (int wv = 1; wv < waves; ++wv)
            s += partial[wv * R * FMX * 64 + e];
        s = s >> 8;
        const int m = block % FMX * 16 + (l & 15);
        const int n = n0 + block / FMX * 16 + 4 * (l >> 4);
        if (m < M) {
            const float rs = ep.row_scale ? ep.row_scale[m] : 1.f;
            by_output_width(ep, [&](auto half) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int nn = n + q < N ? n + q : N - 1;
                    s[q] = epilogue_value_of<half()>(ep, s[q], ep.bias ? ep.bias[nn] : 0, rs, ep.col_scale ? ep.col_scale[nn] : 1.f);
                }
                store_out4<half()>(Y, (size_t)m * N + n, s, N - n, n + 3 < N && (N & 3) == 0);
            });
        }
    }
}

// No more waves than units.  (As few as need no more turns than that was slower: 16 x 28672 x 8320
// 38 us with six waves, 30 with eight; three of eight working 16 x 65536 x 1152 19, three alone 12.7.)
template <int FMX, int R, int MAX_WAVES>
hipError_t launch_form(const void *a, const void *b, void *c, int m, int n, int k, const Epilogue &ep, hipStream_t stream)
{
    const int units = (k / 2 + kUnitBytes - 1) / kUnitBytes;
    const int waves = units < MAX_WAVES ? units : MAX_WAVES;
    skinny_any_kernel<FMX, R, MAX_WAVES><<<(unsigned)((n + 16 * R - 1) / (16 * R)), waves * 64, waves * R * FMX * 1024, stream>>>(
        (const uint8_t *)a, (const uint8_t *)b, c, m, n, k, ep);
    return hipGetLastError();
}

// Groups of W and waves per workgroup.  While 16 rows per CU hold W there is one group per workgroup,
// on sixteen waves where K gives them two units each and 128 registers hold a unit (16 x 4096 x
// 14344: 11.5 us with eight waves, 9.6 with sixteen; 32 rows of X 13.7 / 11.9).  Beyond, workgroups
// share a CU: with 16 rows of X one group each still (two: 28672 x 8200 34.3 instead of 30.3), with more
// a second group halves the traffic of X (32 x 28672 x 8200 42.7 instead of 51.8, 64 rows of X 57 instead of 70).
template <int FMX>
hipError_t launch_rows(const void *a, const void *b, void *c, int m, int n, int k, const Epilogue &ep, const DeviceInfo &dev, hipStream_t stream)
{
    const bool one_round = n <= dev.cu_count * 16;
    if constexpr (FMX == 1) {
        if (one_round)
            return launch_form<FMX, 1, 16>(a, b, c, m, n, k, ep, stream);
    } else {
        if (!one_round)
            return launch_form<FMX, 2, 8>(a, b, c, m, n, k, ep, stream);
        if constexpr (FMX == 2)
            if (k > 7168)
                return launch_form<FMX, 1, 16>(a, b, c, m, n, k, ep, stream);
    }
    return launch_form<FMX, 1, 8>(a, b, c, m, n, k, ep, stream);
}

}  // namespace

bool skinny_any_supports(int m, int n, int k) { return m >= 1 && m <= 64 && n >= 1 && k >= 32 && k % 8 == 0 && k <= kAnyMaxK; }

// Everywhere but for a few workgroups with a long chain each, where the FP6 kernel splits K over
// workgroups (us, this kernel / FP6): 64 x 128 x 16200 17.7 / 15.2, 64 x 256 x 12296 14.5 / 13.6, 64 x 256
// x 8200 10.5 / 11.0, 64 x 512 x 16200 17.7 / 18.7, 48 x 128 x 16200 14.2 / 15.2.
bool skinny_any_preferred(int m, int n, int k) { return !(m > 48 && n <= 256 && k > 8192); }

// K a multiple of 128: rows start on 64-byte boundaries, fragment-form loads of 64 bytes per row lose
// little, and skinny_basic_kernel needs no transposition.  Long K is faster here (us, this kernel / that
// one): 16 x 4096 x 14464 10.3 / 12.5, 64 x 4096 x 14464 18.7 / 26.8, 16 x 28672 x 8320 30 / 43, 33 x 28672
// x 8320 46 / 56; but 33 x 4096 x 14464 15.3 / 14.2, 33 x 4096 x 4224 7.4 / 5.8, 16 x 16384 x 3200 10.5 / 9.4.
bool skinny_any_preferred_to_basic(int m, int n, int k, const DeviceInfo &dev)
{
    return k > 8192 && (m <= 16 || m > 48 || n > dev.cu_count * 16);
}

hipError_t launch_skinny_any(const void *a, const void *b, void *c, int m, int n, int k, const Epilogue &ep, const DeviceInfo &dev,
                             hipStream_t stream)
{
    switch ((m + 15) / 16) {
    case 1:
        return launch_rows<1>(a, b, c, m, n, k, ep, dev, stream);
    case 2:
        return launch_rows<2>(a, b, c, m, n, k, ep, dev, stream);
    case 3:
        return launch_rows<3>(a, b, c, m, n, k, ep, dev, stream);
    default:
        return launch_rows<4>(a, b, c, m, n, k, ep, dev, stream);
    }
}

}  // namespace int4linear
