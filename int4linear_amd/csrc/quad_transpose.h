// Lanes that have loaded 64 contiguous bytes of a row per quad hold MFMA fragments after this.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

namespace int4linear {

#if defined(__HIPCC__)
typedef int quad_v4i __attribute__((ext_vector_type(4)));

// Transposes a 4 x 4 arrangement of 16-byte values inside every quad of lanes: on return
// r[t] of lane j (j = lane % 4) holds what r[j] of lane t of the same quad held.  Two
// exchange steps (lane distance 2, then 1), each a quad permutation and a select.
__device__ __forceinline__ void quad_transpose(quad_v4i &r0, quad_v4i &r1, quad_v4i &r2, quad_v4i &r3, int lane)
{
    const bool up2 = (lane & 2) != 0, up1 = (lane & 1) != 0;
    auto exchange = [](quad_v4i &a, quad_v4i &b, bool upper, auto ctrl) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int fa = __builtin_amdgcn_mov_dpp(a[c], decltype(ctrl)::value, 0xF, 0xF, true);
            const int fb = __builtin_amdgcn_mov_dpp(b[c], decltype(ctrl)::value, 0xF, 0xF, true);
            a[c] = upper ? fb : a[c];
            b[c] = upper ? b[c] : fa;
        }
    };
    exchange(r0, r2, up2, std::integral_constant<int, 0x4E>{});  // quad_perm [2,3,0,1]
    exchange(r1, r3, up2, std::integral_constant<int, 0x4E>{});
    exchange(r0, r1, up1, std::integral_constant<int, 0xB1>{});  // quad_perm [1,0,3,2]
    exchange(r2, r3, up1, std::integral_constant<int, 0xB1>{});
}
#endif

}  // namespace int4linear
