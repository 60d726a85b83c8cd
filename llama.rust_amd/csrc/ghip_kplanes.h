// ghip_kplanes.h -- Q6_K weights as two int8 operands of the integer matrix
// cores, made in registers (ghip_kq.hip, ghip_moe.hip).
#pragma once
#include "ghip_common.h"

typedef int v4i __attribute__((ext_vector_type(4)));
typedef short v2s __attribute__((ext_vector_type(2)));

// 16 values p = s * (q - 32) as the planes p & 127 and p >> 7
DEV void kq_planes(uint4 q, int s, v4i &l, v4i &h) {
    const v2s s2 = {(short)s, (short)s}, m2 = {(short)(-32 * s), (short)(-32 * s)};
    const uint32_t x[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const v2s a = __builtin_bit_cast(v2s, __builtin_amdgcn_perm(0u, x[i], 0x0c010c00u)) * s2 + m2;
        const v2s b = __builtin_bit_cast(v2s, __builtin_amdgcn_perm(0u, x[i], 0x0c030c02u)) * s2 + m2;
        const uint32_t ua = __builtin_bit_cast(uint32_t, a), ub = __builtin_bit_cast(uint32_t, b);
        const v2s ha = a >> 7, hb = b >> 7;
        l[i] = (int)(__builtin_amdgcn_perm(ub, ua, 0x06040200u) & 0x7f7f7f7fu);
        h[i] = (int)__builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, hb), __builtin_bit_cast(uint32_t, ha), 0x06040200u);
    }
}
