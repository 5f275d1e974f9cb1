// Work descriptors of the narrow passes fused with a key inner product (narrow_passes.h).
#pragma once

#include "arith.h"

namespace ckh {

// A key inner product over one limb: sum_j digit_j key_j, digit j at dig + j dig_stride (own for digit
// own_j, when set), read through the Galois permutation when galois != 0. Key part j's b limb is at
// key + 2 j key_poly, its a limb key_poly further; a job covers both parts.
struct LimbIp {
    const u64* dig;
    u64 dig_stride;
    const u64* own;
    const u64* key;
    u64 key_poly;
    u64 galois;
    u32 ndig, own_j;
};

// out (part a: out_part words further) <- the inverse row pass of the inner product.
struct IpInvJob {
    LimbIp ip;
    u64* out;
    u64 out_part;
    u32 prime, pad;
};

// out_b / out_a <- (inner product - NTT(z)) inv (+ add), where t (part a: t_part words further) holds
// z's column pass.
struct IpFinJob {
    LimbIp ip;
    const u64* t;
    u64 t_part;
    u64 *out_b, *out_a;
    const u64 *add_b, *add_a;
    u64 inv, inv_s;
    FTw inv_f;
    u32 prime, add_galois;  // add_galois: add_b is read through this Galois permutation (0: as it is)
};

}  // namespace ckh
