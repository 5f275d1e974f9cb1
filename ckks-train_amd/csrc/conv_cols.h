// The base conversion of one target fused with the column pass of its forward NTT: one tile of 4096
// coefficients is converted from the sources (y form, in coefficient order) straight into the
// registers of the column pass, so the converted limb never goes to memory in coefficient form.
// Written so that a host program can include it too (the CPU replay in tests/emu); the includer
// has included ntt_passes.h and conv_arith.h.
//
// Every target reads the sources again (at most 8 tiles of 32 KB, which the targets of one tile
// share in the L2 of their XCD) and forms its own overflow estimate: 5 more operations per word and
// source than a conversion of all targets at once, against one write and one read of the limb. With
// at most 4 sources that always pays (the 32 x 32 product at N = 2^15: 913 -> 805 us for the
// conversions and column passes). With more, the kernel is bound by VALU and latency (73 % busy at 4
// waves per SIMD): 256 switches at 2^16 take 7.23 ms against 6.51 ms as two kernels, sixteen hoisted
// rotations the same, one switch 63 against 73 us and one launch less per conversion.
#pragma once

#include "conv_arith.h"
#include "conv_col_ref.h"
#include "ntt_passes.h"

namespace ckh {

namespace fast {

// Work item -> (ref, tile, target): items are ordered [conversion][tile][target], so item / tiles
// is some ref of the item's conversion.
CKH_DEV u32 conv_col_item(const ConvColRef& R, u32 item, u32 tiles, u32& tile) {
    const u32 local = item - R.first * tiles;
    tile = local / R.ntgt;
    return local % R.ntgt;
}

// Words a thread loads ahead of their conversion: as many as leave 4 waves per SIMD (3 with 8 sources).
template <u32 MAXS>
constexpr u32 CONV_AHEAD = MAXS <= 2 ? 8 : MAXS <= 4 ? 4 : 2;

// W words of target g, word k that of coefficient base + (k << shift), as a column pass takes them: f64
// primes signed below 2 q, integer primes below 4 q.
template <u32 W, u32 MAXS, class Ar, class Tgt>
CKH_DEV void conv_words(const Ar& ar, const ConvSrc* srcs, const ConvColRef& R, const Tgt& g, const PrimeConst* pc,
                        u32 log_n, u32 base, u32 shift, typename Ar::V (&v)[W]) {
    constexpr u32 G = CONV_AHEAD<MAXS> < W ? CONV_AHEAD<MAXS> : W;
    // An absent source reads the first one; its constants are 0.
    u64 off[MAXS];
    double inv[MAXS];
#pragma unroll
    for (u32 j = 0; j < MAXS; ++j) {
        off[j] = j < R.nsrc ? (u64)j << log_n : 0;
        inv[j] = j < R.nsrc ? cst(srcs + R.src_first + j)->inv : 0.0;
    }
    const bool exact = R.nsrc > 1;
    auto words = [&](auto&& load_y, auto&& convert) {
#pragma unroll
        for (u32 k0 = 0; k0 < W; k0 += G) {
            u64 x[G][MAXS];
#pragma unroll
            for (u32 w = 0; w < G; ++w)
#pragma unroll
                for (u32 j = 0; j < MAXS; ++j) x[w][j] = glb(R.in + off[j])[base + ((k0 + w) << shift)];
#pragma unroll
            for (u32 w = 0; w < G; ++w) {
                double yd[MAXS], f = 0.0;
#pragma unroll
                for (u32 j = 0; j < MAXS; ++j) {
                    yd[j] = load_y(x[w][j]);
                    const double prod = yd[j] * inv[j];
                    f = f + prod;
                }
                v[k0 + w] = convert(x[w], yd, exact ? (u32)f : 0u);
            }
        }
    };
    if (R.small) {
        words([](u64 x) { return u2d(x); },
              [&](u64 (&y)[MAXS], double (&yd)[MAXS], u32 e) {
#pragma unroll
                  for (u32 j = 0; j < MAXS; ++j) {
                      y[j] -= WRAP_CENTER;
                      yd[j] -= (double)WRAP_CENTER;
                  }
                  return ar.from_wrapped(conv_wrap_small<MAXS>(g, y, yd, e, (double)e));
              });
    } else if constexpr (Ar::F64) {
        words([](u64 x) { return u64_to_f64_rn(x); },
              [&](u64 (&y)[MAXS], double (&yd)[MAXS], u32 e) { return ar.from_canon(conv_wrap_large<MAXS>(g, y, yd, e)); });
    } else {
        const PrimeConst C = pc_int(pc);
        words([](u64 x) { return u64_to_f64_rn(x); },
              [&](u64 (&y)[MAXS], double (&)[MAXS], u32 e) { return ar.from_canon(conv_dot60<MAXS>(g, C, y, e, exact)); });
    }
}

// The words of a tile in the column pass's k-layout.
template <u32 M, u32 MAXS, class Ar, class Tgt>
CKH_DEV void conv_tile(const Ar& ar, const ConvSrc* srcs, const ConvColRef& R, const Tgt& g, const PrimeConst* pc,
                       u32 log_n, u32 tile, u32 tid, typename Ar::V (&v)[16]) {
    constexpr u32 R2 = M - 4, TCL = TL - M, TC = 1u << TCL;
    const u32 B = log_n - M;
    conv_words<16, MAXS>(ar, srcs, R, g, pc, log_n, ((tid >> TCL) << B) + tile * TC + (tid & (TC - 1)), R2 + B, v);
}

}  // namespace fast
}  // namespace ckh
