// Centered exact fast base conversion: the tables of a conversion and the per-coefficient
// arithmetic of the vector kernel, written so that a host program can include it too (the CPU
// replay of the conversion in tests/emu). The includer has included arith.h and defines cst(p)
// (a pointer to read-only tables), pc_int(p) (a prime's integer-reduction constants) and glb(p)
// (a global-memory view of a pointer).
//
// For sources q_0..q_{k-1} (product Q) and coefficient-form residues x_j, every target r gets
//   y_j = [x_j + (q_j >> 1)]_{q_j} * (Q/q_j)^-1 mod q_j
//   e   = floor(sum_j f64(y_j) * f64(1/q_j))             (k > 1 only)
//   out = sum_j y_j (Q/q_j mod r) - e (Q mod r) - ((Q-1)/2 mod r)   mod r
// which is BaseConverter::convert_exact([x + h]_Q) - h
// (crates/ckks-train-core/src/baseconv.rs:171-233; keyswitch.rs:140-210; baseconv.rs:258-291,
// 459-511). The modular sums give unique residues in any order. The f64 estimate is the one
// non-modular step: it uses the CPU's exact sequence (round-to-nearest u64->f64 conversion,
// round-to-nearest product with the host-computed reciprocal, round-to-nearest sum in source
// order from +0.0, then floor), so every includer compiles it without FMA contraction.
//
// Conversions of at most 8 sources (WRAP_SMALL / WRAP_LARGE below) take one quotient for the whole
// sum T = sum_j y_j c_j + e (-Q) - (Q-1)/2: an f64 sum F of y_j (c_j / r) estimates T / r, and
// T - k r (k = rint(F)) is formed exactly modulo 2^64 from 32-bit halves, where its small size
// makes it exact. Per source and target that is three 32 x 32 multiply-adds and one f64 FMA,
// instead of a modular product each (7 operations), six piece products, or the nine operations of
// an exact 128-bit sum with its carries.
#pragma once

#include "arith.h"

namespace ckh {

constexpr u32 MAX_SRC = 16;
constexpr u32 WRAP_SRC = 8;  // sources of the single-quotient form

// One source prime q_j of a conversion from Q = prod q_j.
struct ConvSrc {
    u64 q;
    u64 h;               // q_j >> 1: [x + (Q-1)/2]_Q has residue x + h mod q_j
    u64 qhinv, qhinv_s;  // (Q / q_j)^-1 mod q_j
    double inv;          // 1.0 / f64(q_j), round to nearest (host computed)
    double qf;           // q_j as f64 (f64 path)
    double qhinv_f, qhinv_q;  // (Q / q_j)^-1 and its quotient by q_j, f64 path
    u32 fp;                   // q_j < 2^50
    u32 prime;                // index into the context's primes
};

// One target prime r of a conversion.
struct ConvTgt {
    u32 prime;  // index into the context's prime constants
    u32 limb;   // output limb index within the job's output polynomial
    u64 qmod, qmod_s;  // Q mod r
    u64 hmod;          // (Q - 1)/2 mod r
    u64 qhat[MAX_SRC];                   // (Q / q_j) mod r
    double qhat_f[MAX_SRC], qhat_q[MAX_SRC];      // f64 path: (Q / q_j) mod r and its quotient by r
    double qhat30_f[MAX_SRC], qhat30_q[MAX_SRC];  // split path: 2^30 (Q / q_j) mod r, quotient by r
    double qmod_f, qmod_q, hmod_f, rf, rinv;
    // nq = -Q mod r (e nq = -e Q mod r), nq_c the same centered in (-r/2, r/2].
    u64 nq;
    double nq_c;
    // Without the single-quotient form: TGT_INT: r at least 2^50, 128-bit integer sums; TGT_FP: r
    // and every source below 2^50, f64 products of the sources; TGT_SPLIT: r below 2^50 with
    // larger sources, each source split into 30-bit halves.
    u32 mode, wrap;
    // The single-quotient form (wrap): c_j centered in (-r/2, r/2] as a two's complement word and
    // its quotient by r (WRAP_LARGE: by 2^11 r); -Q mod r likewise; the negated divisor -r
    // (WRAP_LARGE: -2^11 r) and r itself; the sum's constant and its quotient.
    u64 cw[WRAP_SRC];
    double cq[WRAP_SRC];
    u64 nqw, nr, r, aw;
    double nqq, aq;
};

enum : u32 { TGT_INT = 0, TGT_FP = 1, TGT_SPLIT = 2 };
// k = rint(F) has to be within 2 of T / r (WRAP_SMALL) or of T / (2^11 r) (WRAP_LARGE). In units of 1, with at
// most 8 terms y c, c centered (|c| < r / 2) and its quotient rounded to nearest:
// WRAP_SMALL: every source below 2^50, any r. The sums run over y_j - 2^49 (the constant takes
// 2^49 sum_j c_j), so |y_j - 2^49| <= 2^49 and F grows by at most 2^48 per term, to 2^51 (where adding
// 1.5 2^52 still rounds to an integer). Errors: each c_j / r is off by 2^-55 at most, 2^-6 in its
// term, 1/8 in all; the FMAs round to half an ulp of 2^48 .. 2^51, 1/32 + 1/16 + 1/16 + 1/8 for the
// first four and 1/8 for each further one (1/4 where the last crosses 2^51), 0.91 in all; the e term
// 2^-50; rint 1/2. That is 1.53 for 8 sources (1.13 for 6), so |T - k r| < 2 r.
// WRAP_LARGE: r below 2^50, sources below 2^60, c_j / (2^11 r) at most 2^-12: F grows by 2^48 per
// term, the rounding of y_j to f64 (2^6) adds 2^-6 per term to the same errors, and the terms left
// out of F (e, the constant: below 5 r, 2^-8): 1.66 for 8 sources, so |T - 2^11 k r| < 2^12 r < 2^62;
// a second quotient of that remainder by r gives the residue.
enum : u32 { WRAP_NONE = 0, WRAP_SMALL = 1, WRAP_LARGE = 2 };
constexpr u64 WRAP_CENTER = 1ull << 49;
constexpr double WRAP_ROUND = 6755399441055744.0;        // 1.5 2^52: adding it rounds to an integer
constexpr u64 WRAP_ROUND_BITS = 0x4338000000000000ull;  // its bits

// A conversion: sources [src_first, src_first + nsrc) of the ConvSrc table (their input limbs
// are src_limb0 + j of the job's input), targets [tgt_first, tgt_first + ntgt) of the ConvTgt
// table. exact = use the f64 overflow estimate (nsrc > 1).
struct ConvPlan {
    u32 src_first, nsrc, tgt_first, ntgt, src_limb0, exact;
};

// One launch row: plan `plan`, input polynomial (its limb 0) at `in`, output at `out`.
struct ConvJob {
    const u64* in;
    u64* out;
    u32 plan, pad;
};

// Round-to-nearest u64 -> f64: both halves convert exactly and the sum rounds once.
CKH_DEV double u64_to_f64_rn(u64 v) {
    const double hi = (double)(u32)(v >> 32) * 4294967296.0;
    const double lo = (double)(u32)v;
    return hi + lo;
}

// The sources of one coefficient: y_j as integers and as f64, and the overflow estimate e.
template <u32 MAXS>
struct ConvY {
    u64 y[MAXS];
    double yd[MAXS];
    u64 e;
    bool small;  // every source below 2^50
};

// Reads the sources of coefficient c (absent ones are 0). yform: the input limbs already hold
// y_j = [x_j + h_j]_{q_j} (Q/q_j)^-1 mod q_j (YForm: an inverse NTT computed it in its last stage).
template <u32 MAXS, class In>
CKH_DEV void conv_sources(const ConvSrc* srcs, const ConvPlan& P, In inp, u32 n, u32 c, bool yform, ConvY<MAXS>& Y) {
    double f = 0.0;
    Y.small = true;
    // every word loaded before any is used: the loads of a coefficient are in flight together
    u64 xs[MAXS];
#pragma unroll
    for (u32 j = 0; j < MAXS; ++j) xs[j] = j < P.nsrc ? (u64)inp[(u64)(P.src_limb0 + j) * n + c] : (u64)0;
#pragma unroll
    for (u32 j = 0; j < MAXS; ++j) {
        Y.y[j] = 0;
        Y.yd[j] = 0.0;
        if (j < P.nsrc) {
            const auto* s = cst(srcs + P.src_first + j);
            const u64 x = xs[j];
            if (s->fp) {
                if (yform) {
                    Y.y[j] = x;
                    Y.yd[j] = u2d(x);
                } else {
                    double sv = u2d(x) + (double)s->h;
                    sv = sv >= s->qf ? sv - s->qf : sv;
                    double v = fmulmod(sv, s->qhinv_f, s->qhinv_q, s->qf);
                    v = v < 0.0 ? v + s->qf : v;
                    Y.yd[j] = v;
                    Y.y[j] = d2u(v);
                }
            } else {
                Y.y[j] = yform ? x : shoup(add_mod(x, s->h, s->q), s->qhinv, s->qhinv_s, s->q);
                Y.yd[j] = u64_to_f64_rn(Y.y[j]);
                Y.small = false;
            }
            if (P.exact) {
                const double prod = Y.yd[j] * s->inv;  // f64(y_j) to nearest, exact below 2^50
                f = f + prod;
            }
        }
    }
    Y.e = P.exact ? (u64)f : 0;  // f >= 0: truncation is floor
}

// l + (a b mod 2^64) from 32-bit halves: the low product joins l, the crossed ones m (read modulo
// 2^32: the word is l + m 2^32).
CKH_DEV void mad_wrap(u64& l, u64& m, u64 a, u64 b) {
    l += (u64)(u32)a * (u32)b;
    m += (u64)(u32)a * (u32)(b >> 32);
    m += (u64)(u32)(a >> 32) * (u32)b;
}
CKH_DEV u64 wrap_word(u64 l, u64 m) {
    CKH_OPAQUE(m);  // else only its low half is summed, as a multiply and an addition per product
    return l + ((u64)(u32)m << 32);
}

// x, or x - m when that is not negative (x below 2^63).
CKH_DEV u64 csub_sign(u64 x, u64 m) {
    const u64 d = x - m;
    return (int64_t)d < 0 ? x : d;
}

// One target g from the sources of a WRAP_SMALL conversion, y_j given minus 2^49: T - k r + 2 r,
// below 4 r.
template <u32 MAXS, class Tgt>
CKH_DEV u64 conv_wrap_small(const Tgt& g, const u64 (&y)[MAXS], const double (&yd)[MAXS], u32 e, double ed) {
    u64 l = g->aw + (g->r << 1), m = 0;
    double F = __builtin_fma(ed, g->nqq, g->aq);
    l += (u64)e * (u32)g->nqw;
    m += (u64)e * (u32)(g->nqw >> 32);
#pragma unroll
    for (u32 j = 0; j < MAXS; ++j) {
        mad_wrap(l, m, y[j], g->cw[j]);
        F = __builtin_fma(yd[j], g->cq[j], F);
    }
    // rint(F) as the low bits of F + 1.5 2^52 (the constant's own bits are in aw)
    mad_wrap(l, m, f64_bits(F + WRAP_ROUND), g->nr);
    return wrap_word(l, m);
}

// One target from the sources of a WRAP_LARGE conversion: congruent to T, below (1 + 2^-20) r.
template <u32 MAXS, class Tgt>
CKH_DEV u64 conv_wrap_large(const Tgt& g, const u64 (&y)[MAXS], const double (&yd)[MAXS], u32 e) {
    const u64 r = g->r;
    u64 l = g->aw + (r << 12), m = 0;
    double F = 0.0;
    l += (u64)e * (u32)g->nqw;
    m += (u64)e * (u32)(g->nqw >> 32);
#pragma unroll
    for (u32 j = 0; j < MAXS; ++j) {
        mad_wrap(l, m, y[j], g->cw[j]);
        F = __builtin_fma(yd[j], g->cq[j], F);
    }
    mad_wrap(l, m, f64_bits(F + WRAP_ROUND), g->nr);
    // U = T - 2^11 k r + 2^12 r in (0, 2^13 r): its quotient by r, rounded down from an estimate
    // 2^-20 low (so never too large, and too small by one at most for the last 2^-20 of r)
    const u64 U = wrap_word(l, m);
    const double ud = __builtin_fma((double)(u32)(U >> 32), 4294967296.0, (double)(u32)U);
    const double kd = __builtin_fma(ud, g->rinv, -0x1p-20);
    const u32 k = (u32)kd;  // a negative estimate (U < 2^-20 r) converts to 0
    return U - (u64)k * r;
}

// One target of at least 2^50 from sources of any size: the exact 128-bit sum, reduced.
template <u32 MAXS, class Tgt>
CKH_DEV u64 conv_dot60(const Tgt& g, const PrimeConst& C, const u64 (&y)[MAXS], u64 e, bool exact) {
    Dot60 acc;
#pragma unroll
    for (u32 j = 0; j < MAXS; ++j) acc.add(y[j], g->qhat[j]);
    u64 hi, lo;
    acc.get(hi, lo);
    u64 o = reduce128(hi, lo, C);
    if (exact) o = sub_mod(o, shoup(e, g->qmod, g->qmod_s, C.q), C.q);
    return sub_mod(o, g->hmod, C.q);
}

// Coefficient c of one conversion (plan P, input polynomial in_p, output out_p, N = n): the
// output words of targets [t0, t1). MAXS bounds the plan's sources. Per-target constants are read
// through cst (the scalar cache on the device). Bound by VALU before the single-quotient form, now
// by memory and latency: ModUp conversions of 256 switches at N = 2^16 (50-bit sources) 2.92 ->
// 1.64 ms, mod_down's (60-bit sources) 2.12 -> 0.98 ms per step. (The unnamed parameter chose between two
// forms of the sums that are both gone; the replay still names it.)
template <u32 MAXS, bool = false>
CKH_DEV void conv_coeff(const ConvSrc* srcs, const ConvTgt* tgts, const PrimeConst* pcs, const ConvPlan& P,
                        const u64* in_p, u64* out_p, u32 n, u32 c, u32 t0, u32 t1, bool yform) {
    ConvY<MAXS> Y;
    conv_sources<MAXS>(srcs, P, glb(in_p), n, c, yform, Y);
    const auto outp = glb(out_p);
    const double ed = (double)(u32)Y.e;
    if constexpr (MAXS <= WRAP_SRC) {
        if (Y.small) {
            // y_j - 2^49, an absent source's as well (its constants are 0)
#pragma unroll
            for (u32 j = 0; j < MAXS; ++j) {
                Y.y[j] -= WRAP_CENTER;
                Y.yd[j] -= (double)WRAP_CENTER;
            }
            for (u32 t = t0; t < t1; ++t) {
                const auto* g = cst(tgts + P.tgt_first + t);
                const u64 o = conv_wrap_small<MAXS>(g, Y.y, Y.yd, (u32)Y.e, ed);
                st_nt(outp, (u64)g->limb * n + c, csub_sign(csub_sign(o, g->r << 1), g->r));
            }
            return;
        }
    }
    for (u32 t = t0; t < t1; ++t) {
        const auto* g = cst(tgts + P.tgt_first + t);
        u64 o;
        if (MAXS <= WRAP_SRC && g->wrap == WRAP_LARGE) {
            o = csub_sign(conv_wrap_large<MAXS>(g, Y.y, Y.yd, (u32)Y.e), g->r);
        } else if (MAXS > WRAP_SRC && g->mode != TGT_INT) {
            // f64 modular products: the source's own (TGT_FP), or its 30-bit halves
            const double r = g->rf, rinv = g->rinv;
            double acc = -g->hmod_f;
            if (g->mode == TGT_FP) {
#pragma unroll
                for (u32 j = 0; j < MAXS; ++j) {
                    acc = acc + fmulmod(Y.yd[j], g->qhat_f[j], g->qhat_q[j], r);
                    if ((j & 3) == 3) acc = freduce(acc, r, rinv);
                }
            } else {
#pragma unroll
                for (u32 j = 0; j < MAXS; ++j) {
                    const double lo = (double)(u32)(Y.y[j] & ((1u << 30) - 1)), hi = (double)(u32)(Y.y[j] >> 30);
                    acc = acc + fmulmod(lo, g->qhat_f[j], g->qhat_q[j], r);
                    acc = acc + fmulmod(hi, g->qhat30_f[j], g->qhat30_q[j], r);
                    if (j & 1) acc = freduce(acc, r, rinv);
                }
            }
            if (P.exact) acc = acc - fmulmod(ed, g->qmod_f, g->qmod_q, r);
            o = d2u(fcanon(acc, r, rinv));
        } else {
            o = conv_dot60<MAXS>(g, pc_int(pcs + g->prime), Y.y, Y.e, P.exact);
        }
        st_nt(outp, (u64)g->limb * n + c, o);
    }
}

// ---------------------------------------------------------------- matrix-core form
//
// Sum_j y_j c_jt computed as sum_p 2^(8p) sum_(j,b) y_j[b] w_p(2^(8b) c_jt mod r_t): y_j[b] are
// the bytes of y_j (offset by -128 to signed), w_p the balanced signed base-256 digits of the
// constant; one 32 x 32 x 32 int8 matrix product multiplies 32 (target, digit) rows by 32
// coefficients over 4 sources. Targets are grouped four at a time, f64-path and integer-path
// targets in separate groups.
constexpr u32 MF_MAX_GROUPS = 12;
struct MfPlan {
    u32 ngroups;  // 0: no matrix form (the vector kernel runs)
    u32 kb;       // K blocks of 32 (sources / 4, rounded up)
    u32 a_off;    // first A tile (64 lanes x 16 bytes) of the plan
    u32 t_off;    // first MfTgt of the plan (4 per group)
};
struct MfTgt {
    double rf, rinv, c32_f, c32_q, bias_f, nq_c;  // f64 path (nq_c: -Q mod r, centered)
    u64 q, nq, corr;                              // integer path (nq: -Q mod r; corr = bias_f)
    double nq_f, corr_f;                          // integer path: nq and corr as f64 (rounded)
    u32 limb;  // output limb; ~0u = padding
    u32 fp;    // 1: f64 recombination (r < 2^50)
};

// One block of the matrix-core conversion: 256 coefficients (block bx) of one job (plan P with
// matrix form F), all targets of the plan; thread tid of 256 (four waves of 64). W provides the
// wave operations: the operand types v4i (16 bytes per lane) and v16i (16 int32 per lane),
// mfma(a, b, d) (the wave's 32 x 32 x 32 int8 product: lane l holds A row l % 32 and B column
// l % 32 at k = 16 (l / 32) + byte, and receives D column l % 32, rows 8 (r / 4) + 4 (l / 32) +
// r % 4 in its element r) and shfl_xor32(v) (lane l ^ 32's value). a_lds / t_lds are the
// block's shared copies of the plan's A tiles and target constants.
// Each wave takes 2 tiles of
// 32 coefficients; lane l works on coefficient l % 32 of a tile and on sources 2h, 2h + 1,
// 4 + 2h, 5 + 2h (h = l / 32), which is exactly its B operand (k = 16 h + i: source 2h + i / 8,
// byte i % 8; second K block: sources + 4). The overflow estimate gathers the partner lane's
// products (lane l ^ 32) and sums them in source order.
template <u32 KB, class W>
CKH_DEV void conv_mf_block(const ConvSrc* srcs, const ConvPlan& P, const MfPlan& F, const typename W::v4i* a_tiles,
                           const MfTgt* tgts, const u64* in_p, u64* out_p, u32 n, u32 bx, u32 tid,
                           typename W::v4i* a_lds, MfTgt* t_lds, bool yform) {
    typedef typename W::v4i v4i;
    typedef typename W::v16i v16i;
    {
        const u32 na = F.ngroups * F.kb * 64;  // the plan's own K blocks (F.kb <= KB)
        for (u32 i = tid; i < na; i += 256) a_lds[i] = a_tiles[(u64)F.a_off * 64 + i];
        const u32 words = F.ngroups * 4 * (u32)(sizeof(MfTgt) / 8);
        const u64* src = (const u64*)(tgts + F.t_off);
        u64* dst = (u64*)t_lds;
        for (u32 i = tid; i < words; i += 256) dst[i] = src[i];
    }
    __syncthreads();
    const u32 lane = tid & 63, w = tid >> 6, h = lane >> 5, nl = lane & 31;
    const auto inp = glb(in_p);
    const auto outp = glb(out_p);
    constexpr u64 FLIP = 0x8080808080808080ull;  // byte - 128: the signed view of each byte
    // The wave's two tiles of 32 coefficients run side by side (two independent products per
    // group, one read of each target's constants for both).
    u32 c[2];
    v4i b[2][KB];
    u64 e[2] = {0, 0};
#pragma unroll
    for (u32 nt = 0; nt < 2; ++nt) {
        c[nt] = bx * 256 + w * 64 + nt * 32 + nl;
        u64 y[2 * KB];
        double pr[2 * KB];
#pragma unroll
        for (u32 q = 0; q < 2 * KB; ++q) {
            const u32 j = 4 * (q / 2) + 2 * h + (q % 2);
            y[q] = 0;
            pr[q] = 0.0;
            if (j < P.nsrc) {
                const auto* sp = cst(srcs + P.src_first + j);
                const u64 x = inp[(u64)(P.src_limb0 + j) * n + c[nt]];
                if (yform) {
                    y[q] = x;
                } else if (sp->fp) {
                    double sv = u2d(x) + (double)sp->h;
                    sv = sv >= sp->qf ? sv - sp->qf : sv;
                    double v = fmulmod(sv, sp->qhinv_f, sp->qhinv_q, sp->qf);
                    v = v < 0.0 ? v + sp->qf : v;
                    y[q] = d2u(v);
                } else {
                    y[q] = shoup(add_mod(x, sp->h, sp->q), sp->qhinv, sp->qhinv_s, sp->q);
                }
                pr[q] = u64_to_f64_rn(y[q]) * sp->inv;
            }
        }
        // e = floor(sum_j f64(y_j) / q_j) in source order j = 0, 1, ... (as the vector kernel)
        if (P.exact) {
            double other[2 * KB];
#pragma unroll
            for (u32 q = 0; q < 2 * KB; ++q) other[q] = W::shfl_xor32(pr[q]);
            double f = 0.0;
#pragma unroll
            for (u32 j = 0; j < 4 * KB; ++j) {
                if (j < P.nsrc) {
                    const u32 hj = (j / 2) % 2, q = 2 * (j / 4) + (j % 2);
                    f = f + (hj == h ? pr[q] : other[q]);
                }
            }
            e[nt] = (u64)f;
        }
#pragma unroll
        for (u32 kb = 0; kb < KB; ++kb) {
            const u64 y0 = y[2 * kb] ^ FLIP, y1 = y[2 * kb + 1] ^ FLIP;
            b[nt][kb] = v4i{(int)(u32)y0, (int)(u32)(y0 >> 32), (int)(u32)y1, (int)(u32)(y1 >> 32)};
        }
    }
    auto product = [&](u32 g, u32 nt) {
        v16i d = {};
#pragma unroll
        for (u32 kb = 0; kb < KB; ++kb)
            if (kb < F.kb)
                d = W::mfma(a_lds[(g * F.kb + kb) * 64 + lane], b[nt][kb], d);
        return d;
    };
    v16i dn0 = product(0, 0), dn1 = product(0, 1);
#pragma unroll 1
    for (u32 g = 0; g < F.ngroups; ++g) {
        const v16i d0 = dn0, d1 = dn1;
        if (g + 1 < F.ngroups) {  // the next group's products overlap this group's recombination
            dn0 = product(g + 1, 0);
            dn1 = product(g + 1, 1);
        }
#pragma unroll
        for (u32 uu = 0; uu < 2; ++uu) {
            const MfTgt& tg = t_lds[4 * g + 2 * h + uu];
            const u32 limb = tg.limb;
            if (limb == ~0u) continue;
            const bool fp = tg.fp;
            const double r = tg.rf, rinv = tg.rinv, c32_f = tg.c32_f, c32_q = tg.c32_q, bias_f = tg.bias_f;
            const double nq_c = tg.nq_c;
#pragma unroll
            for (u32 nt = 0; nt < 2; ++nt) {
                const v16i& d = nt ? d1 : d0;
                // X = lo + hi 2^32, lo / hi = sum of four digit planes each (|.| < 2^45, exact);
                // planes p and p + 1 combine in int32 first (|d| < 2^20: |d_p + 256 d_(p+1)| < 2^29)
                const int l01 = d[8 * uu + 0] + d[8 * uu + 1] * 256, l23 = d[8 * uu + 2] + d[8 * uu + 3] * 256;
                const int h01 = d[8 * uu + 4] + d[8 * uu + 5] * 256, h23 = d[8 * uu + 6] + d[8 * uu + 7] * 256;
                const double lo = __builtin_fma((double)l23, 65536.0, (double)l01);
                const double hi = __builtin_fma((double)h23, 65536.0, (double)h01);
                u64 o;
                if (fp) {
                    // e < 8: e nq_c is exact and the sum stays an integer below 2^53
                    double acc = lo + fmulmod(hi, c32_f, c32_q, r) + bias_f;
                    acc = __builtin_fma((double)e[nt], nq_c, acc);
                    o = d2u(fcanon(acc, r, rinv));
                } else {
                    // V = X + A with X = lo + hi 2^32 (|lo|, |hi| < 2^45) and A = e nq + corr
                    // (below 2^64). k = rint(V / r) from f64 estimates: their error (below 2^27 on
                    // |V| < 2^79, then the reciprocal's) moves V / r by less than 2^-30, so
                    // |V - k r| < r; V - k r is then computed exactly in wrapping 64-bit arithmetic
                    // and one addition of r makes it non-negative.
                    const double T = __builtin_fma(hi, 4294967296.0, lo) +
                                     __builtin_fma((double)e[nt], tg.nq_f, tg.corr_f);
                    const int64_t k = (int64_t)__builtin_rint(T * rinv);
                    const u64 lo64 = (u64)((int64_t)l01 + (int64_t)l23 * 65536);
                    const u64 hi64 = (u64)((int64_t)h01 + (int64_t)h23 * 65536);
                    const u32 ee = (u32)e[nt];
                    const u64 A = (u64)ee * (u32)tg.nq + (((u64)ee * (u32)(tg.nq >> 32)) << 32) + tg.corr;
                    const u64 R = lo64 + (hi64 << 32) + A - (u64)k * tg.q;
                    o = (int64_t)R < 0 ? R + tg.q : R;
                }
                outp[(u64)limb * n + c[nt]] = o;
            }
        }
    }
}

}  // namespace ckh
