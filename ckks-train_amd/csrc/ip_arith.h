// The key inner product per coefficient (the body of k_inner_product) and the NTT-form Galois
// index, written so that a host program can include them too (the CPU replay in tests/emu). The
// includer has included arith.h and defines glb(p) and brev32(x) (32-bit bit reversal).
#pragma once

#include "arith.h"

namespace ckh {

// One limb of a key-switch inner product: digit j's limb at dig + j * dig_stride (or own for
// digit own_j when own is set), read through the Galois permutation when galois != 0; key part
// j's b limb at key + 2 j key_poly, its a limb key_poly further; acc_b / acc_a receive the sums.
struct IpJob {
    const u64* dig;
    u64 dig_stride;
    const u64* key;
    u64 key_poly;
    u64* acc_b;
    u64* acc_a;
    u64 galois;
    const u64* own;
    u32 ndig, prime, own_j, pad;
};

// NTT-form Galois permutation: sigma_g(a)[i] = a[perm(i)],
// perm(i) = bitrev(((g * (2 bitrev(i) + 1)) mod 2N - 1) / 2)
// (crates/ckks-train-core/src/rns.rs:5-17,147-157), computed inline instead of read from a table.
CKH_DEV u32 galois_index(u32 i, u64 g, u32 log_n) {
    const u32 rev = (brev32(i) >> (32 - log_n)) * 2 + 1;
    const u32 raw = (u32)(((g * rev) >> 1) & ((1u << log_n) - 1));
    return brev32(raw) >> (32 - log_n);
}

// acc_b = sum_j d_j * b_j and acc_a = sum_j d_j * a_j per limb of Q_l * P
// (crates/ckks-train-ckks/src/keyswitch.rs:254-303; residues are unique, so any exact summation
// order gives the reference's words). Primes below 2^50 sum f64 modular products (reduced every
// four digits); larger primes sum exact 128-bit products and reduce once. Digit limbs may be read
// through the Galois permutation (hoisted rotations, evaluator.rs:596-604).
// Digits are taken IP_GROUP at a time, every word of a group loaded before any product, so the
// loads of a group are in flight together.
constexpr u32 IP_GROUP = 4;

// How ip_words reads and writes W consecutive words from word W c of a limb: one at a time here; the
// kernel's own takes two in one 16-byte access.
struct IpWord {
    static constexpr u32 W = 1;
    CKH_DEV static void load(const u64* p, u64 c, u64 (&w)[1]) { w[0] = glb(p)[c]; }
    CKH_DEV static void load_key(const u64* p, u64 c, u64 (&w)[1]) { w[0] = glb(p)[c]; }
    CKH_DEV static void store(u64* p, u64 c, const u64 (&w)[1]) { glb(p)[c] = w[0]; }
    // the words of a digit read through the Galois permutation
    CKH_DEV static void gather(const u64* p, u64 c, u64 g, u32 log_n, u64 (&w)[1]) {
        w[0] = glb(p)[galois_index((u32)c, g, log_n)];
    }
};

template <class Mem>
CKH_DEV void ip_words(const IpJob& J, const PrimeConst& C, u32 log_n, u32 c) {
    constexpr u32 W = Mem::W;
    u64 dv[IP_GROUP][W], bv[IP_GROUP][W], av[IP_GROUP][W];
    auto load_group = [&](u32 j0) {
#pragma unroll
        for (u32 u = 0; u < IP_GROUP; ++u) {
            const u32 j = j0 + u;
            if (j < J.ndig) {
                const u64* d = (J.own && j == J.own_j) ? J.own : J.dig + j * J.dig_stride;
                if (J.galois)
                    Mem::gather(d, c, J.galois, log_n, dv[u]);
                else
                    Mem::load(d, c, dv[u]);
                Mem::load_key(J.key + (2 * j) * J.key_poly, c, bv[u]);
                Mem::load_key(J.key + (2 * j + 1) * J.key_poly, c, av[u]);
            }
        }
    };
    u64 ob[W], oa[W];
    if (C.q < FP_PRIME_BOUND) {
        const double q = C.qf, qinv = C.qinv;
        double sb[W], sa[W];
#pragma unroll
        for (u32 w = 0; w < W; ++w) sb[w] = sa[w] = 0.0;
        for (u32 j0 = 0; j0 < J.ndig; j0 += IP_GROUP) {
            load_group(j0);
#pragma unroll
            for (u32 u = 0; u < IP_GROUP; ++u) {
                if (j0 + u < J.ndig) {
#pragma unroll
                    for (u32 w = 0; w < W; ++w) {
                        const double d = u2d(dv[u][w]), b = u2d(bv[u][w]), a = u2d(av[u][w]);
                        sb[w] += fmulmod(d, b, b * qinv, q);
                        sa[w] += fmulmod(d, a, a * qinv, q);
                    }
                }
            }
            // four products (|.| < 0.7 q each) since the last reduction
#pragma unroll
            for (u32 w = 0; w < W; ++w) {
                sb[w] = freduce(sb[w], q, qinv);
                sa[w] = freduce(sa[w], q, qinv);
            }
        }
#pragma unroll
        for (u32 w = 0; w < W; ++w) {
            ob[w] = d2u(fcanon(sb[w], q, qinv));
            oa[w] = d2u(fcanon(sa[w], q, qinv));
        }
    } else {
        Dot60 sb[W], sa[W];
        for (u32 j0 = 0; j0 < J.ndig; j0 += IP_GROUP) {
            load_group(j0);
#pragma unroll
            for (u32 u = 0; u < IP_GROUP; ++u) {
                if (j0 + u < J.ndig) {
#pragma unroll
                    for (u32 w = 0; w < W; ++w) {
                        sb[w].add(dv[u][w], bv[u][w]);
                        sa[w].add(dv[u][w], av[u][w]);
                    }
                }
            }
        }
#pragma unroll
        for (u32 w = 0; w < W; ++w) {
            u64 hi, lo;
            sb[w].get(hi, lo);
            ob[w] = reduce128(hi, lo, C);
            sa[w].get(hi, lo);
            oa[w] = reduce128(hi, lo, C);
        }
    }
    Mem::store(J.acc_b, c, ob);
    Mem::store(J.acc_a, c, oa);
}

CKH_DEV void ip_coeff(const IpJob& J, const PrimeConst& C, u32 log_n, u32 c) { ip_words<IpWord>(J, C, log_n, c); }

}  // namespace ckh
