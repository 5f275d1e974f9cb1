// The passes of ntt_passes.h with 4 words per thread, for launches that would leave compute units
// idle: a tile of 1024 words on 256 threads, in rounds of two stages with an LDS exchange between
// rounds. Same sub-transforms, arithmetic and intermediates as the 16-word passes, so either may
// follow the other. Written so that a host program can include it too (the CPU replay in tests/emu);
// the includer has included ntt_passes.h, conv_cols.h and ip_arith.h.
//
// A small launch is bound by the chain of one wave: with 16 words a wave issues some 1300 instructions,
// 840 of them f64, alone on its SIMD (2.4 us of a pass's 5.5); with 4 words a quarter of that, on four
// times as many compute units, for one or two exchanges more. All twiddles (at most 12 a thread) come
// straight from the tables and are loaded with the words, before any arithmetic. A pass over a few limbs:
// 5.5 -> 3.1 us; one switch at N = 2^12 61.7 -> 37.2 us, a product with relinearization and rescale at
// 2^14 125 -> 67 us. (A whole limb per workgroup, both passes in one launch, was slower at 2^13: 15 us
// against two launches of 5.5, one compute unit's arithmetic.) In larger launches the narrow row passes
// still win by their occupancy (7 waves per SIMD) until the traffic is what bounds them.
#pragma once

#include "conv_cols.h"
#include "ip_arith.h"
#include "narrow_jobs.h"
#include "ntt_passes.h"

namespace ckh {
namespace fast {

constexpr u32 LW = 2, NW = 1u << LW;             // words per thread
constexpr u32 NTL = 8 + LW, NTILE = 1u << NTL;   // words per tile
constexpr u32 NLDS = NTILE + NTILE / 16;
// A column tile of 2^8 rows takes twice the threads: 8 columns are a whole 64-byte sector. Against 4
// columns a switch of 13 limbs at N = 2^15 takes 73 against 80 us, of 12 limbs at 2^16 97 against 107;
// 16 columns on 1024 threads: 74 and 92, but 47 against 41 us for one limb at 2^15.
template <u32 M>
constexpr u32 NCL = M == 8 ? NTL + 1 : NTL;  // log2 of a column tile's words
template <u32 M>
constexpr u32 NCT = 1u << (NCL<M> - LW);  // its threads
template <u32 M>
constexpr u32 NCLDS = (1u << NCL<M>) + (1u << NCL<M>) / 16;

// The sub-transform of 2^M words: 2^(M - LW) threads o hold NW words each; in the layout of shift p
// thread o's word k has index sub(o, k, p) (bits p .. p + LW - 1 vary over k).
CKH_DEV constexpr u32 sub(u32 o, u32 k, u32 p) { return ((o >> p) << (p + LW)) | (k << p) | (o & ((1u << p) - 1)); }
template <u32 M>
constexpr u32 ROUNDS = (M + LW - 1) / LW;
template <u32 M>
CKH_DEV constexpr u32 fwd_shift(u32 r) {
    return M > LW * (r + 1) ? M - LW * (r + 1) : 0;
}
template <u32 M>
CKH_DEV constexpr u32 inv_shift(u32 r) {
    return LW * r < M - LW ? LW * r : M - LW;
}

// A thread's twiddles: w[r][i][m], stage i of round r, word pairs k with k >> (bit + 1) = m.
template <u32 M, class Ar>
struct NarrowTw {
    typename Ar::W w[ROUNDS<M>][LW][NW / 2];
};
// tab: the table from the sub-transform's first entry of each stage: entry(s, j), j < 2^s.
template <u32 M, class Ar, class Entry>
CKH_DEV void narrow_fwd_tw(NarrowTw<M, Ar>& t, u32 o, Entry entry) {
#pragma unroll
    for (u32 r = 0; r < ROUNDS<M>; ++r) {
        const u32 p = fwd_shift<M>(r);
#pragma unroll
        for (u32 i = 0; i < LW; ++i) {
            const u32 s = LW * r + i;
            if (s >= M) continue;
            const u32 b = M - 1 - s - p;
#pragma unroll
            for (u32 m = 0; m < (NW / 2) >> b; ++m) t.w[r][i][m] = entry(s, sub(o, m << (b + 1), p) >> (M - s));
        }
    }
}
template <u32 M, class Ar, class Entry>
CKH_DEV void narrow_inv_tw(NarrowTw<M, Ar>& t, u32 o, bool last, Entry entry) {
#pragma unroll
    for (u32 r = 0; r < ROUNDS<M>; ++r) {
        const u32 p = inv_shift<M>(r);
#pragma unroll
        for (u32 i = 0; i < LW; ++i) {
            const u32 u = LW * r + i;
            if (u >= M || (last && u + 1 == M)) continue;
            const u32 b = u - p;
#pragma unroll
            for (u32 m = 0; m < (NW / 2) >> b; ++m) t.w[r][i][m] = entry(M - 1 - u, sub(o, m << (b + 1), p) >> (u + 1));
        }
    }
}

// The forward stages of one sub-transform: v enters in the layout of shift M - LW, leaves in that of
// shift 0. slot(i): the LDS slot of index i; each exchange writes the slots the thread read before it.
template <u32 M, class Ar, class Lds, class Slot, class Sync>
CKH_DEV void narrow_fwd(const Ar& ar, const NarrowTw<M, Ar>& t, typename Ar::V (&v)[NW], Lds lds, u32 o, Slot slot, Sync sync) {
#pragma unroll
    for (u32 r = 0; r < ROUNDS<M>; ++r) {
        const u32 p = fwd_shift<M>(r);
        if (r) {
            sync();
#pragma unroll
            for (u32 k = 0; k < NW; ++k) v[k] = ar.from_mid(lds[slot(sub(o, k, p))]);
        }
#pragma unroll
        for (u32 i = 0; i < LW; ++i) {
            const u32 s = LW * r + i;
            if (s >= M) continue;
            const u32 b = M - 1 - s - p;
#pragma unroll
            for (u32 k = 0; k < NW; ++k) {
                if (k & (1u << b)) continue;
                ct_stage<Ar, M>(ar, s, v[k], v[k + (1u << b)], t.w[r][i][k >> (b + 1)]);
            }
        }
        if (r + 1 < ROUNDS<M>) {
#pragma unroll
            for (u32 k = 0; k < NW; ++k) lds[slot(sub(o, k, p))] = ar.to_mid(v[k]);
        }
    }
}

// The inverse stages: v enters in the layout of shift 0, leaves in that of shift M - LW. LAST: the last
// stage is the transform's (gs_final, with ar.add when ADD).
template <u32 M, bool LAST, bool ADD, class Ar, class Lds, class Slot, class Sync>
CKH_DEV void narrow_inv(const Ar& ar, const NarrowTw<M, Ar>& t, typename Ar::V (&v)[NW], Lds lds, u32 o, Slot slot, Sync sync) {
#pragma unroll
    for (u32 r = 0; r < ROUNDS<M>; ++r) {
        const u32 p = inv_shift<M>(r);
        if (r) {
            sync();
#pragma unroll
            for (u32 k = 0; k < NW; ++k) v[k] = ar.from_mid(lds[slot(sub(o, k, p))]);
        }
#pragma unroll
        for (u32 i = 0; i < LW; ++i) {
            const u32 u = LW * r + i;
            if (u >= M) continue;
            const u32 b = u - p;
#pragma unroll
            for (u32 k = 0; k < NW; ++k) {
                if (k & (1u << b)) continue;
                if (LAST && u + 1 == M)
                    ar.template gs_final<ADD>(v[k], v[k + (1u << b)]);
                else
                    ar.gs(v[k], v[k + (1u << b)], t.w[r][i][k >> (b + 1)]);
            }
        }
        if (r + 1 < ROUNDS<M>) {
#pragma unroll
            for (u32 k = 0; k < NW; ++k) lds[slot(sub(o, k, p))] = ar.to_mid(v[k]);
        }
    }
}

// The place of a thread in a column tile (2^M rows of TC columns) or a row tile (rows of 2^M words).
template <u32 M>
struct NarrowCol {
    static constexpr u32 TCL = NCL<M> - M;
    u32 B, c, o;  // words per row (log2), the thread's column, its part of it
    CKH_DEV NarrowCol(u32 log_n, u32 tile, u32 tid)
        : B(log_n - M), c((tile << TCL) + (tid & ((1u << TCL) - 1))), o(tid >> TCL) {}
    CKH_DEV u64 word(u32 r) const { return ((u64)r << B) + c; }
    CKH_DEV u32 slot(u32 r) const { return pad((r << TCL) + (c & ((1u << TCL) - 1))); }
};
template <u32 M>
struct NarrowRow {
    u32 rr, o, row;  // the row in the tile, the thread's part of it, the row in the limb
    CKH_DEV NarrowRow(u32 tile, u32 tid)
        : rr(tid >> (M - LW)), o(tid & ((1u << (M - LW)) - 1)), row((tile << (NTL - M)) + rr) {}
    CKH_DEV u32 word(u32 c) const { return (row << M) + c; }
    CKH_DEV u32 slot(u32 c) const { return pad((rr << M) + c); }
};
struct BlockSync {
    CKH_DEV void operator()() const { __syncthreads(); }
};
struct WaveSync {  // a row of at most 256 words belongs to at most 64 adjacent threads
    CKH_DEV void operator()() const { CKH_WAVE_SYNC(); }
};

template <class Ar>
struct ColEntry {
    const Ar& ar;
    CKH_DEV auto operator()(u32 s, u32 j) const { return ar.tw((1u << s) + j); }
};
template <class Ar>
struct RowEntry {
    const Ar& ar;
    u32 A, row;
    CKH_DEV auto operator()(u32 s, u32 j) const { return ar.tw((1u << (A + s)) + (row << s) + j); }
};

// ---------------------------------------------------------------- passes

// fill(v): the tile's words in the layout of shift M - LW (row sub(o, k, M - LW), column P.c).
template <u32 M, class Ar, class Lds, class Fill>
CKH_DEV void narrow_fwd_cols(const Ar& ar, const NarrowCol<M>& P, u64* out_p, Lds lds, Fill fill) {
    NarrowTw<M, Ar> t;
    narrow_fwd_tw<M>(t, P.o, ColEntry<Ar>{ar});
    typename Ar::V v[NW];
    fill(v);
    narrow_fwd<M>(ar, t, v, lds, P.o, [&](u32 r) { return P.slot(r); }, BlockSync{});
    const auto out = glb(out_p);
#pragma unroll
    for (u32 k = 0; k < NW; ++k) out[P.word(sub(P.o, k, 0))] = ar.to_mid(v[k]);
}

// The words of a row pass, in the layout of shift 0 (NW consecutive words from P.word(NW o)), not canonical.
template <u32 M, class Ar, class Lds, class Pre>
CKH_DEV void narrow_fwd_rows(const Ar& ar, const NarrowRow<M>& P, const u64* in_p, Lds lds, u32 log_n,
                             typename Ar::V (&v)[NW], Pre pre) {
    NarrowTw<M, Ar> t;
    const auto in = glb(in_p);
    u64 x[NW];
#pragma unroll
    for (u32 k = 0; k < NW; ++k) x[k] = in[P.word(sub(P.o, k, M - LW))];
    narrow_fwd_tw<M>(t, P.o, RowEntry<Ar>{ar, log_n - M, P.row});
    pre();
#pragma unroll
    for (u32 k = 0; k < NW; ++k) v[k] = ar.from_mid(x[k]);
    narrow_fwd<M>(ar, t, v, lds, P.o, [&](u32 c) { return P.slot(c); }, WaveSync{});
}

template <u32 M, class Ar, class Lds>
CKH_DEV void narrow_fwd_rows_store(const Ar& ar, u64* io_p, Lds lds, u32 log_n, u32 tile, u32 tid) {
    const NarrowRow<M> P(tile, tid);
    typename Ar::V v[NW];
    narrow_fwd_rows<M>(ar, P, io_p, lds, log_n, v, NoPre{});
    const auto out = glb(io_p);
#pragma unroll
    for (u32 k = 0; k < NW; ++k) out[P.word(NW * P.o + k)] = ar.fwd_final(v[k]);
}

// fill(v): NW consecutive words per thread (the layout of shift 0), canonical.
template <u32 M, class Ar, class Lds, class Fill>
CKH_DEV void narrow_inv_rows(const Ar& ar, const NarrowRow<M>& P, u64* out_p, Lds lds, u32 log_n, Fill fill) {
    NarrowTw<M, Ar> t;
    narrow_inv_tw<M>(t, P.o, false, RowEntry<Ar>{ar, log_n - M, P.row});
    typename Ar::V v[NW];
    fill(v);
    narrow_inv<M, false, false>(ar, t, v, lds, P.o, [&](u32 c) { return P.slot(c); }, WaveSync{});
    const auto out = glb(out_p);
#pragma unroll
    for (u32 k = 0; k < NW; ++k) out[P.word(sub(P.o, k, M - LW))] = ar.to_mid(v[k]);
}

template <u32 M, bool ADD, class Ar, class Lds>
CKH_DEV void narrow_inv_cols(const Ar& ar, u64* io_p, Lds lds, u32 log_n, u32 tile, u32 tid) {
    const NarrowCol<M> P(log_n, tile, tid);
    const auto io = glb(io_p);
    NarrowTw<M, Ar> t;
    u64 x[NW];
#pragma unroll
    for (u32 k = 0; k < NW; ++k) x[k] = io[P.word(sub(P.o, k, 0))];
    narrow_inv_tw<M>(t, P.o, true, ColEntry<Ar>{ar});
    typename Ar::V v[NW];
#pragma unroll
    for (u32 k = 0; k < NW; ++k) v[k] = ar.from_mid(x[k]);
    narrow_inv<M, true, ADD>(ar, t, v, lds, P.o, [&](u32 r) { return P.slot(r); }, BlockSync{});
#pragma unroll
    for (u32 k = 0; k < NW; ++k) io[P.word(sub(P.o, k, M - LW))] = ar.canon_out(v[k]);
}

// ---------------------------------------------------------------- inner product

// Digits of an inner product loaded before their products. Four keep 160-194 registers (2-3 waves per
// SIMD); two take 114-132 and a switch of 24 limbs at N = 2^16 171 against 177 us, but where the rows have 2^6
// words a launch is small and waits for one group more: 32.7 against 32.2 us at 2^12.
template <u32 M>
constexpr u32 NARROW_IP_GROUP = M == 6 ? 4 : 2;

// Words i0 .. i0 + NW - 1 of one part of an inner product. f64 primes: signed sums, |.| <= q / 2; integer
// primes: canonical words. A group's digits and keys are loaded before its products.
template <u32 G, class Ar>
CKH_DEV void limb_ip(const Ar& ar, const LimbIp& J, u32 part, const PrimeConst* pc, u32 log_n, u32 i0, typename Ar::V (&out)[NW]) {
    u32 di[NW];
#pragma unroll
    for (u32 k = 0; k < NW; ++k) di[k] = J.galois ? galois_index(i0 + k, J.galois, log_n) : i0 + k;
    [[maybe_unused]] double s[NW];
    [[maybe_unused]] Dot60 d[NW];
#pragma unroll
    for (u32 k = 0; k < NW; ++k) s[k] = 0.0;
    for (u32 j0 = 0; j0 < J.ndig; j0 += G) {
        u64 dv[G][NW], kv[G][NW];
#pragma unroll
        for (u32 u = 0; u < G; ++u) {
            const u32 j = j0 + u;
            if (j < J.ndig) {
                const auto dig = glb((J.own && j == J.own_j) ? J.own : J.dig + j * J.dig_stride);
                const auto key = glb(J.key + (2 * j + part) * J.key_poly);
#pragma unroll
                for (u32 k = 0; k < NW; ++k) {
                    dv[u][k] = dig[di[k]];
                    kv[u][k] = key[i0 + k];
                }
            }
        }
#pragma unroll
        for (u32 u = 0; u < G; ++u) {
            if (j0 + u < J.ndig) {
#pragma unroll
                for (u32 k = 0; k < NW; ++k) {
                    if constexpr (Ar::F64) {
                        const double b = u2d(kv[u][k]);
                        s[k] += fmulmod(u2d(dv[u][k]), b, b * ar.qinv, ar.q);
                    } else {
                        d[k].add(dv[u][k], kv[u][k]);
                    }
                }
            }
        }
        // at most four products (|.| < 0.7 q each) since the last reduction
        if constexpr (Ar::F64) {
#pragma unroll
            for (u32 k = 0; k < NW; ++k) s[k] = freduce(s[k], ar.q, ar.qinv);
        }
    }
#pragma unroll
    for (u32 k = 0; k < NW; ++k) {
        if constexpr (Ar::F64) {
            out[k] = s[k];
        } else {
            u64 hi, lo;
            d[k].get(hi, lo);
            out[k] = reduce128(hi, lo, pc_int(pc));
        }
    }
}

// One part of an inner product and its inverse row pass.
template <u32 M, class Ar, class Lds>
CKH_DEV void narrow_ip_inv_rows(const Ar& ar, const IpInvJob& J, u32 part, const PrimeConst* pc, Lds lds, u32 log_n,
                                u32 tile, u32 tid) {
    const NarrowRow<M> P(tile, tid);
    narrow_inv_rows<M>(ar, P, J.out + part * J.out_part, lds, log_n,
                       [&](typename Ar::V(&v)[NW]) { limb_ip<NARROW_IP_GROUP<M>>(ar, J.ip, part, pc, log_n, P.word(NW * P.o), v); });
}

// (a - t) inv (+ add) of NW consecutive words: t the row pass's words (f64: |.| <= 2.6 q), a the first
// operand (f64: below q in magnitude; else canonical).
template <class Ar>
CKH_DEV void narrow_finish(const Ar& ar, const typename Ar::V (&a)[NW], const typename Ar::V (&t)[NW], bool has_add, const u64 (&add)[NW], u64* out_p,
                           u64 inv, u64 inv_s, const FTw& inv_f, u64 q, u32 i0) {
    const auto out = glb(out_p);
#pragma unroll
    for (u32 k = 0; k < NW; ++k) {
        if constexpr (Ar::F64) {
            double v = fmulmod(a[k] - t[k], inv_f.w, inv_f.wq, ar.q);
            if (has_add) v = v + u2d(add[k]);
            out[i0 + k] = d2u(fcanon(v, ar.q, ar.qinv));
        } else {
            u64 v = shoup(sub_mod(a[k], ar.fwd_final(t[k]), q), inv, inv_s, q);
            if (has_add) v = add_mod(v, add[k], q);
            out[i0 + k] = v;
        }
    }
}

// NW consecutive words of an optional addend, read through a Galois permutation when g != 0.
CKH_DEV void load_addend(const u64* p, u32 g, u32 i0, u32 log_n, u64 (&add)[NW]) {
    if (!p) return;
#pragma unroll
    for (u32 k = 0; k < NW; ++k) add[k] = glb(p)[g ? galois_index(i0 + k, g, log_n) : i0 + k];
}

// The row pass, the inner product of one part and the finish.
template <u32 M, class Ar, class Lds>
CKH_DEV void narrow_ip_fin(const Ar& ar, const IpFinJob& J, u32 part, const PrimeConst* pc, u64 q, Lds lds, u32 log_n,
                           u32 tile, u32 tid) {
    const NarrowRow<M> P(tile, tid);
    const u32 i0 = P.word(NW * P.o);
    typename Ar::V v[NW], a[NW];
    const u64* add_p = part ? J.add_a : J.add_b;
    u64 add[NW] = {};
    narrow_fwd_rows<M>(ar, P, J.t + part * J.t_part, lds, log_n, v, [&] {
        load_addend(add_p, part ? 0 : J.add_galois, i0, log_n, add);
        limb_ip<NARROW_IP_GROUP<M>>(ar, J.ip, part, pc, log_n, i0, a);
    });
    narrow_finish(ar, a, v, add_p != nullptr, add, part ? J.out_a : J.out_b, J.inv, J.inv_s, J.inv_f, q, i0);
}

// The row pass and finish of rescale / mod_down with the first operand in memory.
template <u32 M, class Ar, class Lds>
CKH_DEV void narrow_fin(const Ar& ar, const u64* in_p, const FinishJob* fin, u64 q, Lds lds, u32 log_n, u32 tile, u32 tid) {
    const NarrowRow<M> P(tile, tid);
    const u32 i0 = P.word(NW * P.o);
    typename Ar::V v[NW], a[NW];
    u64 add[NW] = {};
    narrow_fwd_rows<M>(ar, P, in_p, lds, log_n, v, [&] {
        load_addend(fin->add, fin->add_galois, i0, log_n, add);
#pragma unroll
        for (u32 k = 0; k < NW; ++k) a[k] = ar.from_canon(glb(fin->a)[i0 + k]);
    });
    narrow_finish(ar, a, v, fin->add != nullptr, add, fin->out, fin->inv, fin->inv_s, fin->inv_f, q, i0);
}

}  // namespace fast
}  // namespace ckh
