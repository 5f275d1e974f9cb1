// The narrow passes (narrow_passes.h) as kernels over batches of limbs, for launches of few tiles.
#include <type_traits>

#include "basis.h"
#include "common.h"
#include "ntt.h"
#include "narrow_passes.h"

namespace ckh {
namespace fast {

// Runs body(ar) with the arithmetic of a prime; tw / twf: the direction's tables.
template <class F>
CKH_DEV void with_prime(const PrimeConst* pcs, const Tw* tw, const FTw* twf, u32 prime, u32 log_n, F body) {
    const PrimeConst* pc = pcs + prime;
    const u64 toff = (u64)prime << log_n;
    if (pc->q < FP_PRIME_BOUND)
        body(FpAr{twf + toff, pc->qf, pc->qinv, pc->n_inv_f, pc->w_n_inv_f, nullptr});
    else
        body(IntAr{tw + toff, pc->q, pc->n_inv, pc->n_inv_s, pc->w_n_inv, pc->w_n_inv_s});
}
// The last inverse stage's constants replaced by those of a conversion source's y form.
CKH_DEV void set_yform(FpAr& ar, const YForm* yf) {
    const auto* y = cst(yf);
    ar.ninv = FTw{y->n_f.w, y->n_f.wq};
    ar.wninv = FTw{y->wn_f.w, y->wn_f.wq};
    ar.add = y->h_f;
}
CKH_DEV void set_yform(IntAr& ar, const YForm* yf) {
    const auto* y = cst(yf);
    ar.n_inv = y->n;
    ar.n_inv_s = y->n_s;
    ar.w_n_inv = y->wn;
    ar.w_n_inv_s = y->wn_s;
    ar.add = y->h;
}

template <u32 M>
__global__ __launch_bounds__(NCT<M>) void k_narrow_fwd_cols(NttTables T, const LimbRef* __restrict__ refs) {
    __shared__ u64 lds[NCLDS<M>];
    const u32 log_n = T.log_n, tile = blockIdx.x & ((1u << (log_n - NCL<M>)) - 1);
    const LimbRef ref = refs[blockIdx.x >> (log_n - NCL<M>)];
    const NarrowCol<M> P(log_n, tile, threadIdx.x);
    with_prime(T.pc, T.fwd, T.fwd_f, ref.prime, log_n, [&](const auto& ar) {
        const auto in = glb(ref.src);
        narrow_fwd_cols<M>(ar, P, ref.dst, (u64*)lds, [&](auto& v) {
#pragma unroll
            for (u32 k = 0; k < NW; ++k) v[k] = ar.from_canon(in[P.word(sub(P.o, k, M - LW))]);
        });
    });
}

// Items and their order as in k_conv_cols, over this tile's size.
template <u32 M, u32 MAXS>
__global__ __launch_bounds__(NCT<M>) void k_narrow_conv_cols(ConvTables C, NttTables T, const ConvColRef* __restrict__ refs,
                                                         u32 items) {
    __shared__ u64 lds[NCLDS<M>];
    const u32 log_n = T.log_n, item = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (item >= items) return;
    const ConvColRef R = refs[item >> (log_n - NCL<M>)];
    u32 tile;
    const u32 t = conv_col_item(R, item, 1u << (log_n - NCL<M>), tile);
    const auto* g = cst(C.tgt + R.tgt_first + t);
    const u32 prime = g->prime;
    const NarrowCol<M> P(log_n, tile, threadIdx.x);
    with_prime(T.pc, T.fwd, T.fwd_f, prime, log_n, [&](const auto& ar) {
        narrow_fwd_cols<M>(ar, P, R.out + ((u64)g->limb << log_n), (u64*)lds, [&](auto& v) {
            conv_words<NW, MAXS>(ar, C.src, R, g, T.pc + prime, log_n, (u32)P.word(P.o), M - LW + P.B, v);
        });
    });
}

template <u32 M, bool FIN>
__global__ __launch_bounds__(NT) void k_narrow_fwd_rows(NttTables T, const LimbRef* __restrict__ refs,
                                                        const FinishJob* __restrict__ fins) {
    __shared__ u64 lds[NLDS];
    const u32 log_n = T.log_n, tile = blockIdx.x & ((1u << (log_n - NTL)) - 1), r = blockIdx.x >> (log_n - NTL);
    const LimbRef ref = refs[r];
    with_prime(T.pc, T.fwd, T.fwd_f, ref.prime, log_n, [&](const auto& ar) {
        if constexpr (FIN)
            narrow_fin<M>(ar, ref.dst, fins + r, T.pc[ref.prime].q, (u64*)lds, log_n, tile, threadIdx.x);
        else
            narrow_fwd_rows_store<M>(ar, ref.dst, (u64*)lds, log_n, tile, threadIdx.x);
    });
}

template <u32 M>
__global__ __launch_bounds__(NT) void k_narrow_inv_rows(NttTables T, const LimbRef* __restrict__ refs) {
    __shared__ u64 lds[NLDS];
    const u32 log_n = T.log_n, tile = blockIdx.x & ((1u << (log_n - NTL)) - 1);
    const LimbRef ref = refs[blockIdx.x >> (log_n - NTL)];
    const NarrowRow<M> P(tile, threadIdx.x);
    with_prime(T.pc, T.inv, T.inv_f, ref.prime, log_n, [&](const auto& ar) {
        const auto in = glb(ref.src);
        narrow_inv_rows<M>(ar, P, ref.dst, (u64*)lds, log_n, [&](auto& v) {
#pragma unroll
            for (u32 k = 0; k < NW; ++k) v[k] = ar.from_canon(in[P.word(NW * P.o + k)]);
        });
    });
}

template <u32 M, bool YF>
__global__ __launch_bounds__(NCT<M>) void k_narrow_inv_cols(NttTables T, const LimbRef* __restrict__ refs,
                                                        const YForm* __restrict__ yf) {
    __shared__ u64 lds[NCLDS<M>];
    const u32 log_n = T.log_n, tile = blockIdx.x & ((1u << (log_n - NCL<M>)) - 1);
    const LimbRef ref = refs[blockIdx.x >> (log_n - NCL<M>)];
    with_prime(T.pc, T.inv, T.inv_f, ref.prime, log_n, [&](auto ar) {
        if constexpr (YF) set_yform(ar, yf + ref.aux);
        narrow_inv_cols<M, YF>(ar, ref.dst, (u64*)lds, log_n, tile, threadIdx.x);
    });
}

// Block -> (job, tile, part): the two parts of a tile share its digits.
template <u32 M>
__global__ __launch_bounds__(NT) void k_narrow_ip_inv_rows(NttTables T, const IpInvJob* __restrict__ jobs) {
    __shared__ u64 lds[NLDS];
    const u32 log_n = T.log_n, tiles = 1u << (log_n - NTL), part = (blockIdx.x >> (log_n - NTL)) & 1;
    const IpInvJob J = jobs[blockIdx.x >> (log_n - NTL + 1)];
    with_prime(T.pc, T.inv, T.inv_f, J.prime, log_n, [&](const auto& ar) {
        narrow_ip_inv_rows<M>(ar, J, part, T.pc + J.prime, (u64*)lds, log_n, blockIdx.x & (tiles - 1), threadIdx.x);
    });
}

template <u32 M>
__global__ __launch_bounds__(NT) void k_narrow_ip_fin(NttTables T, const IpFinJob* __restrict__ jobs) {
    __shared__ u64 lds[NLDS];
    const u32 log_n = T.log_n, tiles = 1u << (log_n - NTL), part = (blockIdx.x >> (log_n - NTL)) & 1;
    const IpFinJob J = jobs[blockIdx.x >> (log_n - NTL + 1)];
    with_prime(T.pc, T.fwd, T.fwd_f, J.prime, log_n, [&](const auto& ar) {
        narrow_ip_fin<M>(ar, J, part, T.pc + J.prime, T.pc[J.prime].q, (u64*)lds, log_n, blockIdx.x & (tiles - 1),
                         threadIdx.x);
    });
}

}  // namespace fast

// f with the number of stages of a row or column pass as a compile-time constant.
template <class F>
static void with_stages(u32 m, F f) {
    if (m == 6)
        f(std::integral_constant<u32, 6>{});
    else if (m == 7)
        f(std::integral_constant<u32, 7>{});
    else
        f(std::integral_constant<u32, 8>{});
}
// Row passes: KERNEL over the tiles of `limbs` limbs.
#define CKH_NARROW_ROWS(LIMBS, KERNEL, ...)                                                              \
    with_stages(t.log_n / 2, [&](auto m) {                                                               \
        constexpr u32 M = m.value;                                                                       \
        hipLaunchKernelGGL((KERNEL), dim3((LIMBS) << (t.log_n - fast::NTL)), dim3(fast::NT), 0, s, __VA_ARGS__); \
    })
#define CKH_NARROW_COLS(LIMBS, KERNEL, ...)                                                              \
    with_stages(t.log_n - t.log_n / 2, [&](auto m) {                                                     \
        constexpr u32 M = m.value;                                                                       \
        hipLaunchKernelGGL((KERNEL), dim3((LIMBS) << (t.log_n - fast::NCL<M>)), dim3(fast::NCT<M>), 0, s, __VA_ARGS__); \
    })

void narrow_forward_cols(const NttTables& t, const LimbRef* refs, u32 nrefs, hipStream_t s) {
    if (nrefs == 0) return;
    CKH_NARROW_COLS(nrefs, fast::k_narrow_fwd_cols<M>, t, refs);
}

void narrow_forward_rows(const NttTables& t, const LimbRef* refs, u32 nrefs, const FinishJob* fin, hipStream_t s) {
    if (nrefs == 0) return;
    if (fin)
        CKH_NARROW_ROWS(nrefs, (fast::k_narrow_fwd_rows<M, true>), t, refs, fin);
    else
        CKH_NARROW_ROWS(nrefs, (fast::k_narrow_fwd_rows<M, false>), t, refs, fin);
}

void narrow_inverse_rows(const NttTables& t, const LimbRef* refs, u32 nrefs, hipStream_t s) {
    if (nrefs == 0) return;
    CKH_NARROW_ROWS(nrefs, fast::k_narrow_inv_rows<M>, t, refs);
}

void narrow_inverse_cols(const NttTables& t, const LimbRef* refs, u32 nrefs, const YForm* yf, hipStream_t s) {
    if (nrefs == 0) return;
    if (yf)
        CKH_NARROW_COLS(nrefs, (fast::k_narrow_inv_cols<M, true>), t, refs, yf);
    else
        CKH_NARROW_COLS(nrefs, (fast::k_narrow_inv_cols<M, false>), t, refs, yf);
}

template <u32 MAXS>
static void conv_cols_s(const ConvTables& c, const NttTables& t, const ConvColRef* refs, u32 nrefs, hipStream_t s) {
    with_stages(t.log_n - t.log_n / 2, [&](auto m) {
        constexpr u32 M = m.value;
        const u32 items = nrefs << (t.log_n - fast::NCL<M>);
        hipLaunchKernelGGL((fast::k_narrow_conv_cols<M, MAXS>), dim3((items + 7) / 8 * 8), dim3(fast::NCT<M>), 0, s, c, t, refs,
                           items);
    });
}

void narrow_conv_cols(const ConvTables& c, const NttTables& t, const ConvColRef* refs, u32 nrefs, u32 max_src,
                      hipStream_t s) {
    if (nrefs == 0) return;
    if (max_src <= 1)
        conv_cols_s<1>(c, t, refs, nrefs, s);
    else if (max_src <= 2)
        conv_cols_s<2>(c, t, refs, nrefs, s);
    else if (max_src <= 4)
        conv_cols_s<4>(c, t, refs, nrefs, s);
    else if (max_src <= 6)
        conv_cols_s<6>(c, t, refs, nrefs, s);
    else
        conv_cols_s<8>(c, t, refs, nrefs, s);
}

void narrow_ip_inverse(const NttTables& t, const IpInvJob* jobs, const LimbRef* refs, u32 njobs, const YForm* yf,
                       hipStream_t s) {
    if (njobs == 0) return;
    CKH_NARROW_ROWS(2 * njobs, fast::k_narrow_ip_inv_rows<M>, t, jobs);
    narrow_inverse_cols(t, refs, 2 * njobs, yf, s);
}

void narrow_ip_finish(const NttTables& t, const IpFinJob* jobs, u32 njobs, hipStream_t s) {
    if (njobs == 0) return;
    CKH_NARROW_ROWS(2 * njobs, fast::k_narrow_ip_fin<M>, t, jobs);
}

}  // namespace ckh
