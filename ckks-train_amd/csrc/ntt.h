// NTT launchers (see ntt.hip for the schedule).
#pragma once
#include "common.h"

namespace ckh {

// Device tables shared by every transform of a context: per-prime constants and, per prime,
// N (w, w') pairs for the forward (psi^i at bitrev(i)) and inverse (psi^-i) directions.
struct NttTables {
    u32 log_n;
    const PrimeConst* pc;
    const Tw* fwd;     // [prime][N]
    const Tw* inv;     // [prime][N]
    const FTw* fwd_f;  // [prime][N], f64 path (primes below 2^50)
    const FTw* inv_f;
    // Row factors of the register-radix row pass (N = 2^(A+M), M = log N / 2 row stages):
    // rf[prime][row][s] = fwd_f[prime][2^(A+s) + row 2^s] for s < M (8 slots per row); ri the
    // same over inv_f. Every row-pass twiddle is a row factor times one of the first 2^M entries.
    const FTw* rf;
    const FTw* ri;
};


// Register-radix passes (ntt_fast.hip) for 2^12 <= N <= 2^16.
bool ntt_fast_supported(u32 log_n);

// The one-launch forward transform (both passes in one persistent launch, the intermediate handed
// from the column pass to the row pass through the L2 of one XCD). Its control block: a ticket
// counter per XCD, CTL_STRIDE words apart, then one done-counter per limb; zero before each
// launch (fused_ctl_words(nrefs) u32 words).
constexpr u32 CTL_STRIDE = 64;
constexpr u32 FUSED_CTL_HEAD = 8 * CTL_STRIDE;
inline u64 fused_ctl_words(u32 nrefs) { return FUSED_CTL_HEAD + nrefs; }
struct FusedCfg {
    u32 nx = 0;      // XCDs (0: the one-launch transform is unavailable)
    u32 lag = 8;     // slots between a limb's first-pass tiles and its second-pass tiles
    u32 grid = 0;    // persistent workgroups
    u32* err = nullptr;  // device word set when a wait overran its bound
};
// XCD count of this device: the workgroups of a probe grid report XCD ids 0..count-1, each id on
// a fair share of them (else 0: the one-launch transform stays off).
u32 xcc_layout_check(hipStream_t stream);
// Workgroups of the one-launch transform that fit on one CU at once.
u32 fused_occupancy();
struct FinishJob;
// ntt_fast_forward (fin null) or ntt_fast_forward_finish in one launch; ctl zeroed, nrefs words
// of done-counters after its head.
void ntt_fast_forward_fused(const NttTables& t, const LimbRef* refs, u32 nrefs, const FinishJob* fin, u32* ctl,
                            const FusedCfg& f, hipStream_t stream);
// ntt_fast_inverse in one launch (row pass, then the column pass in place on dst).
void ntt_fast_inverse_fused(const NttTables& t, const LimbRef* refs, u32 nrefs, u32* ctl, const FusedCfg& f,
                            hipStream_t stream);
void ntt_fast_forward(const NttTables& t, const LimbRef* refs, u32 nrefs, hipStream_t stream);
// yf non-null: every ref leaves in the y form of the conversion source yf[ref.aux] (YForm).
void ntt_fast_inverse(const NttTables& t, const LimbRef* refs, u32 nrefs, hipStream_t stream,
                      const YForm* yf = nullptr);
// Forward NTT whose row pass ends with fin[r]: out = (a - NTT(src)) * inv (+ add) instead of
// storing the transform (fin is a FinishJob array, one per ref).
void ntt_fast_forward_finish(const NttTables& t, const LimbRef* refs, const FinishJob* fin, u32 nrefs,
                             hipStream_t stream);

// The two passes of ntt_fast_forward separately (column pass: src -> dst; row pass: in place on
// dst; between them dst holds f64 intermediates, not residues).
void ntt_fast_forward_cols(const NttTables& t, const LimbRef* refs, u32 nrefs, hipStream_t stream);
void ntt_fast_forward_rows(const NttTables& t, const LimbRef* refs, u32 nrefs, hipStream_t stream);

// The row pass alone with the finish of ntt_fast_forward_finish.
void ntt_fast_forward_rows_finish(const NttTables& t, const LimbRef* refs, const FinishJob* fin, u32 nrefs,
                                  hipStream_t stream);

// Base conversions of at most WRAP_SRC sources (y form) fused with the column pass of every target:
// each ref's limb holds the column pass's f64 / lazy intermediates afterwards, as after
// ntt_fast_forward_cols.
struct ConvTables;
struct ConvColRef;
void conv_cols_launch(const ConvTables& c, const NttTables& t, const ConvColRef* refs, u32 nrefs, u32 max_src,
                      hipStream_t stream);

// The narrow passes (ntt_narrow.hip), for launches of few tiles: each pass of the transforms, the fused
// conversion, the inner product + inverse transform in y form (jobs: njobs limbs, both parts each; refs:
// the 2 njobs limbs whose inverse column pass follows, in place) and the row pass + inner product + finish.
//
// Where the line lies, in 4096-word tiles of a launch: the row passes and, up to N = 2^14, the column
// passes are faster narrow up to some thousand tiles (64 switches at 2^12: 134 against 146 us, 24 at 2^14:
// 199 against 218, four at 2^16: 494 against 509; sixteen hoisted rotations at 2^16 1102 against 1147 us
// with every row pass narrow, whose finish takes 279 us narrow and 227 wide at 9728 tiles). Above 2^14
// the column passes change over once the chip is full: 320 tiles against 640 or more, 134 against 140
// us for an 18-limb switch at 2^16 and 183 against 184 for 24 limbs, against none the same switch of 8
// limbs 85 against 98; all column passes narrow, a batch of 256 switches takes 19.5 against 16.4 ms.
//
// Transforms of their own (narrow_alone) change over at 128 tiles: the narrow passes load 12 twiddles for 4
// words, which bounds 50-bit limbs from about 256 tiles on (forward at 2^14, wide / narrow: 64 tiles 10.2 /
// 8.2 us, 256 12.0 / 19.0, 3,840 88 / 123), where a key switch's launches hold 60-bit limbs, whose wide
// passes read the whole table too.
constexpr u32 NARROW_ALONE_TILES = 128;
inline bool narrow_alone(u32 log_n, u32 nrefs) { return ((u64)nrefs << (log_n - 12)) <= NARROW_ALONE_TILES; }
constexpr u32 NARROW_TILES = 4096, NARROW_COL8_TILES = 320;
inline bool narrow_rows(u32 log_n, u32 nrefs) { return ((u64)nrefs << (log_n - 12)) <= NARROW_TILES; }
inline bool narrow_cols(u32 log_n, u32 nrefs) {
    return ((u64)nrefs << (log_n - 12)) <= (log_n > 14 ? NARROW_COL8_TILES : NARROW_TILES);
}
struct IpInvJob;
struct IpFinJob;
void narrow_forward_cols(const NttTables& t, const LimbRef* refs, u32 nrefs, hipStream_t stream);
void narrow_forward_rows(const NttTables& t, const LimbRef* refs, u32 nrefs, const FinishJob* fin, hipStream_t stream);
void narrow_inverse_rows(const NttTables& t, const LimbRef* refs, u32 nrefs, hipStream_t stream);
void narrow_inverse_cols(const NttTables& t, const LimbRef* refs, u32 nrefs, const YForm* yf, hipStream_t stream);
void narrow_conv_cols(const ConvTables& c, const NttTables& t, const ConvColRef* refs, u32 nrefs, u32 max_src,
                      hipStream_t stream);
void narrow_ip_inverse(const NttTables& t, const IpInvJob* jobs, const LimbRef* refs, u32 njobs, const YForm* yf,
                       hipStream_t stream);
void narrow_ip_finish(const NttTables& t, const IpFinJob* jobs, u32 njobs, hipStream_t stream);

void rows_ip_launch(const NttTables& t, const RowIpJob* jobs, u32 njobs, hipStream_t stream);

void rows_ip_fin_launch(const NttTables& t, const RowIpFinJob* jobs, u32 njobs, hipStream_t stream);

// ref.dst <- NTT(ref.src) for each of the nrefs descriptors (device array). src may equal
// dst (in place). Inputs reduced, outputs reduced.
void ntt_forward(const NttTables& t, const LimbRef* refs, u32 nrefs, hipStream_t stream);
void ntt_inverse(const NttTables& t, const LimbRef* refs, u32 nrefs, hipStream_t stream);

}  // namespace ckh
