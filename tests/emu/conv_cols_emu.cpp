// CPU replay of the base conversion fused with its targets' column pass (ckks-train_amd/csrc/
// conv_cols.h, the body of k_conv_cols): every work item of a launch over the conversions of a
// context's plans (50-bit sources to 50- and 60-bit targets, 60-bit sources to 50- and 60-bit
// targets, mixed sources; full and shorter digits in one launch, at the launch's source bound),
// followed by the row pass, against the oracle's conversion and transform. Every target word is
// written exactly once, no f64 product leaves its bounds, every LDS slot is used once per phase.
// Test infrastructure only (built and run by tests/test_conv_cols.py).
#include <algorithm>
#include <barrier>
#include <random>
#include <thread>

#include "emu_prelude.h"
#include "conv_cols.h"
#include "conv_tables.h"
#include "ntt_tables.h"

extern "C" {
int or_ntt_forward_limbs(u64 n, const u64* q, u64 limbs, u64* a);
int or_ntt_primes_skip(unsigned bits, u64 n, u64 skip, u64 count, u64* out);
void or_convert(const u64* from, u64 k, const u64* to, u64 t, u64 n, const u64* src, u64* out, int exact);
}

using namespace ckh;
using namespace ckh::fast;

namespace {

typedef unsigned __int128 u128;
u64 mulm(u64 a, u64 b, u64 q) { return (u64)((u128)a * b % q); }

template <class F>
void run_group(emu::Lds& lds, F f) {
    auto done = [&]() noexcept { lds.end_phase(); };
    std::barrier bar(256, done);
    emu::Group g{&lds, [&bar] { bar.arrive_and_wait(); }};
    emu::current() = &g;
    std::vector<std::thread> th;
    for (u32 t = 0; t < NT; ++t)
        th.emplace_back([&f, t] {
            threadIdx.x = t;
            f();
        });
    for (auto& x : th) x.join();
    lds.end_phase();
    emu::current() = nullptr;
}

std::vector<u64> primes_of(unsigned bits, u64 count) {
    std::vector<u64> v(count);
    if (or_ntt_primes_skip(bits, 1ull << 16, 0, count, v.data()) != 0) emu::die("no primes");
    return v;
}

struct Conv {
    std::vector<u32> src, tgt;  // indices into the primes
};

template <u32 M, u32 MAXS>
void replay(u32 log_n, const std::vector<u64>& primes, const std::vector<Conv>& convs, std::mt19937_64& rng, int pattern) {
    const u64 n = 1ull << log_n;
    const u32 tiles = 1u << (log_n - TL);
    const HostNttTables nt = build_ntt_tables(primes, log_n, true);
    HostConvTables T;
    std::vector<std::vector<u64>> ins, outs, xs;
    std::vector<ConvColRef> refs;
    for (const Conv& c : convs) {
        std::vector<std::pair<u32, u32>> tg;
        for (u32 i = 0; i < c.tgt.size(); ++i) tg.push_back({c.tgt[i], i});
        T.add_plan(primes, c.src, tg, 0, false, 0);
        std::vector<u64> x(c.src.size() * n), y(x.size());
        const ConvPlan& P = T.plans.back();
        for (u32 j = 0; j < c.src.size(); ++j) {
            const ConvSrc& s = T.srcs[P.src_first + j];
            for (u64 i = 0; i < n; ++i) {
                const u64 r = rng();
                // y_j = q_j - 1 (the largest), 0 (the most negative after centering), or random
                const u64 yv = pattern == 1 ? s.q - 1 : pattern == 2 ? ((r & 1) ? s.q - 1 : 0) : pattern == 3 ? 0 : r % s.q;
                y[j * n + i] = yv;
                u64 qh = 1 % s.q;  // x = y (Q / q_j) - h
                for (u32 k : c.src)
                    if (primes[k] != s.q) qh = mulm(qh, primes[k] % s.q, s.q);
                x[j * n + i] = (mulm(yv, qh, s.q) + s.q - s.h) % s.q;
            }
        }
        xs.push_back(x);
        ins.push_back(y);
        outs.push_back(std::vector<u64>(c.tgt.size() * n, 0x5a5a5a5a5a5a5a5aull));
    }
    std::vector<std::unique_ptr<emu::Tracked>> tr;
    emu::registry().clear();
    for (size_t k = 0; k < convs.size(); ++k) {
        const ConvPlan& P = T.plans[k];
        u32 small = 1;
        for (u32 j = 0; j < P.nsrc; ++j) small = small && T.srcs[P.src_first + j].fp;
        const u32 first = (u32)refs.size();
        refs.insert(refs.end(), P.ntgt, {ins[k].data(), outs[k].data(), first, P.ntgt, P.src_first, P.tgt_first, P.nsrc, small});
        tr.push_back(std::make_unique<emu::Tracked>(ins[k].data(), ins[k].size(), "sources"));
        emu::registry().push_back(tr.back().get());
        tr.push_back(std::make_unique<emu::Tracked>(outs[k].data(), outs[k].size(), "targets"));
        emu::registry().push_back(tr.back().get());
    }
    emu::Lds lds(LDS_WORDS);
    emu::LdsView lv{&lds};
    for (u32 item = 0; item < refs.size() * tiles; ++item) {
        const ConvColRef& R = refs[item / tiles];
        u32 tile;
        const u32 t = conv_col_item(R, item, tiles, tile);
        const ConvTgt* g = &T.tgts[R.tgt_first + t];
        const PrimeConst* pc = &nt.pc[g->prime];
        u64* out = R.out + (u64)g->limb * n;
        run_group(lds, [&] {
            const u32 tid = threadIdx.x;
            if (pc->q < FP_PRIME_BOUND) {
                const FpAr ar{nt.fwd_f.data() + (u64)g->prime * n, pc->qf, pc->qinv, {}, {}, nullptr};
                double v[16];
                conv_tile<M, MAXS>(ar, T.srcs.data(), R, g, pc, log_n, tile, tid, v);
                fwd_cols_tile<M>(ar, v, out, lv, log_n, tile, tid);
            } else {
                const IntAr ar{nt.fwd.data() + (u64)g->prime * n, pc->q, 0, 0, 0, 0};
                u64 v[16];
                conv_tile<M, MAXS>(ar, T.srcs.data(), R, g, pc, log_n, tile, tid, v);
                fwd_cols_tile<M>(ar, v, out, lv, log_n, tile, tid);
            }
        });
    }
    const u32 B = log_n / 2, rows = 1u << (log_n - B);
    for (size_t k = 0; k < convs.size(); ++k) {
        const Conv& c = convs[k];
        for (size_t i = 0; i < outs[k].size(); ++i)
            if (tr[2 * k + 1]->writes[i] != 1 || tr[2 * k + 1]->reads[i] != 0) emu::die("a target word not written exactly once", (double)i);
        std::vector<u64> sq, tq, sh(xs[k]);
        for (u32 s : c.src) sq.push_back(primes[s]);
        for (u32 t : c.tgt) tq.push_back(primes[t]);
        for (size_t j = 0; j < sq.size(); ++j)
            for (u64 i = 0; i < n; ++i) sh[j * n + i] = (sh[j * n + i] + (sq[j] >> 1)) % sq[j];
        std::vector<u64> want(tq.size() * n);
        or_convert(sq.data(), sq.size(), tq.data(), tq.size(), n, sh.data(), want.data(), sq.size() > 1);
        for (size_t t = 0; t < tq.size(); ++t) {
            const u64 r = tq[t];
            u64 qm = 1 % r;
            for (u64 s : sq) qm = mulm(qm, s % r, r);
            const u64 half = mulm((qm + r - 1) % r, (r + 1) / 2, r);
            for (u64 i = 0; i < n; ++i) want[t * n + i] = (want[t * n + i] + r - half) % r;
        }
        or_ntt_forward_limbs(n, tq.data(), tq.size(), want.data());
        for (size_t t = 0; t < tq.size(); ++t) {
            u64* limb = outs[k].data() + t * n;
            const u32 prime = c.tgt[t];
            const PrimeConst& pc = nt.pc[prime];
            for (u32 tile = 0; tile < tiles; ++tile)
                run_group(lds, [&] {
                    auto go = [&](const auto& ar) {
                        if (B == 6) fwd_rows<6>(ar, limb, limb, lv, log_n, nullptr, pc.q, tile);
                        else if (B == 7) fwd_rows<7>(ar, limb, limb, lv, log_n, nullptr, pc.q, tile);
                        else fwd_rows<8>(ar, limb, limb, lv, log_n, nullptr, pc.q, tile);
                    };
                    if (pc.q < FP_PRIME_BOUND)
                        go(FpAr{nt.fwd_f.data() + (u64)prime * n, pc.qf, pc.qinv, {}, {}, nt.rf.data() + (u64)prime * rows * ROW_FACTOR_SLOTS});
                    else
                        go(IntAr{nt.fwd.data() + (u64)prime * n, pc.q, 0, 0, 0, 0});
                });
            for (u64 i = 0; i < n; ++i)
                if (limb[i] != want[t * n + i]) {
                    std::fprintf(stderr, "conversion %zu target %zu word %llu pattern %d\n", k, t, (unsigned long long)i, pattern);
                    emu::die("fused conversion differs from the oracle");
                }
        }
    }
    std::printf("N = 2^%u, at most %u sources, pattern %d: exact\n", log_n, MAXS, pattern);
    std::fflush(stdout);
}

}  // namespace

int main() {
    std::mt19937_64 rng(771);
    const std::vector<u64> q50 = primes_of(50, 10), q60 = primes_of(60, 9), q40 = primes_of(40, 2);
    std::vector<u64> P(q50);
    P.insert(P.end(), q60.begin(), q60.end());  // 10..18
    P.insert(P.end(), q40.begin(), q40.end());  // 19, 20
    // sources up to the launch's bound and clipped ones in one launch
    for (int pat : {0, 1, 2, 3}) {
        replay<6, 2>(12, P, {{{0, 1}, {2, 10}}, {{3}, {4, 19, 11}}, {{12, 13}, {0, 20}}, {{10, 19}, {0, 11}}}, rng, pat);
        replay<6, 6>(12, P, {{{0, 1, 2, 3, 4, 5}, {6, 10}}, {{0, 1, 2}, {8, 19}}, {{10, 11, 12, 13, 14, 15}, {0, 20, 16}}}, rng, pat);
        replay<6, 8>(12, P, {{{0, 1, 2, 3, 4, 5, 6, 7}, {8, 10}}, {{10, 11, 12, 13, 14, 15, 16, 17}, {0, 18}}}, rng, pat);
    }
    replay<6, 1>(12, P, {{{0}, {1, 10}}, {{10}, {0, 11}}}, rng, 0);
    replay<7, 4>(13, P, {{{0, 1, 2}, {6, 10}}, {{10, 11, 12, 13}, {1, 19}}}, rng, 2);
    replay<7, 4>(14, P, {{{0, 1, 2, 3}, {6, 10}}}, rng, 0);
    replay<8, 6>(15, P, {{{10, 11, 12, 13}, {0}}, {{0, 1, 2, 3, 4, 5}, {10}}}, rng, 1);
    replay<8, 6>(16, P, {{{0, 1, 2, 3, 4, 5}, {6}}}, rng, 2);
    std::printf("EMU OK\n");
    return 0;
}
