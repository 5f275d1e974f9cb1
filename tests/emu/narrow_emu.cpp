// CPU replay of the narrow passes (ckks-train_amd/csrc/narrow_passes.h): both transforms for N = 2^12 ..
// 2^16, and at 2^12 and 2^13 a key switch's apply stage (inner product + inverse transform in y form;
// conversion + column pass; row pass + inner product + finish, with and without the Galois permutation, an
// own digit and addends, part b's read through the same permutation; row pass + finish), for 50-, 40- and 60-bit primes, against the oracle's
// transforms and conversion and 128-bit sums. LDS: between two barriers no thread touches a slot that
// another one writes. Test infrastructure only (built by tests/test_narrow.py).
#include <algorithm>
#include <barrier>
#include <memory>
#include <random>
#include <thread>

#include "emu_prelude.h"
#include "narrow_passes.h"
#include "conv_tables.h"
#include "ntt_tables.h"

extern "C" {
int or_ntt_forward_limbs(u64 n, const u64* q, u64 limbs, u64* a);
int or_ntt_inverse_limbs(u64 n, const u64* q, u64 limbs, u64* a);
int or_ntt_primes_skip(unsigned bits, u64 n, u64 skip, u64 count, u64* out);
void or_convert(const u64* from, u64 k, const u64* to, u64 t, u64 n, const u64* src, u64* out, int exact);
void or_galois_perm_ntt(u64 n, u64 g, uint32_t* perm);
u64 or_galois_elt(u64 n, int step);
}

using namespace ckh;
using namespace ckh::fast;

namespace {

typedef unsigned __int128 u128;
u64 mulm(u64 a, u64 b, u64 q) { return (u64)((u128)a * b % q); }

// LDS with an owner per slot and phase: 0 untouched, t + 1 one thread's, ~0u read by several.
struct OwnLds {
    std::vector<u64> w;
    std::vector<std::atomic<u32>> owner;
    std::vector<std::atomic<u32>> written;
    explicit OwnLds(size_t n) : w(n), owner(n), written(n) {}
    void touch(u32 i, bool write) {
        if (i >= w.size()) emu::die("LDS index out of range", i);
        const u32 me = threadIdx.x + 1;
        if (write) written[i] = 1;
        u32 was = 0;
        if (!owner[i].compare_exchange_strong(was, me) && was != me) {
            if (write || written[i]) emu::die("LDS slot shared by a writing thread and another in one phase", i);
            owner[i] = ~0u;
        }
        if (owner[i] == ~0u && written[i]) emu::die("LDS slot written while others read it", i);
    }
    void end_phase() {
        for (auto& o : owner) o = 0;
        for (auto& o : written) o = 0;
    }
};
struct OwnRef {
    OwnLds* l;
    u32 i;
    operator u64() const {
        l->touch(i, false);
        return l->w[i];
    }
    const OwnRef& operator=(u64 v) const {
        l->touch(i, true);
        l->w[i] = v;
        return *this;
    }
};
struct OwnView {
    OwnLds* l;
    OwnRef operator[](u32 i) const { return OwnRef{l, i}; }
};

template <class F>
void run_group(OwnLds& lds, u32 threads, F f) {
    auto done = [&]() noexcept { lds.end_phase(); };
    std::barrier bar(threads, done);
    emu::Group g{nullptr, [&bar] { bar.arrive_and_wait(); }};
    emu::current() = &g;
    std::vector<std::thread> th;
    for (u32 t = 0; t < threads; ++t)
        th.emplace_back([&f, t] {
            threadIdx.x = t;
            f(t);
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

template <u32 LOGN>
struct Replay {
    static constexpr u64 n = 1ull << LOGN;
    static constexpr u32 B = LOGN / 2, A = LOGN - B, TILES = 1u << (LOGN - NTL), CTILES = 1u << (LOGN - NCL<A>);
    std::vector<u64> primes;
    HostNttTables nt;
    std::mt19937_64 rng{4711};
    OwnLds lds{std::max(NLDS, NCLDS<A>)};
    std::vector<std::unique_ptr<emu::Tracked>> tr;
    explicit Replay(const std::vector<u64>& p) : primes(p), nt(build_ntt_tables(p, LOGN, true)) {}

    void track(const std::vector<u64>& v, const char* name) {
        tr.push_back(std::make_unique<emu::Tracked>(v.data(), v.size(), name));
        emu::registry().push_back(tr.back().get());
    }
    void untrack() {
        emu::registry().clear();
        tr.clear();
    }
    std::vector<u64> limb(u32 prime, int pat = 0) {
        std::vector<u64> v(n);
        for (auto& x : v) x = pat == 1 ? primes[prime] - 1 : pat == 2 ? ((rng() & 1) ? primes[prime] - 1 : 0) : rng() % primes[prime];
        return v;
    }
    static void same(const std::vector<u64>& a, const u64* b, const char* what) {
        for (u64 i = 0; i < n; ++i)
            if (a[i] != b[i]) emu::die(what, (double)i);
    }
    template <class F>
    void with(u32 prime, bool fwd, F f) {
        const PrimeConst& pc = nt.pc[prime];
        if (pc.q < FP_PRIME_BOUND)
            f(FpAr{(fwd ? nt.fwd_f : nt.inv_f).data() + prime * n, pc.qf, pc.qinv, pc.n_inv_f, pc.w_n_inv_f, nullptr});
        else
            f(IntAr{(fwd ? nt.fwd : nt.inv).data() + prime * n, pc.q, pc.n_inv, pc.n_inv_s, pc.w_n_inv, pc.w_n_inv_s});
    }
    static void set_y(FpAr& ar, const YForm& y) { ar.ninv = y.n_f, ar.wninv = y.wn_f, ar.add = y.h_f; }
    static void set_y(IntAr& ar, const YForm& y) { ar.n_inv = y.n, ar.n_inv_s = y.n_s, ar.w_n_inv = y.wn, ar.w_n_inv_s = y.wn_s, ar.add = y.h; }

    // The narrow forward passes alone, and each with the 16-word pass of the other kind.
    void transforms(u32 prime, int pat) {
        const std::vector<u64> in = limb(prime, pat);
        std::vector<u64> f(n, ~0ull), b(n, ~0ull), want(in);
        track(in, "in");
        track(f, "fwd");
        track(b, "inv");
        OwnView lv{&lds};
        with(prime, true, [&](const auto& ar) {
            for (u32 tile = 0; tile < CTILES; ++tile)
                run_group(lds, NCT<A>, [&](u32 tid) {
                    const NarrowCol<A> P(LOGN, tile, tid);
                    narrow_fwd_cols<A>(ar, P, f.data(), lv, [&](auto& v) {
                        for (u32 k = 0; k < NW; ++k) v[k] = ar.from_canon(glb(in.data())[P.word(sub(P.o, k, A - LW))]);
                    });
                });
            for (u32 tile = 0; tile < TILES; ++tile)
                run_group(lds, NT, [&](u32 tid) { narrow_fwd_rows_store<B>(ar, f.data(), lv, LOGN, tile, tid); });
        });
        or_ntt_forward_limbs(n, &primes[prime], 1, want.data());
        same(f, want.data(), "narrow forward transform differs");
        with(prime, false, [&](const auto& ar) {
            for (u32 tile = 0; tile < TILES; ++tile)
                run_group(lds, NT, [&](u32 tid) {
                    const NarrowRow<B> P(tile, tid);
                    narrow_inv_rows<B>(ar, P, b.data(), lv, LOGN, [&](auto& v) {
                        for (u32 k = 0; k < NW; ++k) v[k] = ar.from_canon(glb(f.data())[P.word(NW * P.o + k)]);
                    });
                });
            for (u32 tile = 0; tile < CTILES; ++tile)
                run_group(lds, NCT<A>, [&](u32 tid) { narrow_inv_cols<A, false>(ar, b.data(), lv, LOGN, tile, tid); });
        });
        same(b, in.data(), "narrow inverse transform differs");
        untrack();
    }

    // One switch's second half on one ring: digits, keys of every limb, mod_down from P to Q.
    void apply(const std::vector<u32>& Q, const std::vector<u32>& P, u32 ndig, u64 galois, bool own, bool add, int pat) {
        HostConvTables T;
        std::vector<std::pair<u32, u32>> tg;
        for (u32 i = 0; i < Q.size(); ++i) tg.push_back({Q[i], i});
        T.add_plan(primes, P, tg, 0, false, 0);
        const std::vector<YForm> yf = T.yform(nt.pc);
        const u64 lw = Q.size() + P.size();
        auto prime_of = [&](u64 l) { return l < Q.size() ? Q[l] : P[l - Q.size()]; };
        std::vector<u64> dig, key, ownv, addv, y(2 * P.size() * n), z(2 * Q.size() * n), out(2 * Q.size() * n);
        for (u32 j = 0; j < ndig; ++j)
            for (u64 l = 0; l < lw; ++l) {
                const auto d = limb(prime_of(l), pat);
                dig.insert(dig.end(), d.begin(), d.end());
            }
        for (u32 j = 0; j < 2 * ndig; ++j)
            for (u64 l = 0; l < lw; ++l) {
                const auto k = limb(prime_of(l), pat);
                key.insert(key.end(), k.begin(), k.end());
            }
        for (u32 q : Q) {
            const auto o = limb(q, pat);
            ownv.insert(ownv.end(), o.begin(), o.end());
        }
        for (u32 part = 0; part < 2; ++part)
            for (u32 q : Q) {
                const auto a = limb(q, pat);
                addv.insert(addv.end(), a.begin(), a.end());
            }
        track(dig, "digits");
        track(key, "key");
        track(ownv, "own");
        track(addv, "addend");
        track(y, "y");
        track(z, "z");
        track(out, "out");
        const u32 own_j = ndig / 2;
        OwnView lv{&lds};
        auto limb_job = [&](u64 l, bool o) {
            return LimbIp{dig.data() + l * n, lw * n, o ? ownv.data() + l * n : nullptr, key.data() + l * n, lw * n, galois, ndig, own_j};
        };
        const u64 yw = P.size() * n, zw = Q.size() * n;
        for (u32 k = 0; k < P.size(); ++k)
            with(P[k], false, [&](auto ar) {
                set_y(ar, yf[k]);
                const IpInvJob J{limb_job(Q.size() + k, false), y.data() + k * n, yw, P[k], 0};
                for (u32 part = 0; part < 2; ++part) {
                    for (u32 tile = 0; tile < TILES; ++tile)
                        run_group(lds, NT, [&](u32 tid) { narrow_ip_inv_rows<B>(ar, J, part, &nt.pc[P[k]], lv, LOGN, tile, tid); });
                    for (u32 tile = 0; tile < CTILES; ++tile)
                        run_group(lds, NCT<A>, [&](u32 tid) { narrow_inv_cols<A, true>(ar, y.data() + part * yw + k * n, lv, LOGN, tile, tid); });
                }
            });
        std::vector<uint32_t> perm(n);
        for (u64 i = 0; i < n; ++i) perm[i] = (uint32_t)i;
        if (galois) or_galois_perm_ntt(n, galois, perm.data());
        auto sum = [&](u64 l, bool o, u32 part) {
            const u64 q = primes[prime_of(l)];
            std::vector<u64> s(n, 0);
            for (u32 j = 0; j < ndig; ++j)
                for (u64 i = 0; i < n; ++i) {
                    const u64 d = o && j == own_j ? ownv[l * n + perm[i]] : dig[(j * lw + l) * n + perm[i]];
                    s[i] = (s[i] + mulm(d, key[((2 * j + part) * lw + l) * n + i], q)) % q;
                }
            return s;
        };
        std::vector<u64> pq, qq;
        for (u32 p : P) pq.push_back(primes[p]);
        for (u32 q : Q) qq.push_back(primes[q]);
        const u32 small = std::all_of(T.srcs.begin(), T.srcs.end(), [](const ConvSrc& s) { return s.fp; });
        for (u32 part = 0; part < 2; ++part) {
            // the P part's coefficients, shifted, converted by the oracle
            std::vector<u64> sh;
            for (u32 k = 0; k < P.size(); ++k) {
                std::vector<u64> s = sum(Q.size() + k, false, part);
                or_ntt_inverse_limbs(n, &pq[k], 1, s.data());
                for (u64 i = 0; i < n; ++i) {
                    const u64 v = (s[i] + (pq[k] >> 1)) % pq[k];
                    if (y[part * yw + k * n + i] != mulm(v, T.srcs[k].qhinv, pq[k]))
                        emu::die("inner product + inverse in y form differs", (double)i);
                    sh.push_back(v);
                }
            }
            std::vector<u64> w(Q.size() * n);
            or_convert(pq.data(), pq.size(), qq.data(), qq.size(), n, sh.data(), w.data(), pq.size() > 1);
            for (u32 l = 0; l < Q.size(); ++l) {
                const u64 q = qq[l];
                u64 pm = 1 % q;
                for (u64 p : pq) pm = mulm(pm, p % q, q);
                const u64 h = mulm((pm + q - 1) % q, (q + 1) / 2, q);
                for (u64 i = 0; i < n; ++i) w[l * n + i] = (w[l * n + i] + q - h) % q;
                or_ntt_forward_limbs(n, &q, 1, w.data() + l * n);
                const u64 inv = hm::inv(pm, q);
                std::vector<u64> s = sum(l, own, part), want(n);
                for (u64 i = 0; i < n; ++i) {
                    want[i] = mulm((s[i] + q - w[l * n + i]) % q, inv, q);
                    if (add) want[i] = (want[i] + addv[part * zw + l * n + (part ? i : perm[i])]) % q;
                }
                const ConvColRef R{y.data() + part * yw, nullptr, 0, 1, 0, l, (u32)P.size(), small};
                const ConvTgt* tgp = &T.tgts[l];
                IpFinJob J{limb_job(l, own), z.data() + l * n, zw, out.data() + l * n, out.data() + zw + l * n,
                           add ? addv.data() + l * n : nullptr, add ? addv.data() + zw + l * n : nullptr, inv, hm::shoup(inv, q),
                           {(double)inv, (double)inv / (double)q}, Q[l], (u32)galois};
                u64* zl = z.data() + part * zw + l * n;
                with(Q[l], true, [&](const auto& ar) {
                    for (u32 tile = 0; tile < CTILES; ++tile)
                        run_group(lds, NCT<A>, [&](u32 tid) {
                            const NarrowCol<A> C(LOGN, tile, tid);
                            narrow_fwd_cols<A>(ar, C, zl, lv, [&](auto& v) {
                                conv_words<NW, 4>(ar, T.srcs.data(), R, tgp, &nt.pc[Q[l]], LOGN, (u32)C.word(C.o), A - LW + C.B, v);
                            });
                        });
                    for (u32 tile = 0; tile < TILES; ++tile)
                        run_group(lds, NT, [&](u32 tid) { narrow_ip_fin<B>(ar, J, part, &nt.pc[Q[l]], q, lv, LOGN, tile, tid); });
                    const u64* got = out.data() + part * zw + l * n;
                    for (u64 i = 0; i < n; ++i)
                        if (got[i] != want[i]) emu::die("narrow row pass + inner product + finish differs", (double)i, l);
                    // the finish alone, its first operand in memory
                    std::copy(s.begin(), s.end(), ownv.begin() + l * n);
                    const FinishJob F{ownv.data() + l * n, zl, out.data() + part * zw + l * n, add ? addv.data() + part * zw + l * n : nullptr,
                                      inv, hm::shoup(inv, q), Q[l], part ? 0 : (u32)galois, {(double)inv, (double)inv / (double)q}};
                    std::fill(out.begin(), out.end(), ~0ull);
                    for (u32 tile = 0; tile < TILES; ++tile)
                        run_group(lds, NT, [&](u32 tid) { narrow_fin<B>(ar, zl, &F, q, lv, LOGN, tile, tid); });
                    for (u64 i = 0; i < n; ++i)
                        if (got[i] != want[i]) emu::die("narrow row pass + finish differs", (double)i, l);
                });
            }
        }
        untrack();
    }
};

template <u32 LOGN>
void run(const std::vector<u64>& P) {
    Replay<LOGN> r(P);
    for (u32 p : {0u, 4u}) r.transforms(p, LOGN % 3);
    const u64 g = or_galois_elt(1ull << LOGN, 5);
    if (LOGN == 12) {
        for (int pat : {1, 2}) r.transforms(8, pat);
        r.apply({0, 1, 4}, {5, 6}, 3, 0, true, true, 0);   // 60-bit special primes; 50- and 60-bit limbs
        r.apply({0, 4}, {2}, 1, g, true, false, 1);        // one special prime, below 2^50
        r.apply({1, 4}, {2, 3}, 2, 0, false, true, 2);
    }
    if (LOGN == 13) r.apply({0, 8}, {5, 6, 7}, 5, g, false, true, 2);  // a 40-bit limb, five digits, permuted
    std::printf("N = 2^%u: narrow passes exact\n", LOGN);
    std::fflush(stdout);
}

}  // namespace

int main() {
    std::vector<u64> P = primes_of(50, 4);
    for (u64 p : primes_of(60, 4)) P.push_back(p);
    for (u64 p : primes_of(40, 1)) P.push_back(p);
    run<12>(P);
    run<13>(P);
    run<14>(P);
    run<15>(P);
    run<16>(P);
    std::printf("EMU OK\n");
    return 0;
}
