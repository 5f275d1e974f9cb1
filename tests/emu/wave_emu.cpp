// CPU replay of the row passes (ckks-train_amd/csrc/ntt_passes.h and narrow_passes.h) with their LDS exchanges
// ordered inside one wave only: CKH_WAVE_SYNC waits for the 64 threads of the caller's wave, and between two
// barriers of the workgroup every LDS slot belongs to the one wave that touched it first. A pass whose exchange
// crossed waves would be ordered by nothing on the device; here it ends the program. The transforms and the
// fused inner product are compared with the oracle as well. Test infrastructure only (built by
// tests/test_wave.py). argv[1]: the threads of a wave (64); with 32, as a planted mistake, the row passes
// whose words are laid out for 64 have to be caught.
#include <barrier>
#include <memory>
#include <random>
#include <thread>

#include "emu_prelude.h"

namespace wave {
inline u32 size = 64;
inline std::vector<std::unique_ptr<std::barrier<>>> bars;  // one per wave of the workgroup
inline void sync() { bars[threadIdx.x / size]->arrive_and_wait(); }
}  // namespace wave
#define CKH_WAVE_SYNC() wave::sync()

#include "narrow_passes.h"
#include "ntt_tables.h"

extern "C" {
int or_ntt_forward_limbs(u64 n, const u64* q, u64 limbs, u64* a);
int or_ntt_inverse_limbs(u64 n, const u64* q, u64 limbs, u64* a);
int or_ntt_primes_skip(unsigned bits, u64 n, u64 skip, u64 count, u64* out);
}

using namespace ckh;
using namespace ckh::fast;

namespace {

// LDS words with the wave that owns each between two barriers of the workgroup (0: none yet).
struct WaveLds {
    std::vector<u64> w = std::vector<u64>(LDS_WORDS);
    std::vector<std::atomic<u32>> owner = std::vector<std::atomic<u32>>(LDS_WORDS);
    void touch(u32 i) {
        if (i >= w.size()) emu::die("LDS index out of range", i);
        const u32 me = threadIdx.x / wave::size + 1;
        u32 was = 0;
        if (!owner[i].compare_exchange_strong(was, me) && was != me) emu::die("LDS slot shared by two waves", i, was, me);
    }
    void end_phase() {
        for (auto& o : owner) o = 0;
    }
};
struct WaveRef {
    WaveLds* l;
    u32 i;
    operator u64() const {
        l->touch(i);
        return l->w[i];
    }
    const WaveRef& operator=(u64 v) const {
        l->touch(i);
        l->w[i] = v;
        return *this;
    }
};
struct WaveView {
    WaveLds* l;
    WaveRef operator[](u32 i) const { return WaveRef{l, i}; }
};

template <class F>
void run_group(WaveLds& lds, u32 threads, F f) {
    auto done = [&]() noexcept { lds.end_phase(); };
    std::barrier bar(threads, done);
    wave::bars.clear();
    for (u32 k = 0; k < threads / wave::size; ++k) wave::bars.push_back(std::make_unique<std::barrier<>>(wave::size));
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

struct Limb {
    u32 log_n;
    u64 q;
    HostNttTables t;
    u64 n() const { return 1ull << log_n; }
};

template <class F>
void with(const Limb& L, bool fwd, F f) {
    const PrimeConst& pc = L.t.pc[0];
    if (L.q < FP_PRIME_BOUND)
        f(FpAr{(fwd ? L.t.fwd_f : L.t.inv_f).data(), pc.qf, pc.qinv, pc.n_inv_f, pc.w_n_inv_f, (fwd ? L.t.rf : L.t.ri).data()});
    else
        f(IntAr{(fwd ? L.t.fwd : L.t.inv).data(), pc.q, pc.n_inv, pc.n_inv_s, pc.w_n_inv, pc.w_n_inv_s});
}

struct Arrays {
    std::vector<std::unique_ptr<emu::Tracked>> t;
    explicit Arrays(std::initializer_list<std::vector<u64>*> v) {
        for (auto* x : v) {
            t.push_back(std::make_unique<emu::Tracked>(x->data(), x->size(), "array"));
            emu::registry().push_back(t.back().get());
        }
    }
    ~Arrays() { emu::registry().clear(); }
};

std::vector<u64> oracle(const Limb& L, std::vector<u64> a, bool fwd) {
    if ((fwd ? or_ntt_forward_limbs : or_ntt_inverse_limbs)(L.n(), &L.q, 1, a.data()) != 0) emu::die("oracle transform failed");
    return a;
}

std::vector<u64> random_limb(const Limb& L, std::mt19937_64& g) {
    std::vector<u64> v(L.n());
    for (auto& x : v) x = g() % L.q;
    return v;
}

void same(const std::vector<u64>& a, const std::vector<u64>& b, const char* what) {
    for (size_t i = 0; i < a.size(); ++i)
        if (a[i] != b[i]) emu::die(what, (double)i);
}

// The column pass of a forward transform, in place (its exchanges are the workgroup's).
template <u32 A>
void cols(const Limb& L, WaveLds& lds, std::vector<u64>& v) {
    with(L, true, [&](const auto& ar) {
        for (u32 tile = 0; tile < L.n() >> TL; ++tile)
            run_group(lds, NT, [&](u32) { fwd_cols<A>(ar, v.data(), v.data(), WaveView{&lds}, L.log_n, tile); });
    });
}

template <u32 A, u32 B>
void replay(const Limb& L, std::mt19937_64& g) {
    WaveLds lds;
    const WaveView lv{&lds};
    const u64 n = L.n(), q = L.q;
    const u32 tiles = (u32)(n >> TL), ntiles = (u32)(n >> NTL);
    const std::vector<u64> x = random_limb(L, g), X = oracle(L, x, true);
    for (bool narrow : {false, true}) {
        std::vector<u64> v = x, u = X;
        Arrays keep{&v, &u};
        cols<A>(L, lds, v);
        with(L, true, [&](const auto& ar) {
            for (u32 tile = 0; tile < (narrow ? ntiles : tiles); ++tile)
                run_group(lds, NT, [&](u32 tid) {
                    if (narrow)
                        narrow_fwd_rows_store<B>(ar, v.data(), lv, L.log_n, tile, tid);
                    else
                        fwd_rows<B>(ar, v.data(), v.data(), lv, L.log_n, nullptr, q, tile, tid);
                });
        });
        same(v, X, "forward transform differs");
        with(L, false, [&](const auto& ar) {
            for (u32 tile = 0; tile < (narrow ? ntiles : tiles); ++tile)
                run_group(lds, NT, [&](u32 tid) {
                    if (narrow) {
                        const NarrowRow<B> P(tile, tid);
                        narrow_inv_rows<B>(ar, P, u.data(), lv, L.log_n, [&](auto& w) {
                            for (u32 k = 0; k < NW; ++k) w[k] = ar.from_canon(glb(u.data())[P.word(NW * P.o + k)]);
                        });
                    } else {
                        inv_rows<B>(ar, u.data(), u.data(), lv, L.log_n, tile, tid);
                    }
                });
            for (u32 tile = 0; tile < tiles; ++tile)
                run_group(lds, NT, [&](u32 tid) { inv_cols<A>(ar, u.data(), lv, L.log_n, tile, tid); });
        });
        same(u, x, "inverse transform differs");
    }

    // the finishes: (a - NTT(x)) inv + add
    const std::vector<u64> a = random_limb(L, g), add = random_limb(L, g);
    const u64 inv = 1 + g() % (q - 1);
    auto mulm = [&](u64 y, u64 z) { return (u64)((unsigned __int128)y * z % q); };
    for (bool narrow : {false, true}) {
        std::vector<u64> v = x, a1 = a, add1 = add, out(n);
        Arrays keep{&v, &a1, &add1, &out};
        cols<A>(L, lds, v);
        const FinishJob F{a1.data(), v.data(), out.data(), add1.data(), inv, hm::shoup(inv, q), 0, 0,
                          {(double)inv, (double)inv / (double)q}};
        with(L, true, [&](const auto& ar) {
            for (u32 tile = 0; tile < (narrow ? ntiles : tiles); ++tile)
                run_group(lds, NT, [&](u32 tid) {
                    if (narrow)
                        narrow_fin<B>(ar, v.data(), &F, q, lv, L.log_n, tile, tid);
                    else
                        fwd_rows<B>(ar, v.data(), v.data(), lv, L.log_n, &F, q, tile, tid);
                });
        });
        for (u64 i = 0; i < n; ++i)
            if (out[i] != (mulm((a[i] + q - X[i]) % q, inv) + add[i]) % q) emu::die("finish differs", (double)i);
    }

    // the fused row pass + inner product + finish (two digits, the second given as it is)
    if (q >= FP_PRIME_BOUND) return;
    std::vector<u64> mid = x, own = random_limb(L, g), key, zb = random_limb(L, g), outb(n), outa(n);
    for (u32 j = 0; j < 4; ++j) {
        const auto k = random_limb(L, g);
        key.insert(key.end(), k.begin(), k.end());
    }
    const std::vector<u64> Z = oracle(L, zb, true);
    Arrays keep{&mid, &own, &key, &zb, &outb, &outa};
    cols<A>(L, lds, mid);
    cols<A>(L, lds, zb);
    RowIpFinJob J{};
    J.ip = {mid.data(), n, own.data(), key.data(), n, nullptr, nullptr, 2, 0, 1, 0};
    with(L, true, [&](const auto& ar) {
        if constexpr (std::decay_t<decltype(ar)>::F64) {
            const FTw iv{(double)inv, (double)inv / (double)q};
            for (u32 tile = 0; tile < tiles; ++tile)
                run_group(lds, NT, [&](u32) {
                    double sb[16], sa[16];
                    rows_ip_sums<B>(ar, J.ip, lv, L.log_n, tile, sb, sa);
                    finish_sum<B>(ar, sb, zb.data(), outb.data(), nullptr, iv, lv, L.log_n, tile);
                    finish_sum<B>(ar, sa, zb.data(), outa.data(), nullptr, iv, lv, L.log_n, tile);
                });
        }
    });
    for (u64 i = 0; i < n; ++i)
        for (u32 part = 0; part < 2; ++part) {
            const u64 s = (mulm(X[i], key[part * n + i]) + mulm(own[i], key[(2 + part) * n + i])) % q;
            if ((part ? outa : outb)[i] != mulm((s + q - Z[i]) % q, inv)) emu::die("fused inner product differs", (double)i);
        }
}

}  // namespace

int main(int argc, char** argv) {
    if (argc > 1) wave::size = (u32)std::atoi(argv[1]);
    std::mt19937_64 g(77);
    for (u32 log_n = 12; log_n <= 16; ++log_n)
        for (unsigned bits : {50u, 60u}) {
            u64 q = 0;
            if (or_ntt_primes_skip(bits, 1ull << log_n, 0, 1, &q) != 0) emu::die("no prime");
            const Limb L{log_n, q, build_ntt_tables({q}, log_n, true)};
            switch (log_n) {
                case 12: replay<6, 6>(L, g); break;
                case 13: replay<7, 6>(L, g); break;
                case 14: replay<7, 7>(L, g); break;
                case 15: replay<8, 7>(L, g); break;
                default: replay<8, 8>(L, g); break;
            }
            std::printf("N=2^%u, %u-bit prime: row exchanges inside one wave\n", log_n, bits);
            std::fflush(stdout);
        }
    std::printf("EMU OK\n");
    return 0;
}
