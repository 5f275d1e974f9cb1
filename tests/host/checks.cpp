// Checks of the runtime's own code on the host model of HIP (hip_model.h): one function per check,
// named on the command line. A failed check ends the program with a message.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <random>
#include <string>

#include "../../ckks-train_amd/csrc/evaluator.h"
#include "../../ckks-train_amd/csrc/hostmath.h"
#include "../../ckks-train_amd/csrc/server.h"
#include "hip_model.h"

using namespace ckh;

#define CHECK(x, ...)                                                      \
    do {                                                                   \
        if (!(x)) {                                                        \
            std::fprintf(stderr, "CHECK FAILED (%s:%d): %s ", __FILE__, __LINE__, #x); \
            std::fprintf(stderr, "" __VA_ARGS__);                          \
            std::fprintf(stderr, "\n");                                    \
            std::exit(1);                                                  \
        }                                                                  \
    } while (0)

// The largest primes = 1 mod 2N below 2^bits, each once.
static std::vector<u64> primes_of(u32 log_n, const std::vector<u32>& bits) {
    std::map<u32, u64> next;
    std::vector<u64> out;
    const u64 m = 2ull << log_n;
    for (u32 b : bits) {
        u64 q = next.count(b) ? next[b] - m : ((1ull << b) - 1) / m * m + 1;
        while (q >= (1ull << b) || !hm::is_prime(q)) q -= m;
        next[b] = q;
        out.push_back(q);
    }
    return out;
}

static std::shared_ptr<Context> make(u32 log_n, u32 nq, u32 np, u32 dnum, u32 streams = 2) {
    std::vector<u32> bits(nq, 50);
    bits.insert(bits.end(), np, 59);
    const std::vector<u64> p = primes_of(log_n, bits);
    ckh_params prm{};
    prm.log_n = log_n;
    prm.nq = nq;
    prm.np = np;
    prm.dnum = dnum;
    prm.q = p.data();
    prm.p = p.data() + nq;
    return std::make_shared<Context>(0, prm, streams);
}

// An upload whose kernel was not launched is an error, not a buffer of stale words.
static void upload_launch_checked() {
    auto c = make(12, 6, 2, 3);
    std::vector<u64> words(8192);
    BufPtr b = c->alloc(words.size());
    model::refuse_launch = true;
    bool failed = false;
    try {
        c->h2d(b->ptr, words.data(), words.size() * 8, c->stream());
    } catch (const Error& e) {
        failed = e.status == CKH_ERR_DEVICE;
    }
    CHECK(failed);
    c->h2d(b->ptr, words.data(), words.size() * 8, c->stream());  // and the next one works
}

// Uploads on the kernel's range of sizes go by the kernel whatever their last bytes, and arrive whole; so do the
// descriptors of batches of odd and even numbers of limbs.
static void uploads_of_every_length() {
    auto c = make(12, 6, 2, 3);
    hipStream_t s = c->stream();
    std::vector<u32> words(8192);
    for (size_t i = 0; i < words.size(); ++i) words[i] = (u32)i * 2654435761u;
    for (size_t bytes : {16388, 16392, 16396, 16400, 16404, 32760, 32764}) {
        BufPtr b = c->alloc(bytes / 8 + 1);
        model::uploads.clear();
        c->h2d(b->ptr, words.data(), bytes, s);
        CHECK(model::uploads.size() == 1 && model::uploads[0].kernel, "%zu bytes", bytes);
        CHECK(hipStreamSynchronize(s) == hipSuccess);
        CHECK(std::memcmp(b->ptr, words.data(), bytes) == 0, "%zu bytes", bytes);
    }
    KskPtr key = ksk_uniform(*c, 5, 0, 1);
    for (u32 count = 60; count < 64; ++count) {
        std::vector<PolyPtr> ps;
        std::vector<const Poly*> in;
        for (u32 i = 0; i < count; ++i) {
            ps.push_back(poly_uniform(*c, i % 3 ? 4 : 5, 0, true, i, 0));
            in.push_back(ps.back().get());
        }
        for (u32 pass = 0; pass < 3; ++pass) {
            model::uploads.clear();
            ks_switch_batch(*c, in, *key);
            CHECK(model::uploads.size() == 1);
            CHECK(model::uploads[0].bytes > 16384 && model::uploads[0].kernel, "%u switches: %zu bytes", count,
                  model::uploads[0].bytes);
        }
    }
}

// Key switches, hoisted rotations, products and rescales are put together at every ring size (undefined shifts of
// the rules end the program).
static void programs_at_every_ring_size() {
    for (u32 log_n = 2; log_n <= 17; ++log_n) {
        auto c = make(log_n, 4, 2, 2);
        const u64 g = galois_elt(c->n, 1);
        Evaluator ev(*c, ksk_uniform(*c, 3, 0, 1), {ksk_uniform(*c, 3, g, 2)});
        Ct a{{poly_uniform(*c, 3, 0, true, 3, 0), poly_uniform(*c, 3, 0, true, 4, 0)}, 1024.0};
        ks_switch(*c, *a.comps[0], *ev.relin);
        ev.rescale(*ev.mul(a, a));
        if (log_n > 2) ev.rotate(a, 1);
        ev.hoisted_rotate(a, {0, 1});
        c->synchronize_all();
    }
}

// Where no candidate is faster the autotuner keeps the present settings, and it times each kernel and grouping of a
// batch that converts apart once, and no grouping where none is used.
static void autotuner_keeps_what_is_not_beaten() {
    const char* keys[] = {"conv_variant", "conv_variant_md", "conv_tg", "fuse_ip", "conv_variant_small", "conv_tg_small",
                          "fuse_ip_small", "ntt_chunk_fwd", "ntt_chunk_inv"};
    auto c = make(12, 12, 6, 2);
    std::map<std::string, int64_t> before;
    for (const char* k : keys) before[k] = c->get_tuning(k);
    const std::string all = c->autotune();
    for (const char* k : keys) CHECK(c->get_tuning(k) == before[k], "%s", k);
    CHECK(all.find("conv1_") == std::string::npos);
    CHECK(all.find("_tg16") == std::string::npos, "%s", all.c_str());

    KskPtr key = ksk_uniform(*c, 11, 0, 1);
    std::vector<PolyPtr> ps;
    std::vector<const Poly*> batch;
    for (u32 i = 0; i < 900; ++i) {  // enough tiles for conversions of their own
        ps.push_back(poly_uniform(*c, 11, 0, true, i, 0));
        batch.push_back(ps.back().get());
    }
    c->set_tuning("conv_tg", 8);
    const std::string ks = c->autotune_ks(batch, *key);
    CHECK(c->get_tuning("conv_tg") == 8);
    CHECK(ks.find("conv0_tg16") != std::string::npos && ks.find("tg24") == std::string::npos, "%s", ks.c_str());
    c->set_tuning("conv_tg", 32);  // as many as 24 or 16 take here: all
    CHECK(c->autotune_ks(batch, *key).find("conv0_tg16") == std::string::npos);
    CHECK(c->get_tuning("conv_tg") == 32);
}

// Largest device memory that f holds beyond what was live before, its result included.
template <class F>
static u64 peak_of(Context& c, F&& f) {
    const u64 before = c.live_bytes;
    u64 peak = 0;
    model::on_launch = [&] { peak = std::max<u64>(peak, c.live_bytes - before); };
    f();
    model::on_launch = nullptr;
    c.synchronize_all();
    return peak;
}

// A product with encrypted diagonals stays within the memory it is admitted by (in the pool that does not round
// sizes, launched directly; 64 KB for the launches' descriptors).
static void encrypted_products_stay_within_their_estimate() {
    const u32 sets[][3] = {{6, 2, 3}, {12, 4, 3}, {24, 6, 4}, {20, 4, 5}};
    for (auto& s : sets) {
        auto c = make(12, s[0], s[1], s[2]);
        c->set_tuning("pool", 0);
        c->set_tuning("graphs", 0);
        std::map<u64, KskPtr> keys;
        for (u32 baby : {1u, 2u, 4u, 8u, 32u})
            for (u32 giant : {1u, 2u, 4u, 16u, 32u})
                for (u32 level : {s[0] - 1, s[0] / 2})
                    for (u32 every : {1u, 3u})
                        for (int32_t offset : {0, -1}) {
                            if (offset <= -(int32_t)(baby * giant)) continue;
                            std::vector<KskPtr> galois;
                            auto need = [&](int32_t step) {
                                const u64 g = galois_elt(c->n, step);
                                if (!keys.count(g)) keys[g] = ksk_uniform(*c, s[0] - 1, g, 7);
                                galois.push_back(keys[g]);
                            };
                            for (u32 k = 1; k < baby; ++k) need((int32_t)k);
                            for (u32 k = 0; k < giant; ++k) need(offset + (int32_t)(baby * k));
                            Evaluator ev(*c, ksk_uniform(*c, s[0] - 1, 0, 1), galois);
                            auto ct = [&] {
                                return Ct{{poly_uniform(*c, level, 0, true, 3, 0), poly_uniform(*c, level, 0, true, 4, 0)}, 1024.0};
                            };
                            const Ct x = ct(), w = ct();
                            std::vector<const Ct*> entries(baby * giant, nullptr);
                            for (u32 i = 0; i < baby * giant; i += every) entries[i] = &w;
                            CtPtr out;
                            const u64 peak = peak_of(*c, [&] { out = ev.matvec_enc(x, entries, baby, giant, 1, offset); });
                            const u64 room = ev.matvec_enc_workspace_bytes(level, baby, giant) + 65536;
                            CHECK(peak <= room, "%u primes, level %u, %u x %u, offset %d: %llu above %llu", s[0], level, baby,
                                  giant, offset, (unsigned long long)peak, (unsigned long long)room);
                        }
    }
}

// A served request is admitted by the memory it holds: never less (but for descriptors), and hoisted rotations,
// whose scratch has one form, by just that.
static void served_requests_are_admitted_by_what_they_hold() {
    auto c = make(12, 12, 4, 3);
    c->set_tuning("pool", 0);
    c->set_tuning("graphs", 0);
    std::vector<KskPtr> galois;
    std::vector<int32_t> steps;
    for (int32_t k = 1; k <= 5; ++k) {
        galois.push_back(ksk_uniform(*c, 11, galois_elt(c->n, k), 7));
        steps.push_back(k);
    }
    auto ev = std::make_shared<Evaluator>(*c, ksk_uniform(*c, 11, 0, 1), galois);
    for (u32 level : {11u, 6u, 1u})
        for (u32 kind : {CKH_OP_RELINEARIZE, CKH_OP_HOISTED_ROTATE, CKH_OP_MUL_RELIN_RESCALE}) {
            auto ct = [&](u32 comps) {
                auto r = std::make_shared<Ct>();
                for (u32 i = 0; i < comps; ++i) r->comps.push_back(poly_uniform(*c, level, 0, true, i, 0));
                r->scale = 1024.0;
                return r;
            };
            auto op = std::make_shared<ServedOp>();
            op->kind = kind;
            op->ev = ev;
            op->a = ct(kind == CKH_OP_RELINEARIZE ? 3 : 2);
            op->b = kind == CKH_OP_MUL_RELIN_RESCALE ? ct(2) : nullptr;
            if (kind == CKH_OP_HOISTED_ROTATE) op->steps = steps;
            c->synchronize_all();
            u64 held = 0;
            ckh_server_stats st{};
            {
                ckh_server_config cfg{};
                cfg.hbm_budget_bytes = 1ull << 40;
                Server srv(cfg);
                held = peak_of(*c, [&] {
                    const u64 ticket = srv.submit(op);
                    OpPtr done;
                    while (!srv.poll(ticket, false, done)) c->synchronize_all();
                    CHECK(done->status == CKH_OK, "%s", done->err.c_str());
                });
                st = srv.stats();
            }
            CHECK(st.peak_bytes + 65536 >= held, "kind %u: %llu held", kind, (unsigned long long)held);
            if (kind == CKH_OP_HOISTED_ROTATE)
                CHECK(st.peak_bytes <= held, "%llu counted, %llu held", (unsigned long long)st.peak_bytes, (unsigned long long)held);
        }
}

// The allocation-failure hook counts what a call allocates in polynomials' worths (nq limbs, a smaller buffer one):
// armed within that count every call fails, and is disarmed; armed after it the call succeeds.
static void allocation_hook_counts_by_size() {
    auto c = make(12, 6, 2, 3);
    c->set_tuning("pool", 0);
    c->set_tuning("graphs", 0);
    std::vector<KskPtr> galois;
    for (int32_t k : {1, 2, 3, 4}) galois.push_back(ksk_uniform(*c, 5, galois_elt(c->n, k), 7));
    Evaluator ev(*c, ksk_uniform(*c, 5, 0, 1), galois);
    Ct a, d;
    for (u32 i = 0; i < 3; ++i) d.comps.push_back(poly_uniform(*c, 5, 0, true, i, 0));
    a.comps = {d.comps[0], d.comps[1]};
    a.scale = d.scale = 1024.0;
    const std::vector<const Ct*> three(3, &d), entries(8, &a);
    const std::function<void()> calls[] = {
        [&] { ks_switch(*c, *a.comps[0], *ev.relin); },
        [&] { ev.relinearize_batch(three); },
        [&] { ev.hoisted_rotate(a, {1, 2, 3}); },
        [&] { ev.hoisted_rotate_batch({{&a, {1, 2}}, {&a, {3}}}); },
        [&] { ev.rotate_batch({{&a, 1}, {&a, 4}}); },
        [&] { ev.rescale(*ev.mul(a, a)); },
        [&] { ev.matvec_enc(a, entries, 4, 2, 1, 0); },
    };
    const u64 unit = 6 * c->n * 8;
    for (auto& call : calls) {
        u64 total = 0;
        model::on_malloc = [&](size_t bytes) { total += std::max<u64>(1, (bytes + unit - 1) / unit); };
        call();
        model::on_malloc = nullptr;
        for (u64 at = 0; at <= total; ++at) {
            c->fail_alloc_after = (int64_t)at;
            bool failed = false;
            try {
                call();
            } catch (const Error& e) {
                failed = e.status == CKH_ERR_DEVICE;
                CHECK(c->fail_alloc_after == -1);
            }
            CHECK(failed == (at < total), "call %zu at %llu of %llu", (size_t)(&call - calls), (unsigned long long)at,
                  (unsigned long long)total);
            c->fail_alloc_after = -1;
        }
    }
}

// A tuning changed by another thread between the sizing of a switch's scratch and its program does not change the
// program's form: the one sized for (here without room for the sums) is the one that runs.
static void a_switch_keeps_the_route_it_was_sized_for() {
    auto c = make(12, 6, 2, 3);
    c->set_tuning("graphs", 0);
    KskPtr key = ksk_uniform(*c, 5, 0, 1);
    PolyPtr d = poly_uniform(*c, 5, 0, true, 2, 0);
    for (u32 which = 0; which < 2; ++which) {
        model::ip_launches = model::ip_finish_launches = 0;
        u32 at = 0;
        model::on_malloc = [&](size_t) {  // the outputs, then the scratch
            if (++at == 2) (which ? c->conv_yform : c->conv_cols) = 0;
        };
        ks_switch(*c, *d, *key);
        model::on_malloc = nullptr;
        CHECK(c->conv_cols == 0 || c->conv_yform == 0);
        CHECK(model::ip_finish_launches == 1 && model::ip_launches == 0);
        c->conv_cols = 1;
        c->conv_yform = 7;
        c->trim_pool(0);  // the next switch allocates again
    }
}

// Memory written by copies still queued on one stream goes to no other stream's buffer, at random steps of both
// streams; with `capture`, while a caller captures the first stream from time to time.
static void cached_blocks(bool capture) {
    auto c = make(12, 6, 2, 3, 2);
    std::mt19937 g(5);
    hipStream_t s[2];
    for (u32 i = 0; i < 2; ++i) {
        c->set_stream(i);
        s[i] = c->stream();
    }
    const size_t words = 4096;
    std::vector<u64> src[2] = {std::vector<u64>(words, 1), std::vector<u64>(words, 2)};
    u64 reused = 0;
    bool capturing = false;
    std::map<u64*, u32> last;  // the stream that used a block last
    struct Held {
        BufPtr b;
        u32 stream;
    };
    std::vector<Held> held;
    for (u32 round = 0; round < 20000; ++round) {
        if (capture && g() % 16 == 0) model::set_capturing(s[0], capturing = !capturing);
        const u32 i = capturing ? 1 : g() % 2;
        c->set_stream(i);
        if (held.size() == 12 || g() % 2) {  // a release, on the stream that used the buffer
            for (size_t k = 0; k < held.size(); ++k)
                if (held[k].stream == i) {
                    held.erase(held.begin() + k);
                    break;
                }
        } else {
            BufPtr b = c->alloc(words);
            auto it = last.find(b->ptr);
            if (it != last.end() && it->second != i) {
                // the copies that the other stream queued on this block have all run
                ++reused;
                CHECK(b->ptr[0] == it->second + 1 && b->ptr[words - 1] == it->second + 1, "round %u", round);
            }
            if (it == last.end() || it->second != i) std::memset(b->ptr, 0xff, words * 8);
            last[b->ptr] = i;
            model::queue_copy(b->ptr, src[i].data(), words * 8, s[i]);
            held.push_back({b, i});
        }
        for (u32 k = g() % 3; k > 0; --k) model::step(s[g() % 2]);
        if (g() % 64 == 0) {
            while (model::step(s[0])) {}
            while (model::step(s[1])) {}
        }
    }
    if (capturing) model::set_capturing(s[0], false);
    CHECK(reused > 100, "%llu", (unsigned long long)reused);
    CHECK(model::records_while_capturing == 0);
    c->synchronize_all();
}
static void cached_blocks_change_streams_after_their_use() { cached_blocks(false); }
static void cached_blocks_under_a_capture() { cached_blocks(true); }

// Another stream's blocks are taken as soon as that stream is idle, or has passed the frees of earlier batches
// while a later one still runs: no block comes from the driver.
static void blocks_of_finished_work_are_taken() {
    auto c = make(12, 6, 2, 3, 2);
    hipStream_t s[2];
    for (u32 i = 0; i < 2; ++i) {
        c->set_stream(i);
        s[i] = c->stream();
        c->alloc(16);  // both streams allocate
    }
    std::vector<u64> src(4096);
    auto use_and_free = [&](u32 stream, u32 blocks) {
        c->set_stream(stream);
        std::vector<BufPtr> b;
        for (u32 k = 0; k < blocks; ++k) {
            b.push_back(c->alloc(src.size()));
            model::queue_copy(b.back()->ptr, src.data(), src.size() * 8, s[stream]);
        }
    };
    use_and_free(0, 4);
    while (model::step(s[0])) {}
    uint64_t before = c->stat_mallocs;
    use_and_free(1, 4);  // stream 0 is idle
    CHECK(c->stat_mallocs == before);
    while (model::step(s[1])) {}

    std::vector<size_t> queued;  // after each batch of 24 blocks
    for (u32 batch = 0; batch < 3; ++batch) {
        c->set_stream(0);
        std::vector<BufPtr> b;
        for (u32 k = 0; k < 24; ++k) b.push_back(c->alloc(src.size() << batch));  // a class of its own each
        for (auto& x : b) model::queue_copy(x->ptr, src.data(), src.size() * 8, s[0]);
        b.clear();
        queued.push_back(model::pending(s[0]));
    }
    const size_t left = queued[2] - queued[1];  // the third batch still to run
    while (model::pending(s[0]) > left) model::step(s[0]);
    before = c->stat_mallocs;
    for (u32 batch = 0; batch < 2; ++batch) {
        c->set_stream(1);
        std::vector<BufPtr> b;
        for (u32 k = 0; k < 16; ++k) b.push_back(c->alloc(src.size() << batch));
    }
    CHECK(c->stat_mallocs == before, "%llu", (unsigned long long)(c->stat_mallocs - before));
    c->synchronize_all();
}

// Staged uploads of two streams arrive whole over many laps of the ring, at random steps of both streams; with
// `capture`, while a caller captures the first stream from time to time.
static void staged_uploads(bool capture) {
    auto c = make(12, 6, 2, 3, 2);
    std::mt19937 g(6);
    hipStream_t s[2];
    for (u32 i = 0; i < 2; ++i) {
        c->set_stream(i);
        s[i] = c->stream();
    }
    struct Sent {
        BufPtr b;
        size_t words;
        u64 tag;
        u32 stream;
    };
    std::vector<Sent> sent;
    bool capturing = false;
    auto verify = [&] {
        for (u32 i = 0; i < 2; ++i) CHECK(hipStreamSynchronize(s[i]) == hipSuccess);
        for (const Sent& x : sent)
            for (size_t w = 0; w < x.words; ++w) CHECK(x.b->ptr[w] == x.tag + w, "word %zu of upload %llu", w, (unsigned long long)x.tag);
        sent.clear();
    };
    size_t total = 0;
    for (u32 round = 0; total < ((size_t)400 << 20); ++round) {
        if (capture && g() % 24 == 0) model::set_capturing(s[0], capturing = !capturing);
        const u32 i = capturing ? 1 : g() % 2;
        c->set_stream(i);
        const size_t words = g() % 8 == 0 ? 1 + g() % 700000 : 1 + g() % 20000;
        std::vector<u64> src(words);
        const u64 tag = (u64)round << 32;
        for (size_t w = 0; w < words; ++w) src[w] = tag + w;
        BufPtr b = c->alloc(words);
        c->h2d(b->ptr, src.data(), words * 8, s[i]);
        total += words * 8;
        sent.push_back({b, words, tag, i});
        for (u32 k = g() % 3; k > 0; --k) model::step(s[g() % 2]);
        if (!capturing && g() % 200 == 0) verify();
    }
    if (capturing) model::set_capturing(s[0], false);
    verify();
    CHECK(model::records_while_capturing == 0);
}
static void staged_uploads_of_two_streams() { staged_uploads(false); }
static void staged_uploads_under_a_capture() { staged_uploads(true); }

// A plan evicted while a caller captures its stream leaves nothing in that capture, and goes once it has ended.
static void plans_evicted_under_a_capture() {
    auto c = make(12, 6, 2, 3, 2);
    c->set_tuning("graph_cache", 1);
    KskPtr key = ksk_uniform(*c, 5, 0, 1);
    std::vector<PolyPtr> ps;
    std::vector<const Poly*> in;
    for (u32 i = 0; i < 4; ++i) {
        ps.push_back(poly_uniform(*c, 5, 0, true, i, 0));
        in.push_back(ps.back().get());
    }
    c->set_stream(0);
    hipStream_t s0 = c->stream();
    for (u32 k = 0; k < 3; ++k) ks_switch_batch(*c, in, *key);  // seen, captured, replayed
    CHECK(c->graph_launches == 2);
    const uint64_t queued = model::pending(s0);
    model::set_capturing(s0, true);
    c->set_stream(1);
    for (u32 k = 0; k < 3; ++k) ks_switch_batch(*c, in, *key);
    CHECK(c->graph_launches == 4);
    CHECK(model::records_while_capturing == 0 && model::pending(s0) == queued);
    CHECK(model::destroyed_graphs == 0);
    model::set_capturing(s0, false);
    for (u32 k = 0; k < 3; ++k) {  // swept once its stream has finished
        c->synchronize_all();
        ks_switch_batch(*c, in, *key);
    }
    CHECK(model::destroyed_graphs == 1);
    c->set_stream(0);
}

int main(int argc, char** argv) {
    const std::map<std::string, void (*)()> checks = {
        {"upload_launch_checked", upload_launch_checked},
        {"uploads_of_every_length", uploads_of_every_length},
        {"programs_at_every_ring_size", programs_at_every_ring_size},
        {"autotuner_keeps_what_is_not_beaten", autotuner_keeps_what_is_not_beaten},
        {"encrypted_products_stay_within_their_estimate", encrypted_products_stay_within_their_estimate},
        {"served_requests_are_admitted_by_what_they_hold", served_requests_are_admitted_by_what_they_hold},
        {"allocation_hook_counts_by_size", allocation_hook_counts_by_size},
        {"a_switch_keeps_the_route_it_was_sized_for", a_switch_keeps_the_route_it_was_sized_for},
        {"cached_blocks_change_streams_after_their_use", cached_blocks_change_streams_after_their_use},
        {"cached_blocks_under_a_capture", cached_blocks_under_a_capture},
        {"blocks_of_finished_work_are_taken", blocks_of_finished_work_are_taken},
        {"staged_uploads_of_two_streams", staged_uploads_of_two_streams},
        {"staged_uploads_under_a_capture", staged_uploads_under_a_capture},
        {"plans_evicted_under_a_capture", plans_evicted_under_a_capture},
    };
    auto it = argc == 2 ? checks.find(argv[1]) : checks.end();
    if (it == checks.end()) {
        std::fprintf(stderr, "no such check\n");
        return 2;
    }
    it->second();
    std::printf("ok\n");
    return 0;
}
