// Key-switch inner product, pointwise arithmetic, NTT-form automorphism and the seeded
// input generator, for gfx950.
#include <algorithm>

#include "ops.h"

namespace ckh {

// Elementwise kernels take two words of a limb per thread, in one 16-byte load each (limbs are
// 16-byte aligned: a multiple of N >= 2 words from a block's start). Bound by memory: the sixteen
// rotations' gathers at N = 2^16 51 -> 45 us, the block sums of the 32 x 32 product at 2^15 270 ->
// 237 us (with each diagonal read once for both components).
typedef u64 u64x2 __attribute__((ext_vector_type(2)));
static dim3 pairs_grid(u32 log_n, u32 rows) { return dim3((((1u << log_n) / 2) + 255) / 256, rows); }
CKH_DEV auto glb2(const u64* p) { return glb((const u64x2*)p); }
CKH_DEV auto glb2(u64* p) { return glb((u64x2*)p); }

// Words 2 c and 2 c + 1 of sigma_g(in): the lowest index bit is the highest of the bit-reversed one,
// where adding N (times the odd g) flips the highest bit of the result only, so perm(2 c + 1) =
// perm(2 c) ^ 1 and a pair comes from a pair, as it is or exchanged.
CKH_DEV u64x2 galois_pair(const u64* in, u32 c, u64 g, u32 log_n) {
    const u32 s = galois_index(2 * c, g, log_n);
    const u64x2 v = glb2(in)[s >> 1];
    return (s & 1) ? u64x2{v[1], v[0]} : v;
}

// The key inner product (ip_arith.h: ip_words), two coefficients per thread. NT_KEY: non-temporal key
// loads, for launches whose every key word is read once (rotations, each under its own key): the
// digits, which all of them read, then stay in the caches. Bound by memory: sixteen hoisted rotations
// at N = 2^16 (19 limbs) 432 -> 381 us, 5.6 TB/s; 410 us without the non-temporal loads, which a key
// shared by 256 switches does not want (1,041 against 892 us).
template <bool NT_KEY>
struct IpPair {
    static constexpr u32 W = 2;
    CKH_DEV static void put(u64x2 v, u64 (&w)[2]) {
        w[0] = v[0];
        w[1] = v[1];
    }
    CKH_DEV static void load(const u64* p, u64 c, u64 (&w)[2]) { put(glb2(p)[c], w); }
    CKH_DEV static void load_key(const u64* p, u64 c, u64 (&w)[2]) {
        if constexpr (NT_KEY)
            put(__builtin_nontemporal_load(glb2(p) + c), w);
        else
            put(glb2(p)[c], w);
    }
    CKH_DEV static void store(u64* p, u64 c, const u64 (&w)[2]) { glb2(p)[c] = u64x2{w[0], w[1]}; }
    CKH_DEV static void gather(const u64* p, u64 c, u64 g, u32 log_n, u64 (&w)[2]) { put(galois_pair(p, (u32)c, g, log_n), w); }
};

template <class Mem>
__global__ __launch_bounds__(256) void k_inner_product(const IpJob* __restrict__ jobs,
                                                       const PrimeConst* __restrict__ pc, u32 log_n) {
    const u32 c = blockIdx.x * 256 + threadIdx.x;
    if (c >= (1u << log_n) / Mem::W) return;
    const IpJob J = jobs[blockIdx.y];
    ip_words<Mem>(J, pc[J.prime], log_n, c);
}

// Below IP_PAIR_BLOCKS workgroups of pairs (4 per CU) a thread takes one coefficient: a launch that
// does not fill the device is bound by latency (one switch at N = 2^12 61.6 against 63.1 us).
constexpr u64 IP_PAIR_BLOCKS = 1024;

void inner_product_launch(const IpJob* jobs, u32 njobs, const PrimeConst* pc, u32 log_n, bool keys_once,
                          hipStream_t stream) {
    if (njobs == 0) return;
    const dim3 pairs = pairs_grid(log_n, njobs);
    if ((u64)pairs.x * pairs.y < IP_PAIR_BLOCKS)
        hipLaunchKernelGGL(k_inner_product<IpWord>, dim3(((1u << log_n) + 255) / 256, njobs), dim3(256), 0, stream, jobs,
                           pc, log_n);
    else if (keys_once)
        hipLaunchKernelGGL(k_inner_product<IpPair<true>>, pairs, dim3(256), 0, stream, jobs, pc, log_n);
    else
        hipLaunchKernelGGL(k_inner_product<IpPair<false>>, pairs, dim3(256), 0, stream, jobs, pc, log_n);
}

__global__ __launch_bounds__(256) void k_copy(const LimbRef* __restrict__ refs, u32 log_n) {
    const u32 c = blockIdx.x * 256 + threadIdx.x;
    if (c >= (1u << log_n) / 2) return;
    const LimbRef r = refs[blockIdx.y];
    glb2(r.dst)[c] = glb2(r.src)[c];
}

void copy_launch(const LimbRef* refs, u32 nrefs, u32 log_n, hipStream_t stream) {
    if (nrefs == 0) return;
    hipLaunchKernelGGL(k_copy, pairs_grid(log_n, nrefs), dim3(256), 0, stream, refs, log_n);
}

// Staged descriptor bytes to the device, 16 per thread and the rest a word per thread (descriptors are of 8
// bytes modulo 16: a program of an odd number of them ends so), read from pinned host memory. A copy command of
// more than 16 KB goes to a DMA engine instead: 19 us of the host, 6 us of copying and a switch of queues on
// either side; the workgroups here read over the bus together.
__global__ __launch_bounds__(256) void k_upload(const uint4* __restrict__ in, uint4* __restrict__ out, u32 n16, u32 words) {
    const u32 i = blockIdx.x * 256 + threadIdx.x;
    if (i < n16)
        out[i] = in[i];
    else if (i - n16 < words)
        ((u32*)(out + n16))[i - n16] = ((const u32*)(in + n16))[i - n16];
}

hipError_t upload_launch(const void* pinned, void* out, u64 bytes, hipStream_t stream) {
    const uint4* in = (const uint4*)pinned;
    uint4* to = (uint4*)out;
    u32 n16 = (u32)(bytes / 16), words = (u32)(bytes % 16 / 4);
    if (n16 + words == 0) return hipSuccess;
    void* args[] = {&in, &to, &n16, &words};
    return hipLaunchKernel((const void*)k_upload, dim3((n16 + words + 255) / 256), dim3(256), args, 0, stream);
}

// Streaming copy of n16 16-byte words (a measurement of the HBM copy rate a kernel reaches).
__global__ __launch_bounds__(256) void k_stream_copy(const uint4* __restrict__ in, uint4* __restrict__ out, u64 n16) {
    const u64 stride = (u64)gridDim.x * 256;
    for (u64 i = (u64)blockIdx.x * 256 + threadIdx.x; i < n16; i += stride) out[i] = in[i];
}

void stream_copy_launch(const void* in, void* out, u64 bytes, hipStream_t stream) {
    const u64 n16 = bytes / 16;
    const u32 blocks = (u32)std::min<u64>((n16 + 255) / 256, 16384);
    if (blocks) hipLaunchKernelGGL(k_stream_copy, dim3(blocks), dim3(256), 0, stream, (const uint4*)in, (uint4*)out, n16);
}

// a * b mod q for reduced a, b: one f64 modular product below 2^50 (about 12 operations instead of
// the 128-bit reduction's 55).
CKH_DEV u64 mul_any(u64 a, u64 b, const PrimeConst& C) {
    if (C.q >= FP_PRIME_BOUND) return mul_mod(a, b, C);
    const double w = u2d(b);
    return d2u(fcanon(fmulmod(u2d(a), w, w * C.qinv, C.qf), C.qf, C.qinv));
}

__global__ __launch_bounds__(256) void k_pointwise(u32 op, const u64* __restrict__ a, const u64* __restrict__ b,
                                                   u64* __restrict__ out, u32 prime0,
                                                   const PrimeConst* __restrict__ pc, u32 log_n) {
    const u32 half = (1u << log_n) / 2;
    const u32 c = blockIdx.x * 256 + threadIdx.x;
    if (c >= half) return;
    const u64 i = (u64)blockIdx.y * half + c;
    const PrimeConst C = pc[prime0 + blockIdx.y];
    const u64x2 x = glb2(a)[i];
    u64x2 y = {0, 0}, v;
    if (op == PW_ADD || op == PW_SUB || op == PW_MUL) y = glb2(b)[i];
#pragma unroll
    for (u32 k = 0; k < 2; ++k) switch (op) {
            case PW_ADD: v[k] = add_mod(x[k], y[k], C.q); break;
            case PW_SUB: v[k] = sub_mod(x[k], y[k], C.q); break;
            case PW_NEG: v[k] = sub_mod(0, x[k], C.q); break;
            case PW_MUL: v[k] = mul_any(x[k], y[k], C); break;
            default: v[k] = x[k]; break;
        }
    glb2(out)[i] = v;
}

void pointwise_launch(PwOp op, const u64* a, const u64* b, u64* out, u32 limbs, u32 prime0, const PrimeConst* pc,
                      u32 log_n, hipStream_t stream) {
    if (limbs == 0) return;
    hipLaunchKernelGGL(k_pointwise, pairs_grid(log_n, limbs), dim3(256), 0, stream, (u32)op, a, b, out, prime0, pc,
                       log_n);
}

// Sums of products of reduced words mod one prime, two words side by side: f64 modular products
// below 2^50 (each below 0.7 q in magnitude; reduced before more than 6 could add up), exact 128-bit
// sums above (folded into a residue before 128 terms).
struct FpSum {
    double s[2] = {0.0, 0.0};
    CKH_DEV void add(u64x2 x, u64x2 w, const PrimeConst& C) {
#pragma unroll
        for (u32 k = 0; k < 2; ++k) {
            const double wd = u2d(w[k]);
            s[k] += fmulmod(u2d(x[k]), wd, wd * C.qinv, C.qf);
        }
    }
    CKH_DEV void fold(const PrimeConst& C) {
#pragma unroll
        for (u32 k = 0; k < 2; ++k) s[k] = freduce(s[k], C.qf, C.qinv);
    }
    CKH_DEV u64x2 get(const PrimeConst& C) const {
        return u64x2{d2u(fcanon(s[0], C.qf, C.qinv)), d2u(fcanon(s[1], C.qf, C.qinv))};
    }
    static constexpr u32 FOLD = 2;  // terms between folds: a tensor's middle component has two products each
};
struct IntSum {
    Dot60 d[2];
    u64 r[2] = {0, 0};
    CKH_DEV void add(u64x2 x, u64x2 w, const PrimeConst&) {
#pragma unroll
        for (u32 k = 0; k < 2; ++k) d[k].add(x[k], w[k]);
    }
    CKH_DEV void fold(const PrimeConst& C) {
#pragma unroll
        for (u32 k = 0; k < 2; ++k) {
            u64 hi, lo;
            d[k].get(hi, lo);
            r[k] = add_mod(r[k], reduce128(hi, lo, C), C.q);
            d[k] = Dot60{};
        }
    }
    CKH_DEV u64x2 get(const PrimeConst& C) {
        fold(C);
        return u64x2{r[0], r[1]};
    }
    static constexpr u32 FOLD = 64;
};

// sum of x_t w_t for both components of x: the diagonal's word is read once for the two.
template <class S>
CKH_DEV void mul_sum_words(const MulSumJob& J, const MulSumTerm* terms, const PrimeConst& C, u32 c) {
    S a, b;
    for (u32 t = 0; t < J.count; ++t) {
        const auto* T = cst(terms + J.first + t);
        const u64x2 w = glb2(T->w)[c];
        a.add(glb2(T->x0)[c], w, C);
        b.add(glb2(T->x1)[c], w, C);
        if (t % S::FOLD == S::FOLD - 1) {
            a.fold(C);
            b.fold(C);
        }
    }
    glb2(J.out0)[c] = a.get(C);
    glb2(J.out1)[c] = b.get(C);
}

__global__ __launch_bounds__(256) void k_mul_sum(const MulSumJob* __restrict__ jobs,
                                                 const MulSumTerm* __restrict__ terms,
                                                 const PrimeConst* __restrict__ pc, u32 log_n) {
    const u32 c = blockIdx.x * 256 + threadIdx.x;
    if (c >= (1u << log_n) / 2) return;
    const MulSumJob J = jobs[blockIdx.y];
    const PrimeConst C = pc[J.prime];
    if (C.q < FP_PRIME_BOUND)
        mul_sum_words<FpSum>(J, terms, C, c);
    else
        mul_sum_words<IntSum>(J, terms, C, c);
}

void mul_sum_launch(const MulSumJob* jobs, const MulSumTerm* terms, u32 njobs, const PrimeConst* pc, u32 log_n,
                    hipStream_t stream) {
    if (njobs == 0) return;
    hipLaunchKernelGGL(k_mul_sum, pairs_grid(log_n, njobs), dim3(256), 0, stream, jobs, terms, pc, log_n);
}

// The tensor product (x0 + x1 s)(y0 + y1 s) of two words' pairs added to the three sums.
template <class S>
CKH_DEV void tensor_add(S& d0, S& d1, S& d2, u64x2 x0, u64x2 x1, u64x2 y0, u64x2 y1,
                        const PrimeConst& C) {
    d0.add(x0, y0, C);
    d1.add(x0, y1, C);
    d1.add(x1, y0, C);
    d2.add(x1, y1, C);
}

template <class S>
CKH_DEV void tensor_sum_words(const TensorJob& J, const TensorTerm* terms, const PrimeConst& C, u32 c) {
    S d0, d1, d2;
    for (u32 t = 0; t < J.count; ++t) {
        const auto* T = cst(terms + J.first + t);
        tensor_add(d0, d1, d2, glb2(T->x0)[c], glb2(T->x1)[c], glb2(T->y0)[c], glb2(T->y1)[c], C);
        if (t % S::FOLD == S::FOLD - 1) {
            d0.fold(C);
            d1.fold(C);
            d2.fold(C);
        }
    }
    glb2(J.out0)[c] = d0.get(C);
    glb2(J.out1)[c] = d1.get(C);
    glb2(J.out2)[c] = d2.get(C);
}

__global__ __launch_bounds__(256) void k_tensor_sum(const TensorJob* __restrict__ jobs,
                                                    const TensorTerm* __restrict__ terms,
                                                    const PrimeConst* __restrict__ pc, u32 log_n) {
    const u32 c = blockIdx.x * 256 + threadIdx.x;
    if (c >= (1u << log_n) / 2) return;
    const TensorJob J = jobs[blockIdx.y];
    const PrimeConst C = pc[J.prime];
    if (C.q < FP_PRIME_BOUND)
        tensor_sum_words<FpSum>(J, terms, C, c);
    else
        tensor_sum_words<IntSum>(J, terms, C, c);
}

void tensor_sum_launch(const TensorJob* jobs, const TensorTerm* terms, u32 njobs, const PrimeConst* pc, u32 log_n,
                       hipStream_t stream) {
    if (njobs == 0) return;
    hipLaunchKernelGGL(k_tensor_sum, pairs_grid(log_n, njobs), dim3(256), 0, stream, jobs, terms, pc, log_n);
}

// One tensor product of whole polynomials, the pointers in the launch itself (no descriptors).
template <class S>
CKH_DEV void tensor_words(const TensorTerm& T, u64* out, u32 limbs, const PrimeConst& C, u64 i, u64 half) {
    S d0, d1, d2;
    tensor_add(d0, d1, d2, glb2(T.x0)[i], glb2(T.x1)[i], glb2(T.y0)[i], glb2(T.y1)[i], C);
    const auto o = glb2(out);
    o[i] = d0.get(C);
    o[limbs * half + i] = d1.get(C);
    o[2 * limbs * half + i] = d2.get(C);
}

__global__ __launch_bounds__(256) void k_tensor(TensorTerm T, u64* out, u32 limbs, const PrimeConst* __restrict__ pc,
                                                u32 log_n) {
    const u32 half = (1u << log_n) / 2;
    const u32 c = blockIdx.x * 256 + threadIdx.x;
    if (c >= half) return;
    const PrimeConst C = pc[blockIdx.y];
    const u64 i = (u64)blockIdx.y * half + c;
    if (C.q < FP_PRIME_BOUND)
        tensor_words<FpSum>(T, out, limbs, C, i, half);
    else
        tensor_words<IntSum>(T, out, limbs, C, i, half);
}

void tensor_launch(const TensorTerm& t, u64* out, u32 limbs, const PrimeConst* pc, u32 log_n, hipStream_t stream) {
    if (limbs == 0) return;
    hipLaunchKernelGGL(k_tensor, pairs_grid(log_n, limbs), dim3(256), 0, stream, t, out, limbs, pc, log_n);
}

__global__ __launch_bounds__(256) void k_add_sum(const AddSumJob* __restrict__ jobs, const u64* const* __restrict__ xs,
                                                 const PrimeConst* __restrict__ pc, u32 log_n) {
    const u32 c = blockIdx.x * 256 + threadIdx.x;
    if (c >= (1u << log_n) / 2) return;
    const AddSumJob J = jobs[blockIdx.y];
    const u64 q = pc[J.prime].q;
    u64x2 acc = {0, 0};
    for (u32 t = 0; t < J.count; ++t) {
        const u64x2 x = glb2(xs[J.first + t])[c];
        acc = u64x2{add_mod(acc[0], x[0], q), add_mod(acc[1], x[1], q)};
    }
    glb2(J.out)[c] = acc;
}

void add_sum_launch(const AddSumJob* jobs, const u64* const* xs, u32 njobs, const PrimeConst* pc, u32 log_n,
                    hipStream_t stream) {
    if (njobs == 0) return;
    hipLaunchKernelGGL(k_add_sum, pairs_grid(log_n, njobs), dim3(256), 0, stream, jobs, xs, pc, log_n);
}

__global__ __launch_bounds__(256) void k_scalar_mul(const u64* __restrict__ a, u64* __restrict__ out,
                                                    const u64* __restrict__ consts, u32 neg,
                                                    const PrimeConst* __restrict__ pc, u32 log_n) {
    const u32 n = 1u << log_n;
    const u32 c = blockIdx.x * 256 + threadIdx.x;
    if (c >= n) return;
    const u64 i = (u64)blockIdx.y * n + c;
    const u64 q = pc[blockIdx.y].q, w = consts[2 * blockIdx.y], ws = consts[2 * blockIdx.y + 1];
    u64 v = shoup(a[i], w, ws, q);
    if (neg) v = sub_mod(0, v, q);
    out[i] = v;
}

void scalar_mul_launch(const u64* a, u64* out, u32 limbs, const u64* consts, bool neg, const PrimeConst* pc,
                       u32 log_n, hipStream_t stream) {
    if (limbs == 0) return;
    const u32 n = 1u << log_n;
    hipLaunchKernelGGL(k_scalar_mul, dim3((n + 255) / 256, limbs), dim3(256), 0, stream, a, out, consts, (u32)neg, pc,
                       log_n);
}

__global__ __launch_bounds__(256) void k_automorphism_ntt(const u64* __restrict__ in, u64* __restrict__ out, u64 g,
                                                          u32 log_n) {
    const u32 c = blockIdx.x * 256 + threadIdx.x;
    if (c >= (1u << log_n) / 2) return;
    const u64 base = (u64)blockIdx.y << log_n;
    glb2(out + base)[c] = galois_pair(in + base, c, g, log_n);
}

void automorphism_ntt_launch(const u64* in, u64* out, u32 limbs, u64 g, u32 log_n, hipStream_t stream) {
    if (limbs == 0) return;
    hipLaunchKernelGGL(k_automorphism_ntt, pairs_grid(log_n, limbs), dim3(256), 0, stream, in, out, g, log_n);
}

// Coefficient form (crates/ckks-train-core/src/poly.rs:255-276): coefficient i moves to
// e = i g mod 2N, negated mod its prime when e >= N (X^N = -1). Written as a gather so every
// output word is stored once, coalesced: output j takes input i = j g^-1 mod 2N (g is odd, so
// invertible mod 2N), as it is when i < N and negated from i - N otherwise, since (i - N) g =
// j - N g = j + N mod 2N for odd g. Limb r of the layout is Q prime r for r <= level, else P prime
// nq + r - level - 1.
__global__ __launch_bounds__(256) void k_automorphism_coeff(const u64* __restrict__ in, u64* __restrict__ out,
                                                            u64 g_inv, u32 level, u32 nq,
                                                            const PrimeConst* __restrict__ pc, u32 log_n) {
    const u32 n = 1u << log_n;
    const u32 j = blockIdx.x * 256 + threadIdx.x;
    if (j >= n) return;
    const u32 r = blockIdx.y;
    const u64 q = pc[r <= level ? r : nq + r - level - 1].q;
    const u64 base = (u64)r * n;
    const u32 i = (u32)((j * g_inv) & (2 * (u64)n - 1));
    if (i < n) {
        out[base + j] = in[base + i];
    } else {
        const u64 c = in[base + i - n];
        out[base + j] = c == 0 ? 0 : q - c;
    }
}

void automorphism_coeff_launch(const u64* in, u64* out, u32 limbs, u32 level, u32 nq, u64 g, const PrimeConst* pc,
                               u32 log_n, hipStream_t stream) {
    if (limbs == 0) return;
    const u64 two_n = 2ull << log_n;
    u64 g_inv = 1;  // g^(2N/2 - 1) = g^-1 in the unit group mod 2N (order dividing N)
    for (u64 e = (two_n >> 1) - 1, b = g % two_n; e; e >>= 1, b = b * b % two_n)
        if (e & 1) g_inv = g_inv * b % two_n;
    const u32 n = 1u << log_n;
    hipLaunchKernelGGL(k_automorphism_coeff, dim3((n + 255) / 256, limbs), dim3(256), 0, stream, in, out, g_inv, level,
                       nq, pc, log_n);
}

__global__ __launch_bounds__(256) void k_automorphism_batch(const AutJob* __restrict__ jobs, u32 log_n) {
    const u32 c = blockIdx.x * 256 + threadIdx.x;
    if (c >= (1u << log_n) / 2) return;
    const AutJob J = jobs[blockIdx.y];
    glb2(J.out)[c] = galois_pair(J.in, c, J.galois, log_n);
}

void automorphism_batch_launch(const AutJob* jobs, u32 njobs, u32 log_n, hipStream_t stream) {
    if (njobs == 0) return;
    hipLaunchKernelGGL(k_automorphism_batch, pairs_grid(log_n, njobs), dim3(256), 0, stream, jobs, log_n);
}

// Stateless seeded generator: word (seed, stream, index) is uniform below q by rejection on
// a splitmix64-style mix of a counter (no modulo bias, as Rng::below in
// crates/ckks-train-core/src/sampler.rs:73-82).
CKH_DEV u64 mix64(u64 z) {
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
    return z ^ (z >> 31);
}

CKH_DEV u64 uniform_word(u64 seed, u64 stream, u64 index, u64 q) {
    const u64 key = mix64(seed ^ mix64(stream + 0x9e3779b97f4a7c15ULL));
    const u64 zone = (~0ULL / q) * q;
    u64 x = 0;
    for (u64 a = 0; a < 64; ++a) {
        x = mix64(key + (index * 64 + a) * 0x9e3779b97f4a7c15ULL);
        if (x < zone) break;
    }
    return x % q;
}

__global__ __launch_bounds__(256) void k_fill_uniform(u64* __restrict__ out, u32 q_limbs, u32 nq, u64 seed,
                                                      u64 stream0, const PrimeConst* __restrict__ pc, u32 log_n) {
    const u32 n = 1u << log_n;
    const u32 c = blockIdx.x * 256 + threadIdx.x;
    if (c >= n) return;
    const u32 li = blockIdx.y;
    const u32 prime = li < q_limbs ? li : nq + (li - q_limbs);
    out[(u64)li * n + c] = uniform_word(seed, stream0 + li, c, pc[prime].q);
}

void fill_uniform_launch(u64* out, u32 q_limbs, u32 p_limbs, u32 nq, u64 seed, u64 stream0, const PrimeConst* pc,
                         u32 log_n, hipStream_t stream) {
    const u32 n = 1u << log_n;
    if (q_limbs + p_limbs == 0) return;
    hipLaunchKernelGGL(k_fill_uniform, dim3((n + 255) / 256, q_limbs + p_limbs), dim3(256), 0, stream, out, q_limbs,
                       nq, seed, stream0, pc, log_n);
}

__global__ __launch_bounds__(256) void k_digest(const u64* __restrict__ data, u64 words, u64* out) {
    __shared__ u64 part[256];
    u64 acc = 0;
    for (u64 i = (u64)blockIdx.x * 256 + threadIdx.x; i < words; i += (u64)gridDim.x * 256)
        acc += mix64(data[i] ^ mix64(i + 0x632be59bd9b4e019ULL));
    part[threadIdx.x] = acc;
    __syncthreads();
    for (u32 w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w) part[threadIdx.x] += part[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) atomicAdd((unsigned long long*)out, (unsigned long long)part[0]);
}

void digest_launch(const u64* data, u64 words, u64* out, hipStream_t stream) {
    u64 blocks = (words + 255) / 256;
    if (blocks > 1024) blocks = 1024;
    if (blocks == 0) return;
    hipLaunchKernelGGL(k_digest, dim3((u32)blocks), dim3(256), 0, stream, data, words, out);
}

}  // namespace ckh
