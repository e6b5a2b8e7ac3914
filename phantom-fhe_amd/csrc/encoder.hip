// CKKS encoder / decoder on the GPU (PhantomCKKSEncoder, src/ckks.cu:17-190;
// special FFT, src/fft.cu).
//
// Slot j of a real-coefficient plaintext m(X) mod X^N + 1 is m(zeta^(5^j)),
// zeta = exp(2 pi i / 2N), j < N/2.  Because zeta^(5^j N/2) = i, with
// z_k = m_k + i m_(k+N/2) (k < N/2) that is sum_k z_k zeta^(k 5^j), and since
// {5^j mod 2N} = {1 + 4t}, it is a length-N/2 DFT of the twisted vector
// w_k = z_k zeta^k read at index t_j = (5^j mod 2N - 1) / 4:
//   decode: w = z * zeta^k, W = DFT+(w), slot_j = W[t_j]
//   encode: W[t_j] = slot_j, w = DFT-(W) / (N/2), z = w * zeta^-k,
//           m_k = round(scale Re z_k), m_(k+N/2) = round(scale Im z_k)
// (the reference's encode packs coefficients the same way,
// src/rns_base.cu:49-72).  The DFT is a radix-2 Stockham FFT in double
// precision, in two launches that also do the slot order and the twist.  A rounded coefficient is reduced into each
// prime exactly at any size a double holds (m 2^e with 2^e mod q by squaring,
// where the reference splits it into 64-bit words, src/rns_base.cu:49-170).
// Decoding composes each coefficient from all of the plaintext's limbs
// (Garner's mixed radix, then centred against floor(Q/2)) as the reference's
// compose_array does (src/rns_base.cu:173-253), so it is exact for any
// |m_k| < Q / 2.
#include <cmath>

#include "internal.h"
#include "modarith.h"

namespace pfa {

namespace {

constexpr int kThreads = 256;

// The DFT, M = 2^(S1 + S2) points, in two launches.  The radix-2 Stockham
// network splits by index: its first S1 stages join the 2^S1 points j0 + t B
// (B = M / 2^S1) of a column j0 and leave them at 2^S1 j0 + w, the other S2
// join the points k0 + q A (A = 2^S1) and leave them at k0 + A w.  A thread
// holds 8 points, so three stages are one round in registers, and rounds meet
// in LDS.  One wave a block (512 points): rounds then cost no wait between
// waves, and M / 512 blocks spread over the CUs.  Every butterfly multiplies
// and adds as the stage-by-stage network does, so the results are its own, bit
// for bit.  Latency bounds it (2^14 points are 256 KB), so what counts is the
// number of launches: a launch a stage, with its sincospi, took 14 for 2^14
// points besides one each for the slot order, the twist and the flag.  2^14
// points: 9.3 + 5.6 us encoding (the first also gathers the slots), 4.2 + 5.4
// us decoding, against 14 x 2.3 us; whole calls at N = 2^15, host part
// included: 12 limbs encoded 154 -> 80 us, 3 limbs decoded 426 -> 372 us.
struct Fft {
    const double2 *in;
    double2 *out;
    const double2 *tw;     // [M / 2] exp(i pi t / (M / 2))
    const double2 *zeta;   // [M] exp(i pi k / N)
    const uint32_t *iperm; // [M] the slot of DFT index i
    uint32_t logm, loga;   // points; stages before this launch
    double sign;           // of the exponent
    uint32_t n_values;     // encode: slots given (the others are 0)
    double scale;          // encode: scale / M
    uint32_t *bits;        // encode: largest coeff_bits
};

enum FftEnd { kEncFirst, kEncLast, kDecFirst, kDecLast };

__device__ __forceinline__ void fft2(double2 &a, double2 &b, double2 w, double sign) {
    const double s = sign * w.y;
    const double tr = __builtin_fma(b.x, w.x, -(b.y * s));
    const double ti = __builtin_fma(b.x, s, b.y * w.x);
    b = double2{a.x - tr, a.y - ti};
    a = double2{a.x + tr, a.y + ti};
}

// R stages, the first of sub-transform length ns = 2^ls (in local points), on
// the points j + u 2^S / 2^R of one column; leaves point j's outputs in order
// w = 0 .. 2^R - 1 (local index 2^R (j - k) + k + w ns).
template <int R>
__device__ __forceinline__ void fft_round(double2 (&x)[1 << R], uint32_t k, uint32_t ls, uint32_t k0, const Fft &f) {
    double2 y[1 << R];
#pragma unroll
    for (int g = 0; g < R; g++) {
        // x: (u, w), u < 2^(R - g), w < 2^g, at u 2^g + w
        const int H = 1 << (R - 1 - g), W = 1 << g;
        const uint32_t shift = f.logm - 1 - f.loga - ls - g;
#pragma unroll
        for (int w = 0; w < W; w++) {
            const uint32_t kl = k + ((uint32_t)w << ls);
            const double2 t = f.tw[(k0 + (kl << f.loga)) << shift];
#pragma unroll
            for (int u = 0; u < H; u++) {
                double2 a = x[u * W + w], b = x[(u + H) * W + w];
                fft2(a, b, t, f.sign);
                y[u * 2 * W + w] = a;
                y[u * 2 * W + w + W] = b;
            }
        }
#pragma unroll
        for (int i = 0; i < (1 << R); i++) x[i] = y[i];
    }
}

__device__ __forceinline__ uint32_t coeff_bits(double v);

template <int END>
__device__ __forceinline__ double2 fft_load(const Fft &f, uint32_t i) {
    if constexpr (END == kEncFirst) {
        const uint32_t j = f.iperm[i];
        return j < f.n_values ? f.in[j] : double2{0.0, 0.0};
    } else if constexpr (END == kDecFirst) {
        const double2 v = f.in[i], z = f.zeta[i];  // z_k zeta^k
        return double2{__builtin_fma(v.x, z.x, -(v.y * z.y)), __builtin_fma(v.x, z.y, v.y * z.x)};
    } else {
        return f.in[i];
    }
}

template <int END>
__device__ __forceinline__ void fft_store(const Fft &f, uint32_t i, double2 v, uint32_t &mb) {
    if constexpr (END == kEncLast) {
        const double2 z = f.zeta[i];  // w_k zeta^-k / M times the scale
        const double s = -z.y;
        const double re = __builtin_fma(v.x, z.x, -(v.y * s)) * f.scale;
        const double im = __builtin_fma(v.x, s, v.y * z.x) * f.scale;
        const uint32_t br = coeff_bits(re), bi = coeff_bits(im);
        mb = max(mb, max(br, bi));
        f.out[i] = double2{re, im};
    } else if constexpr (END == kDecLast) {
        f.out[f.iperm[i]] = v;
    } else {
        f.out[i] = v;
    }
}

template <int S, int END>
__global__ void __launch_bounds__(64) k_fft(Fft f) {
    constexpr int PTS = 1 << S, COLS = 512 / PTS, RL = S % 3 ? S % 3 : 3, NR = (S - RL) / 3;  // NR rounds of 3, one of RL
    constexpr bool FIRST = END == kEncFirst || END == kDecFirst;
    __shared__ double2 lds[512 + 64];
    const uint32_t col = threadIdx.x % COLS, tl = threadIdx.x / COLS;
    const uint32_t c0 = blockIdx.x * COLS + col;
    const uint32_t k0 = FIRST ? 0 : c0;
    // point t of this column comes from c0 + t 2^(logm - S) in either half
    const uint32_t step = f.logm - S;
    auto at = [&](uint32_t i) { return (i + (i >> 3)) * COLS + col; };
    if (END == kEncFirst && blockIdx.x == 0 && threadIdx.x == 0) *f.bits = 1;
    double2 x[8];
#pragma unroll
    for (int u = 0; u < 8; u++) x[u] = fft_load<END>(f, c0 + ((tl + u * (PTS / 8)) << step));
#pragma unroll
    for (int r = 0; r < NR; r++) {
        if (r) {
#pragma unroll
            for (int u = 0; u < 8; u++) x[u] = lds[at(tl + u * (PTS / 8))];
            __syncthreads();
        }
        const uint32_t ls = 3 * r, k = tl & ((1u << ls) - 1);
        fft_round<3>(x, k, ls, k0, f);
#pragma unroll
        for (int w = 0; w < 8; w++) lds[at(8 * (tl - k) + k + ((uint32_t)w << ls))] = x[w];
        __syncthreads();
    }
    uint32_t mb = 1;
    // the last round: 8 / 2^RL groups of 2^RL points, each at j + v PTS / 2^RL before and after
#pragma unroll
    for (int g = 0; g < (8 >> RL); g++) {
        const uint32_t j = tl + g * (PTS / 8);
        double2 z[1 << RL];
#pragma unroll
        for (int u = 0; u < (1 << RL); u++) z[u] = lds[at(j + u * (PTS >> RL))];
        fft_round<RL>(z, j, S - RL, k0, f);
#pragma unroll
        for (int w = 0; w < (1 << RL); w++) {
            const uint32_t p = j + w * (PTS >> RL);
            fft_store<END>(f, FIRST ? c0 * PTS + p : c0 + (p << f.loga), z[w], mb);
        }
    }
    if constexpr (END == kEncLast) {
        for (int d = 32; d; d >>= 1) mb = max(mb, (uint32_t)__shfl_xor((int)mb, d));
        if (threadIdx.x == 0) atomicMax(f.bits, mb);
    }
}

// The FFT's tables: exp(i pi t / (M / 2)), t < M / 2, then exp(i pi k / N), k < M.
__global__ void k_fft_tables(double2 *tw, double2 *zeta, uint32_t M) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= M) return;
    double s, c;
    if (i < M / 2) {
        sincospi((double)i / (double)(M / 2), &s, &c);
        tw[i] = double2{c, s};
    }
    sincospi((double)i / (double)(2 * M), &s, &c);
    zeta[i] = double2{c, s};
}

// a b mod q for any a, b < 2^64 (ratio = floor(2^128 / q))
__device__ __forceinline__ uint64_t mulmod_any(uint64_t a, uint64_t b, uint64_t q, ulonglong2 rt) {
    return barrett128(mul_wide(a, b), q, rt.x, rt.y);
}

// x mod q for a double x >= 0 that holds an integer: below 2^62 directly,
// above it as m 2^e (53-bit m, e >= 10) with 2^e mod q by squaring.
__device__ __forceinline__ uint64_t dbl_int_mod(double x, uint64_t q, ulonglong2 rt) {
    if (x < 4611686018427387904.0) return barrett128(U128{(uint64_t)x, 0}, q, rt.x, rt.y);  // 2^62
    const uint64_t bits = (uint64_t)__double_as_longlong(x);
    uint32_t e = (uint32_t)((bits >> 52) & 0x7ff) - 1075u;
    const uint64_t m = (bits & ((1ull << 52) - 1)) | (1ull << 52);
    uint64_t p = 1, b = 2;  // primes here are at least 2N + 1
    for (; e; e >>= 1) {
        if (e & 1u) p = mulmod_any(p, b, q, rt);
        b = mulmod_any(b, b, q, rt);
    }
    return mulmod_any(barrett128(U128{m, 0}, q, rt.x, rt.y), p, q, rt);
}

// The reference's size check (src/ckks.cu:112-126): ceil(log2(max(|v|, 1))) + 1
// bits, exact from the binary exponent; not finite: ~0u.
__device__ __forceinline__ uint32_t coeff_bits(double v) {
    const double a = fabs(v);
    if (!(a < __builtin_huge_val())) return ~0u;
    if (a <= 1.0) return 1;
    int ex;
    const double m = frexp(a, &ex);  // a = m 2^ex, m in [0.5, 1)
    return (uint32_t)(m > 0.5 ? ex : ex - 1) + 1;
}

// Unrounded coefficients u_k = (m_k, m_(k+M)) -> RNS residues of primes
// [kLimbGroup blockIdx.y, ...) of the L first.  A thread a coefficient pair and
// a few limbs: with all limbs in one thread, 2^14 pairs were 256 waves of a
// chain of 2 L reductions each (12 limbs 14.9 -> 4.4 us).
// Block (0, 0) hands the largest coeff_bits, complete here, to the host.
constexpr uint32_t kLimbGroup = 2;
__global__ void __launch_bounds__(kThreads)
    k_enc_round(const double2 *u, uint64_t *out, const uint64_t *mod, const ulonglong2 *ratio, uint32_t L, uint32_t N,
                const uint32_t *bits, uint32_t *host_bits) {
    const uint32_t M = N / 2, k = blockIdx.x * kThreads + threadIdx.x;
    if (k == 0 && blockIdx.y == 0) *host_bits = *bits;
    const double2 v = u[k];
    const double x[2] = {rint(v.x), rint(v.y)};
    const uint32_t l0 = blockIdx.y * kLimbGroup, l1 = min(l0 + kLimbGroup, L);
    for (uint32_t l = l0; l < l1; l++) {
        const uint64_t q = mod[l];
        const ulonglong2 rt = ratio[l];
        for (int h = 0; h < 2; h++) {
            const double a = fabs(x[h]);
            uint64_t t = dbl_int_mod(a < __builtin_huge_val() ? a : 0.0, q, rt);
            if (x[h] < 0 && t) t = q - t;
            out[(size_t)l * N + k + h * M] = t;
        }
    }
}

// Unrounded coefficients -> the reference's level-independent single-chain
// coefficients (src/single_chain_plaintext.cu:93-150): the rounded
// coefficient's residue mod q0, centred into (-q0/2, q0/2].
__global__ void __launch_bounds__(kThreads)
    k_enc_round_signed(const double2 *u, int64_t *out, uint32_t N, uint64_t q0, ulonglong2 r0, const uint32_t *bits,
                       uint32_t *host_bits) {
    const uint32_t M = N / 2, k = blockIdx.x * kThreads + threadIdx.x;
    if (k == 0) *host_bits = *bits;
    const double2 v = u[k];
    const double x[2] = {rint(v.x), rint(v.y)};
    for (int h = 0; h < 2; h++) {
        const double a = fabs(x[h]);
        uint64_t t = dbl_int_mod(a < __builtin_huge_val() ? a : 0.0, q0, r0);
        if (x[h] < 0 && t) t = q0 - t;
        out[k + h * M] = t > q0 / 2 ? -(int64_t)(q0 - t) : (int64_t)t;
    }
}

// Coefficient i of the L coefficient-form limbs as a double times inv_scale,
// centred (compose_array, src/rns_base.cu:173-253): Garner's mixed-radix
// digits v_j (x = sum_j v_j prod_{i<j} q_i, each v_j < q_j) are written over
// the limbs in place, x is compared with floor(Q/2) digit by digit from the top
// (the digits of (Q - 1) / 2 by long division in the same radix), and the
// value is x or -(Q - x).  inv[i][j] = q_i^-1 mod q_j as Shoup pairs.
__device__ double compose_one(uint64_t *coef, size_t i, const uint64_t *mod, const ulonglong2 *ratio,
                              const ulonglong2 *inv, uint32_t Q, uint32_t L, uint32_t N, double inv_scale) {
    for (uint32_t j = 1; j < L; j++) {
        const uint64_t q = mod[j];
        const ulonglong2 rt = ratio[j];
        uint64_t t = coef[(size_t)j * N + i];
        for (uint32_t l = 0; l < j; l++) {
            const uint64_t v = barrett128(U128{coef[(size_t)l * N + i], 0}, q, rt.x, rt.y);
            const ulonglong2 f = inv[(size_t)l * Q + j];
            t = shoup(sub_mod(t, v, q), f.x, f.y, q);
        }
        coef[(size_t)j * N + i] = t;
    }
    int cmp = 0;
    uint64_t r = 0;
    for (uint32_t j = L; j-- > 0;) {
        const uint64_t q = mod[j], v = coef[(size_t)j * N + i];
        const uint64_t d = r * q + (q - 1);  // < 2 q
        const uint64_t h = d >> 1;
        r = d & 1;
        if (cmp == 0) cmp = v > h ? 1 : (v < h ? -1 : 0);
    }
    // x, or Q - x = (Q - 1 - x) + 1 with digits q_j - 1 - v_j and a carry
    const bool neg = cmp > 0;
    double res = 0.0, wj = inv_scale;
    uint64_t carry = 1;
    for (uint32_t j = 0; j < L; j++) {
        const uint64_t q = mod[j], v = coef[(size_t)j * N + i];
        uint64_t dj = v;
        if (neg) {
            dj = q - 1 - v + carry;
            carry = dj == q ? 1 : 0;
            dj = carry ? 0 : dj;
        }
        if (dj) res += (double)dj * wj;  // zero digits skipped: wj may have overflowed
        wj *= (double)q;
    }
    return neg ? -res : res;
}

// Coefficient-form limbs -> z_k = (m_k + i m_(k+M)) / scale, a thread a coefficient.
__global__ void __launch_bounds__(kThreads)
    k_dec_compose(uint64_t *coef, double *z, const uint64_t *mod, const ulonglong2 *ratio, const ulonglong2 *inv,
                  uint32_t Q, uint32_t L, uint32_t N, double inv_scale) {
    const uint32_t M = N / 2, i = blockIdx.x * kThreads + threadIdx.x;
    z[2 * (i & (M - 1)) + (i >= M)] = compose_one(coef, i, mod, ratio, inv, Q, L, N, inv_scale);
}

template <int END>
void launch_fft(const Fft &f, uint32_t S, hipStream_t s) {
    const dim3 grid((1u << f.logm) / 512), block(64);
    switch (S) {
        case 4: hipLaunchKernelGGL((k_fft<4, END>), grid, block, 0, s, f); break;
        case 5: hipLaunchKernelGGL((k_fft<5, END>), grid, block, 0, s, f); break;
        case 6: hipLaunchKernelGGL((k_fft<6, END>), grid, block, 0, s, f); break;
        case 7: hipLaunchKernelGGL((k_fft<7, END>), grid, block, 0, s, f); break;
        case 8: hipLaunchKernelGGL((k_fft<8, END>), grid, block, 0, s, f); break;
        default: fail(PFA_ERR_INVALID_ARGUMENT, "unsupported FFT size");
    }
}

// Both launches: `in` through `mid` to `out` (N is 2^10 .. 2^17, so either
// part has 4 to 8 stages).
template <int FIRST, int LAST>
void fft(const Ctx &c, Fft f, const double2 *in, double2 *mid, double2 *out, hipStream_t s) {
    f.tw = c.fft_tw;
    f.zeta = c.fft_tw + c.N / 4;
    f.iperm = c.slot_iperm;
    f.logm = c.logN - 1;
    const uint32_t s1 = f.logm / 2;
    f.in = in;
    f.out = mid;
    f.loga = 0;
    launch_fft<FIRST>(f, s1, s);
    f.in = mid;
    f.out = out;
    f.loga = s1;
    launch_fft<LAST>(f, f.logm - s1, s);
}

// Slots -> unrounded coefficients (m_k, m_(k+M)) in w, the largest coeff_bits in *bits.
double2 *encode_coeffs_f64(const Ctx &c, Scratch &sc, const double *values, size_t n_values, double scale,
                           uint32_t *bits, hipStream_t s) {
    const uint32_t M = c.N / 2;
    double2 *buf = sc.alloc<double2>(2 * (size_t)M);
    Fft f{};
    f.sign = -1.0;
    f.n_values = (uint32_t)n_values;
    f.scale = scale / (double)M;
    f.bits = bits;
    fft<kEncFirst, kEncLast>(c, f, (const double2 *)values, buf, buf + M, s);
    return buf + M;
}

// The arena's mapped host word, which a kernel of stream s writes and the host
// reads after waiting for s: a copy from device memory waits for its own
// launch as well.
uint32_t *host_word(Arena &a, uint32_t **dev) {
    if (!a.word) {
        PFA_HIP(hipHostMalloc((void **)&a.word, 64, hipHostMallocMapped));
        PFA_HIP(hipHostGetDevicePointer((void **)&a.word_dev, a.word, 0));
    }
    *dev = a.word_dev;
    return a.word;
}

}  // namespace

void encoder_init(Ctx &c) {
    const uint32_t M = c.N / 2, m2 = 2 * c.N;
    std::vector<uint32_t> iperm(M);
    uint64_t p = 1;
    for (uint32_t j = 0; j < M; j++) {
        iperm[(p - 1) / 4] = j;
        p = (p * 5) % m2;
    }
    c.slot_iperm = c.upload(iperm);
    c.fft_tw = c.upload(std::vector<double2>(M / 2 + M));
    hipLaunchKernelGGL(k_fft_tables, dim3((M + kThreads - 1) / kThreads), dim3(kThreads), 0, hipStreamPerThread,
                       c.fft_tw, c.fft_tw + M / 2, M);
    PFA_HIP(hipGetLastError());
    PFA_HIP(hipStreamSynchronize(hipStreamPerThread));
    std::vector<ulonglong2> inv((size_t)c.Q * c.Q, ulonglong2{0, 0});
    for (uint32_t i = 0; i < c.Q; i++)
        for (uint32_t j = i + 1; j < c.Q; j++) {
            const uint64_t q = c.moduli[j], v = invmod(c.moduli[i] % q, q);
            inv[(size_t)i * c.Q + j] = ulonglong2{v, shoup_of(v, q)};
        }
    c.crt_inv = c.upload(inv);
}

// Bit length of q_0 q_1 ... q_(L-1) (the reference's total_coeff_modulus_bit_count
// of the level with L primes), by exact multi-word products.
static uint32_t total_bits(const Ctx &c, uint32_t L) {
    std::vector<uint64_t> p{1};
    for (uint32_t i = 0; i < L; i++) {
        u128 carry = 0;
        for (uint64_t &w : p) {
            const u128 t = (u128)w * c.moduli[i] + carry;
            w = (uint64_t)t;
            carry = t >> 64;
        }
        if (carry) p.push_back((uint64_t)carry);
    }
    return 64 * (uint32_t)(p.size() - 1) + (64 - (uint32_t)__builtin_clzll(p.back()));
}

static ulonglong2 host_ratio(uint64_t q) { return ulonglong2{(uint64_t)(~(u128)0 / q), (uint64_t)((~(u128)0 / q) >> 64)}; }

// The reference's scale bound (src/ckks.cu:87-89 encode, :148-151 decode).
static void check_scale(double scale, uint32_t tb, int extra) {
    require(scale > 0 && std::isfinite(scale) && (int)std::log2(scale) + extra < (int)tb, "scale out of bounds");
}

}  // namespace pfa

using namespace pfa;

extern "C" {

int pfa_ckks_encode(const pfa_context *ctx, const double *values, size_t n_values, double scale, uint64_t *out,
                    size_t L, void *stream) {
    return guarded([&] {
        const Ctx &c = *ctx_of(ctx);
        require(out && (values || n_values == 0), "null argument");
        const uint32_t M = c.N / 2;
        require(n_values >= 1, "Input vector is empty");
        require(n_values <= M, "Input vector exceeds max slots");
        require(L >= 1 && L <= c.Q, "plaintext limb count out of range");
        const uint32_t tb = total_bits(c, (uint32_t)L);
        check_scale(scale, tb, 1);
        const hipStream_t s = as_stream(stream);
        Scratch sc(c, s);
        uint32_t *flag = sc.alloc<uint32_t>(1), *word_dev;
        const volatile uint32_t *word = host_word(arena_for(c, s), &word_dev);
        const double2 *u = encode_coeffs_f64(c, sc, values, n_values, scale, flag, s);
        hipLaunchKernelGGL(k_enc_round, dim3(M / kThreads, ((uint32_t)L + kLimbGroup - 1) / kLimbGroup),
                           dim3(kThreads), 0, s, u, out, c.mod, c.ratio, (uint32_t)L, c.N, flag, word_dev);
        PFA_HIP(hipGetLastError());
        NttLaunch fw{out, out, 0, 0, 1, (uint32_t)L};
        ntt_forward(c, fw, s);
        PFA_HIP(hipStreamSynchronize(s));
        require(*word < tb, "encoded values are too large");  // src/ckks.cu:122-126
    });
}

int pfa_ckks_encode_coeffs(const pfa_context *ctx, const double *values, size_t n_values, double scale,
                           int64_t *coeffs, void *stream) {
    return guarded([&] {
        const Ctx &c = *ctx_of(ctx);
        require(coeffs && (values || n_values == 0), "null argument");
        const uint32_t M = c.N / 2;
        require(n_values >= 1, "Input vector is empty");
        require(n_values <= M, "Input vector exceeds max slots");
        // encoded at chain index 1 (all of Q), then reduced mod q0 and centred
        const uint32_t tb = total_bits(c, c.Q);
        check_scale(scale, tb, 1);
        const hipStream_t s = as_stream(stream);
        Scratch sc(c, s);
        uint32_t *flag = sc.alloc<uint32_t>(1), *word_dev;
        const volatile uint32_t *word = host_word(arena_for(c, s), &word_dev);
        const double2 *u = encode_coeffs_f64(c, sc, values, n_values, scale, flag, s);
        hipLaunchKernelGGL(k_enc_round_signed, dim3(M / kThreads), dim3(kThreads), 0, s, u, coeffs, c.N, c.moduli[0],
                           host_ratio(c.moduli[0]), flag, word_dev);
        PFA_HIP(hipGetLastError());
        PFA_HIP(hipStreamSynchronize(s));
        require(*word < tb, "encoded values are too large");
    });
}

int pfa_ckks_decode(const pfa_context *ctx, const uint64_t *in, size_t L, double scale, double *values, void *stream) {
    return guarded([&] {
        const Ctx &c = *ctx_of(ctx);
        require(in && values, "null argument");
        require(L >= 1 && L <= c.Q, "plaintext limb count out of range");
        check_scale(scale, total_bits(c, (uint32_t)L), 0);
        const hipStream_t s = as_stream(stream);
        const uint32_t M = c.N / 2;
        Scratch sc(c, s);
        uint64_t *coef = sc.alloc((size_t)L * c.N);
        double2 *buf = sc.alloc<double2>(2 * (size_t)M);
        NttLaunch inv{in, coef, 0, 0, 1, (uint32_t)L};
        ntt_inverse(c, inv, s);
        hipLaunchKernelGGL(k_dec_compose, dim3(c.N / kThreads), dim3(kThreads), 0, s, coef, (double *)buf, c.mod, c.ratio,
                           c.crt_inv, c.Q, (uint32_t)L, c.N, 1.0 / scale);
        Fft f{};
        f.sign = 1.0;
        fft<kDecFirst, kDecLast>(c, f, buf, buf + M, (double2 *)values, s);
        PFA_HIP(hipGetLastError());
    });
}

}  // extern "C"
