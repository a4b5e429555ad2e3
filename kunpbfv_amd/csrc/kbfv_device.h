// Device-side modular arithmetic for gfx950 (CDNA4, wave64).
//
// All residues are uint64 below 2^60 (the 60-bit chains and the plain
// modulus), so lazy values up to 4q fit in 62 bits.  CDNA4 has no 64x64
// multiply; the compiler expands 64-bit products into 32-bit
// v_mad_u64_u32 / v_mul_hi_u32 / v_mul_lo_u32 sequences.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

struct __align__(16) kbfv_tw {
    uint64_t w;   // twiddle
    uint64_t ws;  // Shoup companion floor(w * 2^64 / q)
};

struct kbfv_u128 {
    uint64_t lo, hi;
};

// 16 bytes of a caller's buffer, which need be aligned to its 8-byte words only
typedef uint64_t kb_u64x2 __attribute__((ext_vector_type(2), aligned(8)));
typedef uint32_t kb_u32x4 __attribute__((ext_vector_type(4), aligned(8)));

__device__ __forceinline__ uint64_t kb_mulhi(uint64_t a, uint64_t b) { return __umul64hi(a, b); }

// a mod q for a in [0, 2q)
__device__ __forceinline__ uint64_t kb_csub(uint64_t a, uint64_t q) {
    uint64_t t = a - q;
    return t < a ? t : a;  // a >= q  <=>  a - q does not wrap
}

// Shoup product x*w mod q, lazily in [0, 2q); valid for any 64-bit x.
__device__ __forceinline__ uint64_t kb_shoup_lazy(uint64_t x, uint64_t w, uint64_t ws, uint64_t q) {
    return x * w - kb_mulhi(x, ws) * q;
}
__device__ __forceinline__ uint64_t kb_shoup(uint64_t x, uint64_t w, uint64_t ws, uint64_t q) {
    return kb_csub(kb_shoup_lazy(x, w, ws, q), q);
}

// full 64x64 -> 128 product
__device__ __forceinline__ kbfv_u128 kb_mul128(uint64_t a, uint64_t b) {
    kbfv_u128 r;
    r.lo = a * b;
    r.hi = kb_mulhi(a, b);
    return r;
}
__device__ __forceinline__ void kb_mac128(kbfv_u128 &acc, uint64_t a, uint64_t b) {
    uint64_t lo = a * b;
    uint64_t hi = kb_mulhi(a, b);
    acc.lo += lo;
    acc.hi += hi + (acc.lo < lo ? 1u : 0u);
}
__device__ __forceinline__ void kb_add128(kbfv_u128 &acc, uint64_t v) {
    acc.lo += v;
    acc.hi += (acc.lo < v ? 1u : 0u);
}
// 128-bit wrap-around subtraction of a 64-bit value
__device__ __forceinline__ void kb_sub128(kbfv_u128 &acc, uint64_t v) {
    uint64_t borrow = acc.lo < v ? 1u : 0u;
    acc.lo -= v;
    acc.hi -= borrow;
}

// Barrett reduction of any 128-bit value with mu = floor(2^128 / q) = (mu_hi, mu_lo).
// The quotient estimate floor(a * mu / 2^128) is at least floor(a / q) - 1, so a
// single conditional subtraction yields the canonical residue in [0, q).
__device__ __forceinline__ uint64_t kb_barrett128(kbfv_u128 a, uint64_t q, uint64_t mu_lo,
                                                  uint64_t mu_hi) {
    uint64_t t = kb_mulhi(a.lo, mu_lo);
    uint64_t m1lo = a.lo * mu_hi, m1hi = kb_mulhi(a.lo, mu_hi);
    uint64_t m2lo = a.hi * mu_lo, m2hi = kb_mulhi(a.hi, mu_lo);
    uint64_t s = t + m1lo;
    uint64_t c1 = s < t ? 1u : 0u;
    uint64_t s2 = s + m2lo;
    uint64_t c2 = s2 < s ? 1u : 0u;
    uint64_t qe = a.hi * mu_hi + m1hi + m2hi + c1 + c2;
    uint64_t r = a.lo - qe * q;
    return kb_csub(r, q);
}

// canonical a*b mod q via Barrett
__device__ __forceinline__ uint64_t kb_mulmod(uint64_t a, uint64_t b, uint64_t q, uint64_t mu_lo,
                                              uint64_t mu_hi) {
    return kb_barrett128(kb_mul128(a, b), q, mu_lo, mu_hi);
}

__device__ __forceinline__ uint64_t kb_addmod(uint64_t a, uint64_t b, uint64_t q) {
    return kb_csub(a + b, q);
}
__device__ __forceinline__ uint64_t kb_submod(uint64_t a, uint64_t b, uint64_t q) {
    return kb_csub(a + q - b, q);
}

// double -> uint64 truncation saturating at 2^64 - 1 for non-negative x (the
// conversion the reference's nvcc build performs for static_cast<uint64_t>)
__device__ __forceinline__ uint64_t kb_f64_to_u64_sat(double x) {
    return x >= 18446744073709551616.0 ? ~0ULL : (uint64_t)x;
}
// uint64 -> double with one rounding (error at most 2^11)
__device__ __forceinline__ double kb_u64_to_f64(uint64_t x) {
    return fma((double)(uint32_t)(x >> 32), 4294967296.0, (double)(uint32_t)x);
}

// a*b + c mod 2^64, one v_mad_u64_u32
__device__ __forceinline__ uint64_t kb_mad32(uint32_t a, uint32_t b, uint64_t c) {
    return (uint64_t)a * b + c;
}
// a*b mod 2^32 as one opaque v_mul_lo_u32.  Written as plain C, the compiler
// folds the cross products below back into 64x64-bit multiplies and expands
// those again with extra v_mad_u64_u32 steps (about twice the instructions).
__device__ __forceinline__ uint32_t kb_mul_lo32(uint32_t a, uint32_t b) {
    uint32_t r;
    asm("v_mul_lo_u32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// 64-bit value + 32-bit value as one v_mad_u64_u32 (b * 1 + a): no carry
// through an SGPR and no register pair to build for b
__device__ __forceinline__ uint64_t kb_add_u32(uint64_t a, uint32_t b) {
    uint32_t one = 1;
    asm("" : "+s"(one));  // a multiplier the optimizer cannot fold away
    return kb_mad32(b, one, a);
}

// Shoup product x*w mod q with an under-estimated quotient, in [0, 4q) for any
// x < 2^64.  floor(x*ws / 2^64) = x1*s1 + hi(x1*s0) + hi(x0*s1) + e with
// e in {0, 1, 2} (the carries of the low words and hi(x0*s0)); leaving e out
// adds at most 2q to the lazy residue x*w - h*q in [0, 2q).  nq = 2^64 - q.
__device__ __forceinline__ uint64_t kb_shoup4(uint64_t x, uint64_t w, uint64_t ws, uint64_t nq) {
    const uint32_t x0 = (uint32_t)x, x1 = (uint32_t)(x >> 32);
    const uint32_t s0 = (uint32_t)ws, s1 = (uint32_t)(ws >> 32);
    const uint64_t h = kb_add_u32(kb_mad32(x1, s1, __umulhi(x1, s0)), __umulhi(x0, s1));
    const uint32_t h0 = (uint32_t)h, h1 = (uint32_t)(h >> 32);
    const uint32_t w0 = (uint32_t)w, w1 = (uint32_t)(w >> 32);
    const uint32_t n0 = (uint32_t)nq, n1 = (uint32_t)(nq >> 32);
    const uint64_t r = kb_mad32(h0, n0, kb_mad32(x0, w0, 0));
    const uint32_t cross = kb_mul_lo32(x0, w1) + kb_mul_lo32(x1, w0) + kb_mul_lo32(h0, n1) +
                           kb_mul_lo32(h1, n0);
    return r + ((uint64_t)cross << 32);
}

// a >= m ? a - m : a for a, m < 2^63, given nm = 2^64 - m: the sign of a - m
// selects word by word (v_bfi_b32), no compare or carry through an SGPR
__device__ __forceinline__ uint64_t kb_csub_sel(uint64_t a, uint64_t nm) {
    const uint64_t t = a + nm;
    const uint32_t msk = (uint32_t)((int32_t)(uint32_t)(t >> 32) >> 31);
    uint32_t lo, hi;
    asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(lo) : "v"(msk), "v"((uint32_t)a), "v"((uint32_t)t));
    asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(hi) : "v"(msk), "v"((uint32_t)(a >> 32)), "v"((uint32_t)(t >> 32)));
    return ((uint64_t)hi << 32) | lo;
}

// Signed 30-bit halves of a residue x < 2^60: x - 2^59 = x1 2^30 + x0 with
// x0 in [-2^29, 2^29), x1 in [-2^29, 2^29].
__device__ __forceinline__ void kb_split30(uint64_t x, int &x0, int &x1) {
    const uint64_t z = x + (1ULL << 29);
    x0 = (int)((uint32_t)z & 0x3fffffffu) - (1 << 29);
    x1 = (int)(uint32_t)(z >> 30) - (1 << 29);
}
// acc += a*b (wrap-around), one v_mad_i64_i32 / v_mad_u64_u32
__device__ __forceinline__ void kb_mad(int64_t &acc, int a, int b) {
    acc = (int64_t)((uint64_t)acc + (uint64_t)((int64_t)a * b));
}
__device__ __forceinline__ void kb_mad(uint64_t &acc, uint32_t a, uint32_t b) { acc += (uint64_t)a * b; }
// Multiplication modulo a prime q = 2^60 - c, 0 < c < 2^28, on signed values.  x =
// x1 2^32 + x0 with x0 signed; the constant w (twiddle) and w' = w 2^32 mod q are
// split at 28 bits into signed 32-bit halves, w = w1 2^28 + w0.  Then
// x w = x0 w + x1 w' = A + 2^28 B, A = x0 w0 + x1 w'0, B = x0 w1 + x1 w'1, and with
// B = v 2^32 + b, 0 <= b < 2^32, the part v 2^60 is v c modulo q: A + 2^28 b + v c.
// Six multiply-adds with no carry between them.  |w|, |w'| <= 2^59 and |w0|, |w'0| <=
// 2^27, so for |x| < 8 (2^60 - 2^32) B stays below 2^63 and for |x| <= X 2^60 the result
// lies between -d 2^60 and (1 + d) 2^60, d = (1/4 + X/32) (1 + c 2^-28).
__host__ __device__ __forceinline__ bool kb_fold_prime(uint64_t q) { return (q >> 28) == (1ULL << 32) - 1; }
__device__ __forceinline__ uint32_t kb_fold_c(uint64_t q) { return (uint32_t)((1ULL << 60) - q); }
// x w + add, w as a pair of packed halves (w0 | w1 << 32); k28 = 2^28
__device__ __forceinline__ uint64_t kb_fmul(uint64_t x, kbfv_tw w, uint32_t c, uint32_t k28, uint64_t add) {
    const int x0 = (int)(uint32_t)x, x1 = (int)(uint32_t)((x + (1ULL << 31)) >> 32);
    int64_t A = (int64_t)add, B = 0;
    kb_mad(B, x0, (int)(uint32_t)(w.w >> 32));
    kb_mad(A, x0, (int)(uint32_t)w.w);
    kb_mad(B, x1, (int)(uint32_t)(w.ws >> 32));
    kb_mad(A, x1, (int)(uint32_t)w.ws);
    uint64_t r = kb_mad32((uint32_t)B, k28, (uint64_t)A);
    int64_t s = (int64_t)r;
    kb_mad(s, (int)(uint32_t)((uint64_t)B >> 32), (int)c);
    return (uint64_t)s;
}
// signed x -> x mod q up to [-8c, 2^60 + 7c]
__device__ __forceinline__ uint64_t kb_sfold(uint64_t x, uint32_t c) {
    const uint32_t hi = (uint32_t)(x >> 32);
    int64_t r = (int64_t)(((uint64_t)(hi & 0x0fffffffu) << 32) | (uint32_t)x);
    kb_mad(r, (int)hi >> 28, (int)c);
    return (uint64_t)r;
}
// any 64-bit x -> x mod q up to [0, 2^60 + 15c]
__device__ __forceinline__ uint64_t kb_ufold(uint64_t x, uint32_t c) {
    const uint32_t hi = (uint32_t)(x >> 32);
    return kb_mad32(hi >> 28, c, ((uint64_t)(hi & 0x0fffffffu) << 32) | (uint32_t)x);
}
// v below 2^122 modulo a prime 2^60 - c, c < 2^28: v = H 2^60 + L is H c + L; of H c's
// upper word product u 2^28 + w the part u 2^60 folds once more.  Half the multiplies of
// a Barrett reduction.
__device__ __forceinline__ uint64_t kb_fold128(kbfv_u128 v, uint32_t c, uint64_t nq) {
    const uint64_t H = v.hi << 4 | v.lo >> 60, L = v.lo & ((1ULL << 60) - 1);
    const uint64_t p = (uint64_t)(uint32_t)(H >> 32) * c;
    const uint64_t w = (uint64_t)((uint32_t)p & 0x0fffffffu) << 32;
    const uint64_t r = kb_mad32((uint32_t)(p >> 28), c, kb_mad32((uint32_t)H, c, L) + w);  // < 2^62
    return kb_csub_sel(kb_ufold(r, c), nq);
}
// v below 2^125 modulo a prime 2^60 - c, c < 2^26: the same with the upper word at 2^64,
// which is 16 c
__device__ __forceinline__ bool kb_fold125_prime(uint64_t q) { return (q >> 26) == (1ULL << 34) - 1; }
__device__ __forceinline__ uint64_t kb_fold125(kbfv_u128 v, uint32_t c, uint64_t nq) {
    const uint32_t c16 = c << 4;                          // below 2^30
    const uint64_t p = (uint64_t)(uint32_t)(v.hi >> 32) * c16;  // below 2^59
    const uint64_t w = (uint64_t)((uint32_t)p & 0x0fffffffu) << 32;
    const uint64_t r = kb_mad32((uint32_t)v.hi, c16, kb_ufold(v.lo, c)) + w;  // below 2^62 + 2^61 + 2^30
    return kb_csub_sel(kb_ufold(kb_mad32((uint32_t)(p >> 28), c, r), c), nq);
}
// signed x, |x| <= 7.9 2^60 -> [0, q)
__device__ __forceinline__ uint64_t kb_fold_canon(uint64_t x, uint64_t q, uint64_t nq, uint32_t c) {
    return kb_csub_sel(kb_ufold(x + (q << 3), c), nq);
}
// Butterflies for primes 2^60 - c, c < 2^28: values are signed, twiddles signed
// halves (kb_fmul).  The product comes on top of its addend, so the sum is free and
// the difference is 2a - (a + t); six multiply-adds in place of the Shoup product's
// ten multiplies, and no conditional subtraction.  A product of |x| <= X 2^60 lies in
// (-d, 1 + d) 2^60, d < 1/2 + X/16.  Forward: [0, 1] grows over four levels to (-1.6,
// 2.6), (-3.3, 4.3), (-5.0, 6.0), (-6.9, 7.9).  Inverse: values in (-0.9, 1.9) give sums
// below 7.6 over two levels, the sums are folded back to [0, 1] there, the products of
// differences below 5.7 stay in (-0.9, 1.9).
__device__ __forceinline__ void ct_fold(uint64_t &a, uint64_t &b, kbfv_tw w, uint32_t c, uint32_t k28) {
    const uint64_t s = kb_fmul(b, w, c, k28, a);
    b = (a << 1) - s;
    a = s;
}

template <bool RED>
__device__ __forceinline__ void gs_fold(uint64_t &a, uint64_t &b, kbfv_tw w, uint32_t c, uint32_t k28) {
    const uint64_t u = a + b;
    b = kb_fmul(a - b, w, c, k28, 0);
    a = RED ? kb_sfold(u, c) : u;
}

// Place in a limb's twiddle table of group x of level g (2^g groups): levels follow each
// other; of a prime near 2^60 (fold) the last five store the groups of one 32-element block
// 2^(log_n - 5) apart, so that lanes of consecutive blocks read consecutive twiddles.
__host__ __device__ __forceinline__ int kb_tw_index(int log_n, int g, int x, bool fold) {
    const int j = g - (log_n - 5);
    return (1 << g) + (!fold || j <= 0 ? x : ((x & ((1 << j) - 1)) << (log_n - 5)) + (x >> j));
}
// Marks a 32-bit register value as changed.  A multiplicand that a loop reads in
// every pass is otherwise widened to 64 bits ahead of the loop and takes a
// register pair for its whole length.
template <class T>
__device__ __forceinline__ void kb_pin(T &x) {
    static_assert(sizeof(T) == 4, "32-bit registers");
    asm volatile("" : "+v"(x));
}
// constants of a reduction by folding at bit s, 2^(s-1) < p < 2^s: 2^s mod p with
// its Shoup companion, 2^64 - p, 2^64 - 2p, 2^64 - 4p, 2^(64+s) mod p, s
struct kb_fold {
    uint64_t w, ws, nq, n2q, n4q, wtop, s;
};
// (top 2^64 + F) 2^60 + L mod p for L < 2^60 and a value below 64 p^2 (WIDE, top <= 3)
// or 16 p^2 (top not read)
template <bool WIDE>
__device__ __forceinline__ uint64_t kb_fold_reduce(uint64_t F, uint32_t top, uint64_t L, const kb_fold &f) {
    if (f.s != 60) {  // uniform; then the value is below 2^124: top is 0 here
        const int s = (int)f.s;
        top = (uint32_t)(F >> (s + 4));
        F = (F << (60 - s)) + (L >> s);
        L &= (1ULL << s) - 1;
    }
    uint64_t r = kb_shoup4(F, f.w, f.ws, f.nq) + L;  // [0, 6p)
    r = kb_csub_sel(r, f.n4q);
    if constexpr (WIDE) {
        r = kb_mad32(top, (uint32_t)f.wtop, r) + ((uint64_t)kb_mul_lo32(top, (uint32_t)(f.wtop >> 32)) << 32);
        r = kb_csub_sel(r, f.n4q);  // [0, 7p) before
    }
    r = kb_csub_sel(r, f.n2q);
    return kb_csub_sel(r, f.nq);
}
