// One-pass NTT / INTT of a limb held in the registers of one workgroup, for primes
// near 2^60 (kb_fold_prime) and launches that give every CU a limb.
//
// The two-pass kernels read and write every limb twice and HBM bounds them at 3.8
// TB/s.  Here N / 32 threads hold 32 values each and run three register rounds, on
// index bits [top 5], [next 5], [low 5] of the element; the values change places
// through LDS in 32-bit halves, so 2^15 elements fit (132 KB with one pad word per
// 32).  Only the exchange between the first two layouts crosses waves: in the other
// two a wave holds the same 2048 consecutive elements and needs no barrier.  The
// first round's twiddles are uniform, the last round's are stored by (twiddle of
// the group, thread) and load coalesced.  A limb of 2^16 runs as two halves, one after the
// other: the forward transform's first level (the inverse's last) couples them and
// parks one half in the output, where each thread re-reads only its own words.
//
// At 2^16 bytes bound it: a large launch moves 1.95 times its limbs (the parked half, and
// twiddles that L2 does not hold beside the limbs) at 4.9 TB/s, a device copy's rate.  At 2^15
// it moves 3.2 to 3.5 TB/s: one workgroup per CU, whose loads, butterflies and stores follow each
// other; LDS conflicts are none and waits on LDS 2 to 5% of the waves' time at both.
#include "kbfv_internal.h"

namespace {

__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// barrier that orders LDS only: global stores and loads stay in flight
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// nothing moves across: bounds the registers in use
__device__ __forceinline__ void step_end() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// word `lane` from a uniform address
__device__ __forceinline__ uint64_t load_at(const uint64_t *p, uint32_t lane) {
    return *(const uint64_t *)((const char *)p + lane * 8u);
}
__device__ __forceinline__ void store_at(uint64_t *p, uint32_t lane, uint64_t v) {
    *(uint64_t *)((char *)p + lane * 8u) = v;
}

enum Layout { LA, LB, LC, LG };  // top, middle, low bits in registers; coalesced

// H = log2 of the elements held at a time
template <int H>
struct Reg {
    static constexpr int T = 1 << (H - 5);  // threads
    static constexpr int L = H - 10;        // low index bits of the B layout's thread
    static constexpr int WORDS = (1 << H) + (1 << (H - 5));
    template <Layout Y>
    __device__ static __forceinline__ int base() {  // LDS word of register 0
        const int t = threadIdx.x;
        if constexpr (Y == LA) return t + (t >> 5);
        if constexpr (Y == LB) return (t >> L) * ((1 << (H - 5)) + (1 << (H - 10))) + (t & ((1 << L) - 1));
        if constexpr (Y == LC) return t * 33;
        return (t >> 6) * 2112 + (t & 63) + ((t & 63) >> 5);
    }
    template <Layout Y>
    __device__ static constexpr int step(int i) {  // ... of register i from there
        if (Y == LA) return i * ((1 << (H - 5)) + (1 << (H - 10)));
        if (Y == LB) return (i << L) + (i >> (5 - L));
        if (Y == LC) return i;
        return i * 66;
    }
};

// From one layout to another, the low words and then the high words.  Across waves only
// to or from LA; there the barrier before the first write (from LA) or after the last
// read (to LA) keeps the exchange apart from its neighbours.
template <int H, Layout FROM, Layout TO>
__device__ __forceinline__ void exchange(uint64_t (&x)[32], uint32_t *lds) {
    using R = Reg<H>;
    const auto sync = [] {
        if constexpr (FROM == LA || TO == LA)
            lds_barrier();
        else
            wave_sync();
    };
    const int bf = R::template base<FROM>(), bt = R::template base<TO>();
    uint32_t lo[32];
    if constexpr (FROM == LA) sync();
#pragma unroll
    for (int i = 0; i < 32; ++i) lds[bf + R::template step<FROM>(i)] = (uint32_t)x[i];
    sync();
#pragma unroll
    for (int i = 0; i < 32; ++i) {
        lo[i] = lds[bt + R::template step<TO>(i)];
        asm volatile("" ::: "memory");  // no paired read: it would put two low words side by side
    }
    sync();
#pragma unroll
    for (int i = 0; i < 32; ++i) lds[bf + R::template step<FROM>(i)] = (uint32_t)(x[i] >> 32);
    sync();
#pragma unroll
    for (int i = 0; i < 32; ++i) {
        x[i] = ((uint64_t)lds[bt + R::template step<TO>(i)] << 32) | lo[i];
        asm volatile("" ::: "memory");
    }
    if constexpr (FROM != LA) sync();
}

struct half_args {
    const kbfv_tw *tab;
    uint64_t q, nq;
    uint32_t c, k28;
    int half;
};

// Twiddle m of level j of a round.  LOG = log2 of the limb, H of the half: level g of
// the half is level g + LOG - H of the limb and the half's number leads the group.
// A uniform twiddle's load waits for `dep`, lest all of them are made ahead.
template <int LOG, int H, Layout Y>
__device__ __forceinline__ kbfv_tw round_tw(const half_args &a, int j, int m, uint32_t dep) {
    constexpr int D = LOG - H;
    const auto at = [&](int uni, uint32_t lane) {
        return *(const kbfv_tw *)((const char *)(a.tab + uni) + lane * (uint32_t)sizeof(kbfv_tw));
    };
    if constexpr (Y == LA) {
        int zero = 0;
        asm volatile("" : "+s"(zero) : "v"(dep));
        return a.tab[(1 << (j + D)) + (a.half << j) + m + zero];
    } else if constexpr (Y == LB) {
        return at((1 << (5 + j + D)) + (a.half << (5 + j)) + m, (threadIdx.x >> Reg<H>::L) << j);
    } else {
        return at((1 << (H - 5 + j + D)) + (m << (LOG - 5)) + (a.half << (H - 5)), threadIdx.x);
    }
}

constexpr int RING = 4;   // twiddles in flight
constexpr int AHEAD = 8;  // words of the parked half in flight

// the round's k-th twiddle, k = 2^j - 1 + m (forward order)
constexpr int tw_level(int k) { return k < 1 ? 0 : k < 3 ? 1 : k < 7 ? 2 : k < 15 ? 3 : 4; }

// NL levels; LEV = transform levels done before, TOTAL of the transform.  Forward values
// are folded every fourth level, the inverse's sums every second; the last level's
// are left to the store.
enum { PLAIN, NINV, UNSCALED };  // the inverse's last level: sum times n^-1, or twiddle without it
template <int LOG, int H, Layout Y, int NL, int LEV, bool FWD, int LAST = PLAIN>
__device__ __forceinline__ void reg_round(uint64_t (&x)[32], const half_args &a, kbfv_tw last = {0, 0}) {
    constexpr int NT = (1 << NL) - 1;
    kbfv_tw ring[RING];
    // forward: levels 0 .. NL-1; inverse: NL-1 .. 0, twiddles in the reverse order
    const auto at = [&](int s, uint32_t dep) {
        const int k = FWD ? s : NT - 1 - s, j = tw_level(k);
        return round_tw<LOG, H, Y>(a, j, k - ((1 << j) - 1), dep);
    };
#pragma unroll
    for (int s = 0; s < RING && s < NT; ++s) ring[s] = at(s, (uint32_t)x[0]);
    int prev = 0;
#pragma unroll
    for (int s = 0; s < NT; ++s) {
        const int k = FWD ? s : NT - 1 - s, j = tw_level(k), m = k - ((1 << j) - 1), h = 16 >> j, i0 = m * 2 * h;
        const kbfv_tw w = LAST == UNSCALED && j == 0 ? last : ring[s % RING];
        if (s + RING < NT) ring[s % RING] = at(s + RING, (uint32_t)x[s ? prev : 0]);
        prev = i0 + h;
        const int lev = LEV + (FWD ? j : NL - 1 - j);
#pragma unroll
        for (int i = i0; i < i0 + h; ++i) {
            if constexpr (FWD) {
                ct_fold(x[i], x[i + h], w, a.c, a.k28);
                if (lev % 4 == 3 && lev != LOG - 1) {
                    x[i] = kb_sfold(x[i], a.c);
                    x[i + h] = kb_sfold(x[i + h], a.c);
                }
            } else if (lev % 2 == 1 && lev != LOG - 1) {
                gs_fold<true>(x[i], x[i + h], w, a.c, a.k28);
            } else {
                gs_fold<false>(x[i], x[i + h], w, a.c, a.k28);
                if (LAST == NINV && j == 0) x[i] = kb_fmul(x[i], last, a.c, a.k28, 0);
            }
            asm volatile("" : "+v"(x[i]), "+v"(x[i + h]));  // computed here, its twiddle done with
            if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// NOSC: N times the INTT, a non-negative representative up to 2^60 + 15c (below 2^60 + 2^32)
template <int LOG, bool FWD, bool NOSC>
__global__ void __launch_bounds__(1 << ((LOG > 15 ? 15 : LOG) - 5), 4)
    k_ntt_reg(const uint64_t *__restrict__ src, uint64_t *__restrict__ dst, const kbfv_tw *__restrict__ tw,
              const kbfv_tw *__restrict__ ninv_tab, const kbfv_tw *__restrict__ w1_tab,
              const uint64_t *__restrict__ mods, int mod0, int limbs, int polys, int batch, long sB, long sY, long sL,
              long dB, long dY, long dL, const uint64_t *__restrict__ src2, int half) {
    constexpr int H = LOG > 15 ? 15 : LOG, HALVES = 1 << (LOG - H), n = 1 << LOG, S = 1 << (H - 5);
    using R = Reg<H>;
    __shared__ uint32_t lds[R::WORDS];
    const int rows = limbs * polys * batch;
    const uint64_t *in;
    uint64_t *out;
    int m;
    const auto locate = [&](int row) {
        const int y = row % polys, bi = row / polys % batch, l = row / polys / batch;
        in = (bi < half ? src + bi * sB : src2 + (bi - half) * sB) + y * sY + l * sL;
        out = dst + bi * dB + y * dY + l * dL;
        m = mod0 + l;
    };
    half_args a;
    a.k28 = 1u << 28;
    asm volatile("" : "+s"(a.k28));
    uint64_t x[32];
    uint32_t t = threadIdx.x, g = (t >> 6) * 2048 + (t & 63);  // LA, LG: word of register 0
    const auto load_a = [&](const uint64_t *p) {
#pragma unroll
        for (int i = 0; i < 32; ++i) x[i] = load_at(p + i * S, t);
    };
    const auto load_g = [&](const uint64_t *p) {
#pragma unroll
        for (int i = 0; i < 32; ++i) x[i] = load_at(p + i * 64, g);
    };
    // One workgroup per CU (H = 15) takes rows in turn: a row's first loads are issued
    // right behind the stores of the one before.  (2040 rows of 2^15 360 us against 390
    // with a workgroup per row, of 2^16 855 against 903.)  Where several workgroups share
    // a CU they overlap by themselves: 2040 rows of 2^14 159 us against 165 in turn.
    int row = blockIdx.x;
    locate(row);
    if constexpr (FWD)
        load_a(in);
    else
        load_g(in + (HALVES - 1) * (n / 2));
    for (;;) {
        a.q = mods[m];
        a.tab = tw + ((size_t)m * 2 + (FWD ? 0 : 1)) * n;
        a.nq = 0 - a.q;
        a.c = kb_fold_c(a.q);
        asm volatile("" : "+s"(a.nq));
        if constexpr (FWD && HALVES == 1) {
#pragma unroll
            for (int i = 0; i < 32; ++i) x[i] = kb_ufold(x[i], a.c);
        }
        if constexpr (FWD && HALVES == 2) {
            // the limb's first level: the sums stay, the differences wait in the output
            const kbfv_tw w = a.tab[1];
            uint64_t v[AHEAD];
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) v[i] = load_at(in + i * S + n / 2, t);
#pragma unroll
            for (int i = 0; i < 32; ++i) {
                uint64_t b = kb_ufold(v[i % AHEAD], a.c);
                if (i + AHEAD < 32) v[i % AHEAD] = load_at(in + (i + AHEAD) * S + n / 2, t);
                x[i] = kb_ufold(x[i], a.c);
                ct_fold(x[i], b, w, a.c, a.k28);
                store_at(out + i * S + n / 2, t, b);
                step_end();
            }
        }
#pragma unroll 1
        for (int k = 0; k < HALVES; ++k) {
            if constexpr (HALVES > 1) {
                // no address outlives its half
                asm volatile("" : "+v"(t), "+v"(g), "+s"(in), "+s"(out));
            }
            if constexpr (FWD) {
                a.half = k;
                reg_round<LOG, H, LA, 5, LOG - H, true>(x, a);
                exchange<H, LA, LB>(x, lds);
                reg_round<LOG, H, LB, H - 10, LOG - H + 5, true>(x, a);
                exchange<H, LB, LC>(x, lds);
                reg_round<LOG, H, LC, 5, LOG - 5, true>(x, a);
#pragma unroll
                for (int i = 0; i < 32; ++i) x[i] = kb_fold_canon(x[i], a.q, a.nq, a.c);
                exchange<H, LC, LG>(x, lds);
#pragma unroll
                for (int i = 0; i < 32; ++i) store_at(out + k * (n / 2) + i * 64, g, x[i]);
                if (k + 1 < HALVES) load_a(out + n / 2);
            } else {
                a.half = HALVES - 1 - k;
#pragma unroll
                for (int i = 0; i < 32; ++i) x[i] = kb_ufold(x[i], a.c);
                exchange<H, LG, LC>(x, lds);
                reg_round<LOG, H, LC, 5, 0, false>(x, a);
                exchange<H, LC, LB>(x, lds);
                reg_round<LOG, H, LB, H - 10, 5, false>(x, a);
                exchange<H, LB, LA>(x, lds);
                if constexpr (HALVES == 1) {
                    reg_round<LOG, H, LA, 5, H - 5, false, NOSC ? UNSCALED : NINV>(x, a,
                                                                                   NOSC ? w1_tab[m] : ninv_tab[m]);
                } else {
                    reg_round<LOG, H, LA, 5, H - 5, false>(x, a);
                    if (k == 0) {
#pragma unroll
                        for (int i = 0; i < 32; ++i) store_at(out + i * S + n / 2, t, x[i]);
                        load_g(in);
                    }
                }
            }
        }
        if constexpr (!FWD) {
            const auto canon = [&](uint64_t v) {
                v = kb_ufold(v + (a.q << 3), a.c);
                return NOSC ? v : kb_csub_sel(v, a.nq);
            };
            if constexpr (HALVES == 1) {
#pragma unroll
                for (int i = 0; i < 32; ++i) store_at(out + i * S, t, canon(x[i]));
            } else {
                const kbfv_tw w = NOSC ? w1_tab[m] : a.tab[1], nv = ninv_tab[m];
                uint64_t v[AHEAD];
#pragma unroll
                for (int i = 0; i < AHEAD; ++i) v[i] = load_at(out + i * S + n / 2, t);
#pragma unroll
                for (int i = 0; i < 32; ++i) {
                    uint64_t b = v[i % AHEAD];
                    if (i + AHEAD < 32) v[i % AHEAD] = load_at(out + (i + AHEAD) * S + n / 2, t);
                    gs_fold<false>(x[i], b, w, a.c, a.k28);
                    if constexpr (!NOSC) x[i] = kb_fmul(x[i], nv, a.c, a.k28, 0);
                    store_at(out + i * S, t, canon(x[i]));
                    store_at(out + i * S + n / 2, t, canon(b));
                    step_end();
                }
            }
        }
        if constexpr (H < 15) break;
        row += gridDim.x;
        if (row >= rows) break;
        locate(row);
        asm volatile("" : "+v"(t), "+v"(g));
        if constexpr (FWD)
            load_a(in);
        else
            load_g(in + (HALVES - 1) * (n / 2));
    }
}

template <int LOG, bool FWD, bool NOSC>
int launch_reg(const kbfv_context *c, const uint64_t *src, uint64_t *dst, int mod0, int limbs, int polys, int batch,
               long sB, long sY, long sL, long dB, long dY, long dL, hipStream_t st, const uint64_t *src2, int half) {
    const long rows = (long)limbs * polys * batch, most = LOG < 15 ? rows : 256;
    KB_REQUIRE(rows < (1L << 30), "NTT grid too large");
    hipLaunchKernelGGL((k_ntt_reg<LOG, FWD, NOSC>), dim3((unsigned)(rows < most ? rows : most)), dim3(1 << ((LOG > 15 ? 15 : LOG) - 5)), 0,
                       st, src, dst, c->t.tw, c->t.ninv, c->t.inv_w1, c->t.mod, mod0, limbs, polys, batch, sB, sY, sL,
                       dB, dY, dL, src2, half);
    KB_LAUNCH_CHECK();
    return KBFV_OK;
}

}  // namespace

int kb_ntt_reg(const kbfv_context *c, int dir, bool noscale, const uint64_t *src, uint64_t *dst, int mod0, int limbs,
               int polys, int batch, long sB, long sY, long sL, long dB, long dY, long dL, hipStream_t st,
               const uint64_t *src2, int half) {
#define KB_REG(LOG_)                                                                                               \
    case LOG_:                                                                                                     \
        if (dir > 0)                                                                                               \
            return launch_reg<LOG_, true, false>(c, src, dst, mod0, limbs, polys, batch, sB, sY, sL, dB, dY, dL, st, \
                                                 src2, half);                                                      \
        if (noscale)                                                                                               \
            return launch_reg<LOG_, false, true>(c, src, dst, mod0, limbs, polys, batch, sB, sY, sL, dB, dY, dL, st, \
                                                 src2, half);                                                      \
        return launch_reg<LOG_, false, false>(c, src, dst, mod0, limbs, polys, batch, sB, sY, sL, dB, dY, dL, st,  \
                                              src2, half);
    switch (c->log_n) {
        KB_REG(12)
        KB_REG(13)
        KB_REG(14)
        KB_REG(15)
        KB_REG(16)
    }
#undef KB_REG
    return KBFV_EINVAL;
}
