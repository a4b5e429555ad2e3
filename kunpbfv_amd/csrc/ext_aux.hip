// External product of large batches through an auxiliary basis of 28-bit primes.
//
// The gadget sum over rows (extprod.hip) needs every digit polynomial transformed
// modulo every ciphertext prime: rows x qn 60-bit transforms per ciphertext.  As
// integers, though, the digits are below 2^w and the row limbs below q, so the
// coefficients of sum_r d_r * row_{r,h,l} stay below rows N 2^w q in size, and that
// integer is found from its residues modulo three or four primes below 2^28: each
// digit is transformed that many times, whatever the chain's length, with 32-bit
// arithmetic.  The row limbs are taken to the same basis once per call, the
// products are summed there, and each sum's residues come back as one integer
// (mixed radix), reduced modulo its q_l.  The result is the same canonical residue.
//
//   coef = INTT_Q(ct)                               (the caller)
//   per chunk of rows:  key = NTT_aux(INTT_Q(rows) mod p)
//                       dig = NTT_aux(digits of coef)
//                       acc += sum_r dig key
//   out = NTT_Q(mixed radix(INTT_aux(acc)))
//
// 32-bit butterflies keep lazy values below 16p: a Shoup product is two low and
// one high 32-bit multiply and lies in [0, 2p) for any operand, so a forward level
// adds 2p and one conditional subtraction of 8p (v_sub, v_min) opens every register
// round of four levels.  Products of two residues are below 2^56: a row chunk
// accumulates with one v_mad_u64_u32 per product and reduces once.
//
// 128 products at N = 2^16, 28 primes, base 2^20 (168 rows, four auxiliary primes):
// 81 ms against 422 ms through 4704 60-bit transforms per ciphertext; of that the row
// products 31.6, the transforms of digits and rows in the basis 29.7, the way back 9.5, the
// 60-bit transforms of ciphertexts, rows and results 10.2.  The row products hold seven waves
// per CU and issue 0.42 VALU instructions per clock and CU, half of what multiply-adds
// reach; a fifth of the waves' time is spent waiting, a third of that on LDS.
#include <algorithm>
#include <cmath>

#include "kbfv_internal.h"
#include "kbfv_ops.h"

namespace {

__device__ __forceinline__ uint32_t shoup32(uint32_t x, uint2 w, uint32_t p) {
    return x * w.x - __umulhi(x, w.y) * p;  // [0, 2p)
}
__device__ __forceinline__ uint32_t csub32(uint32_t x, uint32_t m) { return min(x, x - m); }
// any x to [0, p); one = (1, floor(2^32 / p))
__device__ __forceinline__ uint32_t canon32(uint32_t x, uint32_t one_s, uint32_t p) {
    return csub32(x - __umulhi(x, one_s) * p, p);
}

template <int LOG_N, bool COLUMN>
struct Geo32 {
    static constexpr int LOG_C0 = (LOG_N + 1) / 2;  // the column pass's levels
    static constexpr int LOG_S = COLUMN ? LOG_C0 : LOG_N - LOG_C0;
    static constexpr int S = 1 << LOG_S;
    static constexpr int LOG_T = COLUMN && LOG_N > 12 ? 13 : 12;  // column rows of 32 words and more
    static constexpr int TILE = 1 << LOG_T, C = TILE / S, T = TILE / 16;
    static constexpr int G0 = COLUMN ? 0 : LOG_N - LOG_S;
    static constexpr int STRIDE = 1 << (LOG_N - LOG_S);  // between a column's elements
    static constexpr int WORDS = COLUMN ? TILE : TILE + TILE / 16;
    static constexpr int LR0 = 4, LR1 = LOG_S - 4;
    static_assert(LR1 >= 1 && LR1 <= 4, "two register rounds");
    __device__ static __forceinline__ int addr(int c, int k) {
        if constexpr (COLUMN) return k * C + c;
        const int e = c * S + k;
        return e + (e >> 4);
    }
};

// LR levels from pass level LAM0 on 2^LR values per group, 16 values per thread;
// ld(c, k) / st(c, k, x) address element k of sub-transform c of the tile, cg is the
// first sub-transform's global number
template <class G, bool FWD, int LR, int LAM0, class LD, class ST>
__device__ __forceinline__ void round32(const uint2 *__restrict__ tab, uint32_t p, uint32_t one_s, int cg, LD ld, ST st) {
    constexpr int RR = 1 << LR, NG = 16 >> LR, Bs = G::S >> LAM0, d = Bs >> LR;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        const int grp = threadIdx.x + g * G::T;
        int c, u;
        if constexpr (G::G0 == 0) {
            c = grp % G::C;
            u = grp / G::C;
        } else {
            u = grp % (G::S >> LR);
            c = grp / (G::S >> LR);
        }
        const int kbase = (u / d) * Bs + u % d;
        uint32_t x[RR];
#pragma unroll
        for (int i = 0; i < RR; ++i) x[i] = ld(c, kbase + i * d);
        auto tw = [&](int j, int m) {
            const int lam = LAM0 + j;
            const int sub = ((kbase >> (G::LOG_S - LAM0)) << j) + m;
            return G::G0 == 0 ? tab[(1 << lam) + sub] : tab[(1 << (lam + G::G0)) + ((cg + c) << lam) + sub];
        };
        if constexpr (FWD) {
#pragma unroll
            for (int j = 0; j < LR; ++j) {
                const int h = RR >> (j + 1);
#pragma unroll
                for (int m = 0; m < (1 << j); ++m) {
                    const uint2 w = tw(j, m);
#pragma unroll
                    for (int i = m * 2 * h; i < m * 2 * h + h; ++i) {
                        uint32_t a = x[i];
                        if (j == 0) a = csub32(a, 8 * p);
                        const uint32_t t = shoup32(x[i + h], w, p);
                        x[i] = a + t;
                        x[i + h] = a + 2 * p - t;
                    }
                }
            }
        } else {
            // inputs below p; the sums double, the products start again below 2p
#pragma unroll
            for (int j = LR - 1; j >= 0; --j) {
                const int h = RR >> (j + 1);
                const uint32_t bound = p << (LR - 1 - j);
#pragma unroll
                for (int m = 0; m < (1 << j); ++m) {
                    const uint2 w = tw(j, m);
#pragma unroll
                    for (int i = m * 2 * h; i < m * 2 * h + h; ++i) {
                        const uint32_t a = x[i], b = x[i + h];
                        x[i] = a + b;
                        x[i + h] = shoup32(a + bound - b, w, p);
                    }
                }
            }
        }
#pragma unroll
        for (int i = 0; i < RR; ++i) st(c, kbase + i * d, x[i]);
    }
}

// Where a transform's elements live.  The products read, per 64 coefficients, all
// rows (or outputs) of one prime, so those lie together: element e of the
// transform (o, i, k) is at o so + i si + k sk + (e / 64) ts + e % 64.
struct lay32 {
    int inner;  // transforms y = o inner + i
    long so, si, sk, ts;
    __device__ __forceinline__ long base(long y, int k) const { return (y / inner) * so + (y % inner) * si + k * sk; }
    __device__ __forceinline__ long at(int e) const { return (e >> 6) * ts + (e & 63); }
};

// ---------------------------------------------------------------- forward
// first pass: columns of the source limb taken into the auxiliary basis.
// DIG: source y = (ciphertext, row): digit `row % nd` of limb `row / nd` of the
// coefficient-form ciphertext; else the residue of 60-bit limb y.  Transform
// (y, k) -> dst, below 16p.  The prime varies fastest, then (DIG)
// the digit, so the workgroups that read one source tile run together.
template <int LOG_N, bool DIG>
__global__ void __launch_bounds__((Geo32<LOG_N, true>::T))
    k32_fwd_col(const uint64_t *__restrict__ src, uint32_t *__restrict__ dst, const uint2 *__restrict__ tw,
                const kb_aux_mod *__restrict__ mods, lay32 lay, int np, int rc, int r0, int nd, int bits, long ct_stride) {
    using G = Geo32<LOG_N, true>;
    __shared__ uint32_t tile[G::WORDS];
    constexpr int groups = G::STRIDE / G::C;
    const int k = blockIdx.x % np;
    int b = blockIdx.x / np;
    const uint64_t *in;
    long y;
    int shift = 0, grp;
    if constexpr (DIG) {
        const int r = b % rc;
        b /= rc;
        grp = b % groups;
        const int ct = b / groups, row = r0 + r;
        in = src + ct * ct_stride + ((long)(row / nd) << LOG_N);
        shift = bits * (row % nd);
        y = (long)ct * rc + r;
    } else {
        grp = b % groups;
        y = b / groups;
        in = src + (y << LOG_N);
    }
    const kb_aux_mod md = mods[k];
    const uint32_t p = md.p;
    const uint2 *tab = tw + ((size_t)k * 2 << LOG_N);
    const int c0 = grp * G::C;
    in += c0;
    uint32_t *out = dst + lay.base(y, k);
    const uint64_t mask = (1ULL << bits) - 1;
    round32<G, true, G::LR0, 0>(
        tab, p, md.one_s, c0,
        [&](int c, int kk) -> uint32_t {
            const uint64_t v = in[kk * G::STRIDE + c];
            if constexpr (DIG) return (uint32_t)((v >> shift) & mask);
            return shoup32((uint32_t)(v >> 32), make_uint2(md.r32, md.r32_s), p) + (uint32_t)v -
                   __umulhi((uint32_t)v, md.one_s) * p;
        },
        [&](int c, int kk, uint32_t x) { tile[G::addr(c, kk)] = x; });
    __syncthreads();
    round32<G, true, G::LR1, G::LR0>(
        tab, p, md.one_s, c0, [&](int c, int kk) { return tile[G::addr(c, kk)]; },
        [&](int c, int kk, uint32_t x) { out[lay.at(kk * G::STRIDE + c0 + c)] = x; });
}

// the tile's rows from global memory in 16-byte loads
template <class G>
__device__ __forceinline__ void rows_in(uint32_t *tile, const uint32_t *__restrict__ g, const lay32 &lay) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int e = (threadIdx.x + j * G::T) * 4;
        const kb_u32x4 v = *(const kb_u32x4 *)(g + lay.at(e));
        uint32_t *t = tile + e + (e >> 4);
        t[0] = v.x, t[1] = v.y, t[2] = v.z, t[3] = v.w;
    }
}

// second pass in place, one transform per blockIdx.x / groups; canonical results
template <int LOG_N>
__global__ void __launch_bounds__((Geo32<LOG_N, false>::T))
    k32_fwd_row(uint32_t *__restrict__ data, const uint2 *__restrict__ tw, const kb_aux_mod *__restrict__ mods, lay32 lay,
                int np) {
    using G = Geo32<LOG_N, false>;
    __shared__ uint32_t tile[G::WORDS];
    constexpr int groups = (1 << LOG_N) / G::TILE;
    const long tr = blockIdx.x / groups;
    const int grp = blockIdx.x % groups, k = (int)(tr % np);
    const kb_aux_mod md = mods[k];
    const uint2 *tab = tw + ((size_t)k * 2 << LOG_N);
    uint32_t *g = data + lay.base(tr / np, k) + (long)grp * (G::TILE / 64) * lay.ts;
    auto ld = [&](int c, int kk) { return tile[G::addr(c, kk)]; };
    auto st = [&](int c, int kk, uint32_t x) { tile[G::addr(c, kk)] = x; };
    rows_in<G>(tile, g, lay);
    __syncthreads();
    round32<G, true, G::LR0, 0>(tab, md.p, md.one_s, grp * G::C, ld, st);
    __syncthreads();
    round32<G, true, G::LR1, G::LR0>(tab, md.p, md.one_s, grp * G::C, ld, st);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int e = (threadIdx.x + j * G::T) * 4;
        const uint32_t *t = tile + e + (e >> 4);
        uint32_t v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = canon32(t[i], md.one_s, md.p);
        *(kb_u32x4 *)(g + lay.at(e)) = kb_u32x4{v[0], v[1], v[2], v[3]};
    }
}

// ---------------------------------------------------------------- inverse, without n^-1
template <int LOG_N>
__global__ void __launch_bounds__((Geo32<LOG_N, false>::T))
    k32_inv_row(uint32_t *__restrict__ data, const uint2 *__restrict__ tw, const kb_aux_mod *__restrict__ mods, lay32 lay,
                int np) {
    using G = Geo32<LOG_N, false>;
    __shared__ uint32_t tile[G::WORDS];
    constexpr int groups = (1 << LOG_N) / G::TILE;
    const long tr = blockIdx.x / groups;
    const int grp = blockIdx.x % groups, k = (int)(tr % np);
    const kb_aux_mod md = mods[k];
    const uint2 *tab = tw + (((size_t)k * 2 + 1) << LOG_N);
    uint32_t *g = data + lay.base(tr / np, k) + (long)grp * (G::TILE / 64) * lay.ts;
    auto ld = [&](int c, int kk) { return tile[G::addr(c, kk)]; };
    auto st = [&](int c, int kk, uint32_t x) { tile[G::addr(c, kk)] = canon32(x, md.one_s, md.p); };
    rows_in<G>(tile, g, lay);
    __syncthreads();
    round32<G, false, G::LR1, G::LR0>(tab, md.p, md.one_s, grp * G::C, ld, st);
    __syncthreads();
    round32<G, false, G::LR0, 0>(tab, md.p, md.one_s, grp * G::C, ld, st);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int e = (threadIdx.x + j * G::T) * 4;
        const uint32_t *t = tile + e + (e >> 4);
        *(kb_u32x4 *)(g + lay.at(e)) = kb_u32x4{t[0], t[1], t[2], t[3]};
    }
}

// last pass in place; any 32-bit representative (the mixed radix takes it so)
template <int LOG_N>
__global__ void __launch_bounds__((Geo32<LOG_N, true>::T))
    k32_inv_col(uint32_t *__restrict__ data, const uint2 *__restrict__ tw, const kb_aux_mod *__restrict__ mods, lay32 lay,
                int np) {
    using G = Geo32<LOG_N, true>;
    __shared__ uint32_t tile[G::WORDS];
    constexpr int groups = G::STRIDE / G::C;
    const long tr = blockIdx.x / groups;
    const int c0 = (blockIdx.x % groups) * G::C, k = (int)(tr % np);
    const kb_aux_mod md = mods[k];
    const uint2 *tab = tw + (((size_t)k * 2 + 1) << LOG_N);
    uint32_t *g = data + lay.base(tr / np, k);
    round32<G, false, G::LR1, G::LR0>(
        tab, md.p, md.one_s, c0, [&](int c, int kk) { return g[lay.at(kk * G::STRIDE + c0 + c)]; },
        [&](int c, int kk, uint32_t x) { tile[G::addr(c, kk)] = canon32(x, md.one_s, md.p); });
    __syncthreads();
    round32<G, false, G::LR0, 0>(
        tab, md.p, md.one_s, c0, [&](int c, int kk) { return tile[G::addr(c, kk)]; },
        [&](int c, int kk, uint32_t x) { g[lay.at(kk * G::STRIDE + c0 + c)] = x; });
}

// ---------------------------------------------------------------- row products
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
constexpr int AM_MINW = 5, AM_MAXW = 8;  // waves of a workgroup
constexpr int AM_MAXR = 56;              // rows held in registers
constexpr int AM_CT = 2;                 // ciphertexts staged together

// acc[ct][k][t][hl][n] (+)= sum_{r < rc} dig[ct][k][t][r][n] key[k][t][hl][r][n] mod
// p_k, n in the 64-coefficient tile t.  A
// thread holds the rows of two outputs hl of its coefficient and walks the
// batch; the digits pass through a double-buffered LDS tile that the workgroup's
// waves (other hl) read.  A lane fetches 16 bytes of it, four rows per wave and
// instruction, into registers before the products and stores them after.
template <int MAXR>
__global__ void __launch_bounds__(64 * AM_MAXW)
    k32_mac(const uint32_t *__restrict__ dig, const uint32_t *__restrict__ key, uint32_t *__restrict__ acc,
            const kb_aux_mod *__restrict__ mods, int np, int hls, int rc, int first, int log_n, int batch) {
    constexpr int PF = (AM_CT * MAXR + 4 * AM_MINW - 1) / (4 * AM_MINW);
    constexpr int ROWS = AM_CT * MAXR + 4;
    __shared__ alignas(16) uint32_t xs[2][ROWS][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int waves = blockDim.x >> 6;
    const int pairs = hls / 2, groups = (pairs + waves - 1) / waves;
    const int tiles = 1 << (log_n - 6);
    // the groups of one tile are 8 workgroups apart: the same XCD
    const int r8 = blockIdx.x / (8 * groups), q8 = blockIdx.x % (8 * groups);
    const int tg = r8 * 8 + q8 % 8;
    const int pair = (q8 / 8) * waves + wave;
    const bool active = pair < pairs;
    const int hl = 2 * min(pair, pairs - 1);
    const int k = tg / tiles;
    const kb_aux_mod md = mods[k];
    uint32_t k0[MAXR], k1[MAXR];
    {
        const uint32_t *kp = key + ((long)tg * hls + hl) * rc * 64 + lane;  // tg = k tiles + t
#pragma unroll
        for (int r = 0; r < MAXR; ++r) {
            const uint32_t a = kp[min(r, rc - 1) * 64], b = kp[(rc + min(r, rc - 1)) * 64];
            k0[r] = r < rc ? a : 0;
            k1[r] = r < rc ? b : 0;
        }
    }
    // row j of a stage is row j % rc of ciphertext j / rc; rows past its end repeat the last
    const long cts = (long)np * tiles * 64;  // of one row or output per ciphertext
    const uint32_t *src = dig + (long)tg * rc * 64 + 4 * (lane & 15);
    const int jl = 4 * wave + (lane >> 4);
    u32x4 pf[PF];
    auto fetch = [&](int ct) {
#pragma unroll
        for (int u = 0; u < PF; ++u) {
            const int j = min(jl + 4 * waves * u, AM_CT * rc - 1);
            const int c = j >= rc ? 1 : 0;
            pf[u] = *(const kb_u32x4 *)(src + (long)min(ct + c, batch - 1) * rc * cts + (j - (c ? rc : 0)) * 64);
        }
    };
    auto commit = [&](int buf) {
#pragma unroll
        for (int u = 0; u < PF; ++u)
            *(u32x4 *)&xs[buf][min(jl + 4 * waves * u, ROWS - 1)][4 * (lane & 15)] = pf[u];  // extra rows into one unused
    };
    static_assert(AM_CT == 2, "two ciphertexts per stage");
    fetch(0);
    commit(0);
    __syncthreads();
    uint32_t *a = acc + ((long)tg * hls + hl) * 64 + lane;
    const long an = hls * cts;
    for (int ct = 0, buf = 0; ct < batch; ct += AM_CT, buf ^= 1, a += AM_CT * an) {
        fetch(min(ct + AM_CT, batch - 1));
        const bool two = ct + 1 < batch;
        uint32_t old[2][2] = {};
        if (!first) {
            old[0][0] = a[0], old[0][1] = a[64];
            if (two) old[1][0] = a[an], old[1][1] = a[an + 64];
        }
        uint64_t s[2][2] = {};
#pragma unroll
        for (int r = 0; r < MAXR; ++r) kb_pin(k0[r]), kb_pin(k1[r]);
        const uint32_t *x0 = &xs[buf][0][lane], *x1 = &xs[buf][rc][lane];
        // four rows ahead of the products; rows past rc meet zero keys
        uint32_t nx[2][4];
#pragma unroll
        for (int i = 0; i < 4; ++i) nx[0][i] = x0[64 * i], nx[1][i] = x1[64 * i];
#pragma unroll
        for (int r = 0; r < MAXR; r += 4) {
            uint32_t u[4], v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) u[i] = nx[0][i], v[i] = nx[1][i];
            if (r + 4 < MAXR) {
#pragma unroll
                for (int i = 0; i < 4; ++i) nx[0][i] = x0[64 * (r + 4 + i)], nx[1][i] = x1[64 * (r + 4 + i)];
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                kb_mad(s[0][0], u[i], k0[r + i]);
                kb_mad(s[0][1], u[i], k1[r + i]);
                kb_mad(s[1][0], v[i], k0[r + i]);
                kb_mad(s[1][1], v[i], k1[r + i]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int o = 0; o < 2; ++o) {
                const uint32_t hi = (uint32_t)(s[c][o] >> 32), lo = (uint32_t)s[c][o];
                const uint32_t v = shoup32(hi, make_uint2(md.r32, md.r32_s), md.p) + lo - __umulhi(lo, md.one_s) * md.p +
                                   old[c][o];  // [0, 5p)
                if (active && (c == 0 || two)) a[c * an + o * 64] = canon32(v, md.one_s, md.p);
            }
        commit(buf ^ 1);
        __syncthreads();
    }
}

// ---------------------------------------------------------------- back to the ciphertext primes
// acc [ct][k][t][hl][64] (N times the coefficients' residues) -> out [ct][hl][N], the
// integer's residue modulo q_l, hl = h qn + l
template <int NP>
__global__ void __launch_bounds__(256)
    k32_lift(const uint32_t *__restrict__ acc, uint64_t *__restrict__ out, const kb_aux_mod *__restrict__ mods,
             const kb_aux_mix *__restrict__ mix, const kb_aux_lift *__restrict__ lift, int qn, int hls, int log_n) {
    const long N = 1L << log_n;
    const int n = blockIdx.x * 256 + threadIdx.x;
    const int hl = blockIdx.y;
    const long y = (long)blockIdx.z * hls + hl;
    const uint32_t *a = acc + ((long)blockIdx.z * NP << log_n) * hls + ((long)(n >> 6) * hls + hl) * 64 + (n & 63);
    uint32_t v[NP];
#pragma unroll
    for (int k = 0; k < NP; ++k) {
        const uint32_t p = mods[k].p;
        uint32_t x = shoup32(a[k * N * hls], mix->own[k], p);
#pragma unroll
        for (int j = 0; j < k; ++j) x = csub32(x + 2 * p - shoup32(v[j], mix->other[k][j], p), 2 * p);
        v[k] = csub32(x, p);
    }
    const bool neg = v[NP - 1] > mods[NP - 1].p / 2;
    const kb_aux_lift &c = lift[hl >= qn ? hl - qn : hl];
    // v0 + v1 p0 (below 2^56), then the higher digits, each product in [0, 4q)
    uint64_t r = kb_shoup4((uint64_t)v[0] + (uint64_t)v[1] * mods[0].p, 1, c.one_s, c.nq);
    r = kb_csub_sel(r, c.n2q);
    r += kb_shoup4(v[2], c.w2, c.w2_s, c.nq);
    if constexpr (NP == 4) {
        r = kb_csub_sel(kb_csub_sel(r, c.n4q), c.n2q);
        r += kb_shoup4(v[3], c.w3, c.w3_s, c.nq);
    }
    r = kb_csub_sel(r, c.n4q);
    r += neg ? (NP == 4 ? c.neg4 : c.neg3) : 0;
    r = kb_csub_sel(r, c.n4q);
    r = kb_csub_sel(r, c.n2q);
    out[(y << log_n) + n] = kb_csub_sel(r, c.nq);
}

template <int LOG_N>
struct Aux {
    using GC = Geo32<LOG_N, true>;
    using GR = Geo32<LOG_N, false>;
    // workgroups of a pass over `transforms` polynomials
    template <class G>
    static int grid(long transforms, dim3 *g) {
        const long blocks = transforms * ((1 << LOG_N) / G::TILE);
        KB_REQUIRE(blocks < (1L << 31), "auxiliary NTT grid too large");
        *g = dim3((unsigned)blocks);
        return KBFV_OK;
    }
    // src: coefficient-form ciphertexts, of which rows r0 .. r0+rc-1 are digits, or limbs
    static int forward(const kbfv_context *c, bool digits, const uint64_t *src, uint32_t *dst, const lay32 &lay, int polys,
                       int np, int rc, int r0, int nd, int bits, hipStream_t st) {
        dim3 gc, gr;
        KB_TRY(grid<GC>((long)polys * np, &gc));
        KB_TRY(grid<GR>((long)polys * np, &gr));
        if (digits)
            hipLaunchKernelGGL((k32_fwd_col<LOG_N, true>), gc, dim3(GC::T), 0, st, src, dst, c->t.aux_tw, c->t.aux_mod,
                               lay, np, rc, r0, nd, bits, 2L * c->qn * c->n);
        else
            hipLaunchKernelGGL((k32_fwd_col<LOG_N, false>), gc, dim3(GC::T), 0, st, src, dst, c->t.aux_tw, c->t.aux_mod,
                               lay, np, 1, 0, 1, 0, 0L);
        KB_LAUNCH_CHECK();
        hipLaunchKernelGGL(k32_fwd_row<LOG_N>, gr, dim3(GR::T), 0, st, dst, c->t.aux_tw, c->t.aux_mod, lay, np);
        KB_LAUNCH_CHECK();
        return KBFV_OK;
    }
    static int inverse(const kbfv_context *c, uint32_t *d, const lay32 &lay, int polys, int np, hipStream_t st) {
        dim3 gc, gr;
        KB_TRY(grid<GC>((long)polys * np, &gc));
        KB_TRY(grid<GR>((long)polys * np, &gr));
        hipLaunchKernelGGL(k32_inv_row<LOG_N>, gr, dim3(GR::T), 0, st, d, c->t.aux_tw, c->t.aux_mod, lay, np);
        KB_LAUNCH_CHECK();
        hipLaunchKernelGGL(k32_inv_col<LOG_N>, gc, dim3(GC::T), 0, st, d, c->t.aux_tw, c->t.aux_mod, lay, np);
        KB_LAUNCH_CHECK();
        return KBFV_OK;
    }
};

int aux_mac(const kbfv_context *c, const uint32_t *dig, const uint32_t *key, uint32_t *acc, int np, int rc, bool first,
            int batch, hipStream_t st) {
    const int hls = 2 * c->qn, groups = (c->qn + AM_MAXW - 1) / AM_MAXW;
    const int waves = std::max((c->qn + groups - 1) / groups, AM_MINW);
    const long blocks = (long)((c->qn + waves - 1) / waves) * np * (c->n / 64);
    KB_REQUIRE(blocks < (1L << 31), "row product grid too large");
#define KB_AM(MR)                                                                                                 \
    if (rc <= MR) {                                                                                               \
        hipLaunchKernelGGL(k32_mac<MR>, dim3((unsigned)blocks), dim3(64 * waves), 0, st, dig, key, acc,           \
                           c->t.aux_mod, np, hls, rc, (int)first, c->log_n, batch);                               \
        KB_LAUNCH_CHECK();                                                                                        \
        return KBFV_OK;                                                                                           \
    }
    KB_AM(8)
    KB_AM(16)
    KB_AM(28)
    KB_AM(AM_MAXR)
#undef KB_AM
    kb_set_error("row chunk out of range");
    return KBFV_EINVAL;
}

template <int LOG_N>
int run(const kbfv_context *c, const uint64_t *rgsw, const uint64_t *coef, uint64_t *out, uint64_t *dig_ws, int batch,
        int rows, int nd, int bits, int np, hipStream_t st) {
    using A = Aux<LOG_N>;
    const long N = c->n, hls = 2L * c->qn;
    // dig_ws holds 8 qn batch limbs: the accumulators, then a chunk's digits; the
    // output holds 2 qn batch: a chunk's rows in the basis, then the limbs on their
    // way there (half a limb per residue polynomial)
    uint32_t *acc = (uint32_t *)dig_ws;
    uint32_t *dig = acc + hls * np * batch * N;
    const long dig_polys = 16L * c->qn * batch - hls * np * batch;  // 32-bit polynomials left
    uint32_t *key = (uint32_t *)out;
    const int rc_max = kb_ext_aux_rows(c, batch, np);
    KB_REQUIRE(rc_max >= 1 && (long)rc_max * np * batch <= dig_polys, "auxiliary workspace too small");
    const int chunks = (rows + rc_max - 1) / rc_max, rc_even = (rows + chunks - 1) / chunks;
    for (int r0 = 0; r0 < rows; r0 += rc_even) {
        const int rc = std::min(rc_even, rows - r0);
        uint64_t *tmp = out + ((long)rc_even * hls * np * N + 1) / 2;
        const int sub = (int)std::max(1L, (hls * batch - (rc_even * hls * np + 1) / 2) / hls);
        for (int s0 = 0; s0 < rc; s0 += sub) {
            const int sn = std::min(sub, rc - s0);
            KB_TRY(kb_ntt(c, -1, rgsw + (r0 + s0) * hls * N, tmp, c->oQ, c->qn, 2 * sn, 1, 0, c->qn * N, N, 0, c->qn * N,
                          N, st));
            const lay32 kl{(int)hls, 64, rc * 64L, rc * hls * N, rc * hls * 64};
            KB_TRY(A::forward(c, false, tmp, key + s0 * 64, kl, (int)(sn * hls), np, 1, 0, 1, 0, st));
        }
        const lay32 dl{rc, (long)np * rc * N, 64, rc * N, rc * 64L};
        KB_TRY(A::forward(c, true, coef, dig, dl, batch * rc, np, rc, r0, nd, bits, st));
        KB_TRY(aux_mac(c, dig, key, acc, np, rc, r0 == 0, batch, st));
    }
    const lay32 al{(int)hls, np * hls * N, 64, hls * N, hls * 64};
    KB_TRY(A::inverse(c, acc, al, (int)(batch * hls), np, st));
    for (int b0 = 0; b0 < batch; b0 += 65535) {  // grid z
        const dim3 grid((unsigned)(N / 256), (unsigned)hls, (unsigned)std::min(batch - b0, 65535));
        const uint32_t *a = acc + hls * np * b0 * N;
        uint64_t *o = out + hls * b0 * N;
        if (np == 3)
            hipLaunchKernelGGL(k32_lift<3>, grid, dim3(256), 0, st, a, o, c->t.aux_mod, c->t.aux_mix, c->t.aux_lift,
                               c->qn, (int)hls, c->log_n);
        else
            hipLaunchKernelGGL(k32_lift<4>, grid, dim3(256), 0, st, a, o, c->t.aux_mod, c->t.aux_mix, c->t.aux_lift,
                               c->qn, (int)hls, c->log_n);
        KB_LAUNCH_CHECK();
    }
    return kb_ntt_inplace(c, +1, out, c->oQ, c->qn, 2 * batch, st);
}

}  // namespace

// rows of a chunk: its digits fit what the accumulators leave of the digit
// workspace, its rows in the basis the output less an eighth for the limbs on their
// way there (with room for one row's only, 17 ciphertexts took 1.31 ms, 16 0.82)
int kb_ext_aux_rows(const kbfv_context *c, int batch, int np) {
    const long hls = 2L * c->qn;
    const long by_dig = (16L * c->qn - hls * np) / np;                 // per ciphertext
    const long by_key = 2L * (batch - (batch + 7) / 8) / np;
    return (int)std::min(std::min(by_dig, by_key), (long)AM_MAXR);
}

// primes the sum needs, 0 if the auxiliary basis cannot hold it
int kb_ext_aux_primes(const kbfv_context *c, int rows, int bits) {
    if (!c->t.aux_tw || bits > 27) return 0;
    uint64_t qmax = 0;
    for (int i = 0; i < c->qn; ++i) qmax = std::max(qmax, c->mod[c->oQ + i]);
    // size of a coefficient's sum; the sign is read off the top digit of the
    // mixed radix, so the basis is four times as wide
    const double need = std::log2((double)rows) + c->log_n + bits + std::log2((double)qmax) + 2.01;
    double have = 0;
    for (int k = 0; k < KB_AUX_PRIMES; ++k) {
        have += std::log2((double)c->aux_p[k]);
        if (k >= 2 && need < have) return k + 1;
    }
    return 0;
}

int kb_external_product_aux(const kbfv_context *c, const uint64_t *rgsw, const uint64_t *coef, uint64_t *out,
                            uint64_t *dig_ws, int batch, int rows, int nd, int bits, int np, hipStream_t st) {
    switch (c->log_n) {
        case 12: return run<12>(c, rgsw, coef, out, dig_ws, batch, rows, nd, bits, np, st);
        case 13: return run<13>(c, rgsw, coef, out, dig_ws, batch, rows, nd, bits, np, st);
        case 14: return run<14>(c, rgsw, coef, out, dig_ws, batch, rows, nd, bits, np, st);
        case 15: return run<15>(c, rgsw, coef, out, dig_ws, batch, rows, nd, bits, np, st);
        default: return run<16>(c, rgsw, coef, out, dig_ws, batch, rows, nd, bits, np, st);
    }
}
