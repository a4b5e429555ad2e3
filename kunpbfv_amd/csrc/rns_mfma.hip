// HPS base conversion and scale-and-round over long chains as int8 MFMA products.
//
// The same functions as rns_conv.hip (include/poly_arithmetic.cuh:1139-1178,
// :1263-1317), for chains whose products are worth the matrix cores.  The
// product runs transposed, out^T[j][p] = sum_i M^T[j][i] X^T[i][p]: the matrix is
// the MFMA A operand (rows = output limbs j), the coefficients the B operand
// (columns = positions p), in the expanded form of kbfv_mfma.h: K runs over
// (i, u) and the products split into 8 digit passes.
//
// One workgroup per CU keeps the whole expanded matrix (64 KB at 32 x 32) in LDS
// for its lifetime; its waves walk tiles of 64 positions on their own, with no
// barrier after the first.  A wave first takes one position per lane: coalesced
// loads, the Shoup products and the double estimate in input order in
// registers, then hands the digits through an 8-row LDS strip of its own into
// the B layout.  The overflow count alpha (and scale-and-round's nu, in two
// 32-bit halves) rides as further K rows.  Per output, the eight biased
// accumulators combine into four 32-bit words; V = sum_k W_k 2^(16k) + const is
// below 2^80 and positive, so its top 32 bits times floor(2^(80+S)/p) give
// the quotient or one less, and one conditional subtraction finishes.
//
// Bound by VALU issue (half of it the inputs' Shoup products and estimate) beside
// the HBM traffic; two waves per SIMD with the next tile's inputs in registers
// beat three without.  28 primes, 128 polynomials at N = 2^16: Q -> R 1.15 ms, R ->
// Q 1.05 ms, scale-and-round 1.45 ms (1.52, 1.45 and 1.65 ms with single-wave
// workgroups that read the matrix from L2 and passed the words through LDS);
// one read and write of each limb takes 0.77, 0.77 and 1.15 ms at 5 TB/s.
#include <algorithm>

#include "kbfv_internal.h"
#include "kbfv_mfma.h"
#include "kbfv_ops.h"

namespace {

constexpr int RG_WAVES = 8;      // 2 per SIMD: registers for the next tile's inputs
constexpr int RG_MT = 4;         // 16-position tiles per wave
constexpr int RG_POS = 64;       // positions per wave (one per lane in the estimate)
constexpr int RG_ROW = 72;       // staged row in words: lane groups g, g + 1 read 32 banks apart
constexpr int RG_CUS = 256;

template <int KC, int NJ, bool SR>
__global__ void __launch_bounds__(64 * RG_WAVES, RG_WAVES / 4)
    k_rns_gemm(const uint64_t *__restrict__ x, long in_stride, uint64_t *__restrict__ y, long out_stride,
               const uint64_t *__restrict__ mat, const kb_conv_in *__restrict__ inp, const double *__restrict__ est, int in_n, int out_n, int log_n,
               int ntiles) {
    // rows from PAD on may be padding or the estimate's (the chunk count is the least that holds them)
    constexpr int PAD = 8 * (KC - 1) - (SR ? 1 : 0);
    constexpr int KP = 8 * KC, MW = NJ * 8 * KC * 64;  // 16-byte words of the matrix
    __shared__ kb_v4i smat[MW];
    __shared__ uint64_t scst[16 * NJ * KB_MX_ROW];
    __shared__ uint64_t stage[RG_WAVES][8 * RG_ROW];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int p16 = lane & 15, g = lane >> 4;
    const long n = 1L << log_n;
    for (int i = threadIdx.x; i < MW; i += 64 * RG_WAVES) smat[i] = ((const kb_v4i *)mat)[i];
    for (int i = threadIdx.x; i < 16 * NJ * KB_MX_ROW; i += 64 * RG_WAVES) scst[i] = mat[2 * MW + i];
    __syncthreads();
    uint64_t *const st = stage[wave];
    uint64_t nx[KP];  // inputs of the next tile
    auto fetch = [&](int t) {
        int zero = 0;
        asm volatile("" : "+s"(zero));
        const uint64_t *xp = x + (long)(t >> (log_n - 6)) * in_stride + (t & ((1 << (log_n - 6)) - 1)) * RG_POS + lane;
#pragma unroll
        for (int i = 0; i < KP; ++i) nx[i] = xp[(min(i, in_n - 1) + zero) * n];
    };
    const int step = gridDim.x * RG_WAVES;
    int t = blockIdx.x * RG_WAVES + wave;
    if (t < ntiles) fetch(t);
    for (; t < ntiles; t += step) {
        // an opaque zero in the index, so that the rows' constants are read where
        // they are used instead of all being kept in (and spilled from) scalar
        // registers across the tiles
        int zero = 0;
        asm volatile("" : "+s"(zero));
        const long poly = t >> (log_n - 6);
        const long n0 = (long)(t & ((1 << (log_n - 6)) - 1)) * RG_POS;
        const uint64_t *xp = x + poly * in_stride + n0;
        uint64_t *yp = y + poly * out_stride + n0;
        kb_v4i bop[RG_MT][KC];
        {
            uint64_t v[KP];
#pragma unroll
            for (int i = 0; i < KP; ++i) v[i] = nx[i];
            double acc = SR ? 0.5 : 0.0;
            // rows past in_n are zero: they leave the estimate as it is
#pragma unroll
            for (int i = 0; i < KP; ++i) {
                const int ii = min(i, in_n - 1) + zero;
                if (i >= PAD) v[i] = i < in_n ? v[i] : 0;
                if constexpr (!SR) {
                    v[i] = kb_shoup4(v[i], inp[ii].w, inp[ii].ws, inp[ii].nq);
                    v[i] = kb_csub_sel(kb_csub_sel(v[i], inp[ii].n2q), inp[ii].nq);
                }
                acc = fma(kb_u64_to_f64(v[i]), est[ii], acc);
                if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
            }
            const uint64_t al = SR ? kb_f64_to_u64_sat(acc) : (uint64_t)(int)llround(acc);
#pragma unroll
            for (int c = 0; c < KC; ++c) {
#pragma unroll
                for (int r = 0; r < 8; ++r) {
                    const int i = 8 * c + r;
                    uint64_t d = v[i];
                    if (i >= PAD && i == in_n) d = SR ? (uint64_t)(uint32_t)al : al;
                    if (SR && i >= PAD && i == in_n + 1) d = al >> 32;
                    st[r * RG_ROW + lane] = kb_digits(d);
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
                for (int mt = 0; mt < RG_MT; ++mt)
                    bop[mt][c] = kb_pack2(st[2 * g * RG_ROW + 16 * mt + p16], st[(2 * g + 1) * RG_ROW + 16 * mt + p16]);
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            }
        }
        fetch(min(t + step, ntiles - 1));
#pragma unroll 1
        for (int nt = 0; nt < NJ; ++nt) {
            // two of the four position tiles at a time: their words fit the registers
#pragma unroll
            for (int h = 0; h < RG_MT; h += 2) {
                uint32_t W[4][2][4], up[2][4];  // [word][tile][i]
                uint64_t dg[4][2];              // scale-and-round: the R limbs' values
                if (SR) {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int m = 0; m < 2; ++m)
                            dg[i][m] = xp[(in_n + min(16 * nt + 4 * g + i, out_n - 1)) * n + 16 * (h + m) + p16];
                }
#pragma unroll
                for (int v = 7; v >= 0; --v) {
                    kb_v4i a[KC], acc[2];
#pragma unroll
                    for (int c = 0; c < KC; ++c) a[c] = smat[((nt * 8 + v) * KC + c) * 64 + lane];
#pragma unroll
                    for (int m = 0; m < 2; ++m)
                        acc[m] = kb_v4i{KB_MX_ACC_BIAS, KB_MX_ACC_BIAS, KB_MX_ACC_BIAS, KB_MX_ACC_BIAS};
#pragma unroll
                    for (int c = 0; c < KC; ++c)
#pragma unroll
                        for (int m = 0; m < 2; ++m) acc[m] = kb_mfma_i8(a[c], bop[h + m][c], acc[m]);
#pragma unroll
                    for (int m = 0; m < 2; ++m)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            if (v & 1)
                                up[m][i] = (uint32_t)acc[m][i];
                            else
                                W[v >> 1][m][i] = (up[m][i] << 8) + (uint32_t)acc[m][i];
                        }
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int j = 16 * nt + 4 * g + i;
                    if (j < out_n) {
                        const uint64_t *cst = scst + KB_MX_ROW * j;
                        const uint64_t off = cst[0], np = cst[1];
                        const uint32_t inv = (uint32_t)cst[2];
#pragma unroll
                        for (int m = 0; m < 2; ++m) {
                            uint64_t A = off;
                            if (SR) A += kb_shoup4(dg[i][m], cst[3], cst[4], np);
                            A = kb_mad32(W[1][m][i], 1u << 16, A);
                            A += W[0][m][i];
                            const uint32_t B = W[2][m][i] + (uint32_t)(A >> 32);
                            const uint32_t top = W[3][m][i] + (B >> 16);
                            const uint32_t q = __umulhi(top, inv) >> KB_MX_QSHIFT;
                            const uint64_t lo = (uint64_t)(B + (W[3][m][i] << 16)) << 32 | (uint32_t)A;
                            uint64_t r = kb_mad32(q, (uint32_t)np, lo);
                            r += (uint64_t)kb_mul_lo32(q, (uint32_t)(np >> 32)) << 32;
                            yp[j * n + 16 * (h + m) + p16] = kb_csub_sel(r, np);
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
    }
}

template <bool SR>
int launch_rns_gemm(const kbfv_context *c, int polys, hipStream_t st, const uint64_t *x, long in_stride, uint64_t *y,
                    long out_stride, const uint64_t *mat, const kb_conv_in *inp, const double *est, int in_n,
                    int out_n) {
    const int kc = (in_n + (SR ? 2 : 1) + 7) / 8, nj = (out_n + 15) / 16;
    const long tiles = (long)polys << (c->log_n - 6);
    KB_REQUIRE(tiles < (1L << 31) - (1 << 20), "base conversion grid too large");
    const dim3 grid((unsigned)std::min<long>(RG_CUS, (tiles + RG_WAVES - 1) / RG_WAVES));
#define KB_RG(KC, NJ)                                                                                        \
    if (kc == KC && nj == NJ) {                                                                               \
        hipLaunchKernelGGL((k_rns_gemm<KC, NJ, SR>), grid, dim3(64 * RG_WAVES), 0, st, x, in_stride, y,      \
                           out_stride, mat, inp, est, in_n, out_n, c->log_n, (int)tiles);                       \
        KB_LAUNCH_CHECK();                                                                                     \
        return KBFV_OK;                                                                                        \
    }
    KB_RG(2, 1)
    KB_RG(3, 1)
    KB_RG(3, 2)
    KB_RG(4, 2)
#undef KB_RG
    kb_set_error("base conversion of %d into %d limbs does not fit the matrix kernel", in_n, out_n);
    return KBFV_EINVAL;
}

}  // namespace

int kb_bconv_mfma(const kbfv_context *c, bool q_to_r, const uint64_t *x, long in_stride, uint64_t *y, long out_stride,
                  int polys, hipStream_t st, bool noscale) {
    const kb_dev_tables &t = c->t;
    return launch_rns_gemm<false>(c, polys, st, x, in_stride, y, out_stride, q_to_r ? t.mx_qr : t.mx_rq,
                                  q_to_r ? (noscale ? t.cv_in_qn : t.cv_in_q) : t.cv_in_r, q_to_r ? t.q_inv : t.r_inv,
                                  q_to_r ? c->qn : c->rn, q_to_r ? c->rn : c->qn);
}

int kb_scale_round_mfma(const kbfv_context *c, const uint64_t *x, uint64_t *y, int polys, hipStream_t st) {
    const kb_dev_tables &t = c->t;
    return launch_rns_gemm<true>(c, polys, st, x, (long)(c->qn + c->rn) * c->n, y, (long)c->rn * c->n, t.mx_sr,
                                 nullptr, t.sr_frac, c->qn, c->rn);
}
