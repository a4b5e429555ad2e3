// HPS base conversion and scale-and-round: one coefficient per thread, every
// input limb of it in registers.
//
// Replaces base_convert_matmul_hps_unroll2_kernel and scaleAndRound_HPS_QR_R
// (include/poly_arithmetic.cuh:1139-1178, :1263-1317).
//   Base conversion Q -> R (and R -> Q):  y_i = [x_i (Q/q_i)^-1]_{q_i};
//     alpha = llround(sum_i y_i / q_i)   (double, input order, explicit fma);
//     out_j = [sum_i y_i [Q/q_i]_{r_j} + alpha [-Q]_{r_j}]_{r_j}.
//   Scale-and-round QR -> R:  nu = 0.5 + sum_{i<qn} x_i frac_i (double);
//     out_j = [sum_{i<qn} x_i M_ij + x_{qn+j} c_j + (uint64)nu]_{r_j}.
// The double estimates are the reference's, in its order; every other step is
// exact, so the outputs are the canonical residues.
//
// Both are products with a constant matrix.  An operand is split once into two
// signed 30-bit halves, x - 2^59 = x1 2^30 + x0 with |x0|, |x1| <= 2^29 (the
// 2^59 times the matrix row is a constant of the row), and a matrix entry is
// taken in [-p/2, p/2] and split the same way on the host, so a row costs
// three v_mad_i64_i32 (x0 m0, x1 m1, (x0+x1)(m0+m1)) into three 64-bit
// accumulators and no carry.  The matrix comes through the scalar cache.  |x0 m0|
// and |x1 m1| are at most 2^58 and the middle product at most 2^59: 31 rows
// fit the outer accumulators, 15 the middle one, which is closed after every
// 15 full rows, scale-and-round's diagonal among them (the third product may wrap: only
// middle = third - first - second has to fit).  Carrying the middle upwards gives the
// sum as f 2^60 + L with L in [0, 2^60); for 2^(s-1) < p < 2^s its quotient H by 2^s fits
// 63 bits and a sign, and the result is [(H + 2^63) (2^s mod p) + (L mod 2^s) +
// const]_p, one Shoup product and three conditional subtractions.
//
// Bound by VALU issue: a multiply-add takes 5.2 cycles of a SIMD, any other
// multiply 4.4, an output about 30 of them besides its rows.  2 primes, 36
// polynomials at N = 2^13: 5.6 us (13.9 as an MFMA product); 4 primes of 36 bits, 20
// polynomials at N = 2^14: 8.7 us (18.0 with 128-bit accumulators and the inputs
// in LDS).
#include <algorithm>

#include "kbfv_internal.h"
#include "kbfv_ops.h"

namespace {

// blockIdx.y: outputs j0 = per blockIdx.y .. of the thread's coefficient
template <int IN, bool SR>
__global__ void __launch_bounds__(256)
    k_rns_conv(const uint64_t *__restrict__ x, long in_stride, uint64_t *__restrict__ y, long out_stride,
               const uint64_t *__restrict__ tab, const kb_conv_in *__restrict__ inp,
               const double *__restrict__ est, int out_n, int per, int log_n, int log_bs) {
    const int j0 = (int)blockIdx.y * per, j1 = min(j0 + per, out_n);
    const long n = 1L << log_n;
    const long poly = blockIdx.x >> (log_n - log_bs);
    const long k = (long)((blockIdx.x & ((1 << (log_n - log_bs)) - 1)) << log_bs) + threadIdx.x;
    const uint64_t *xp = x + poly * in_stride + k;
    uint64_t *yp = y + poly * out_stride + k;

    uint64_t v[IN];
#pragma unroll
    for (int i = 0; i < IN; ++i) v[i] = xp[i * n];
    int x0[IN], x1[IN], xs[IN];
    double acc = SR ? 0.5 : 0.0;
#pragma unroll
    for (int i = 0; i < IN; ++i) {
        if constexpr (!SR) {
            v[i] = kb_shoup4(v[i], inp[i].w, inp[i].ws, inp[i].nq);
            v[i] = kb_csub_sel(kb_csub_sel(v[i], inp[i].n2q), inp[i].nq);
        }
        acc = fma(kb_u64_to_f64(v[i]), est[i], acc);
        kb_split30(v[i], x0[i], x1[i]);
        xs[i] = x0[i] + x1[i];
    }
    const int alpha = SR ? 0 : (int)llround(acc);
    const uint64_t nu = SR ? kb_f64_to_u64_sat(acc) : 0;

    constexpr int RW = kb_conv_row_words(IN);
    // rows of full size (scale-and-round's diagonal is one, alpha's row is small) per middle
    // accumulator, and the number of accumulators
    constexpr int G = 15, NG = (IN + (SR ? 1 : 0) + G - 1) / G;
    static_assert(NG * G >= IN + (SR ? 1 : 0), "a middle accumulator holds 15 full rows");
    uint64_t diag = SR ? xp[(IN + j0) * n] : 0;
#pragma unroll 1
    for (int j = j0; j < j1; ++j) {
        const uint64_t *row = tab + (long)j * RW;
        const int *m = (const int *)row;
#pragma unroll
        for (int i = 0; i < IN; ++i) kb_pin(x0[i]), kb_pin(x1[i]), kb_pin(xs[i]);
        uint64_t dnext = 0;
        if (SR) dnext = xp[(IN + min(j + 1, j1 - 1)) * n];
        int64_t lo = 0, hi = 0, mid[NG];
        uint64_t outer = 0;  // lo + hi of the groups before
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            int64_t mm = 0;
#pragma unroll
            for (int i = g * G; i < IN && i < g * G + G; ++i) {
                kb_mad(lo, x0[i], m[3 * i]);
                kb_mad(hi, x1[i], m[3 * i + 1]);
                kb_mad(mm, xs[i], m[3 * i + 2]);
            }
            if (g == NG - 1) {  // the last group takes the extra row
                if constexpr (SR) {
                    int d0, d1;
                    kb_split30(diag, d0, d1);
                    kb_mad(lo, d0, m[3 * IN]);
                    kb_mad(hi, d1, m[3 * IN + 1]);
                    kb_mad(mm, d0 + d1, m[3 * IN + 2]);
                } else {
                    kb_mad(lo, alpha, m[3 * IN]);
                    kb_mad(mm, alpha, m[3 * IN + 2]);
                }
            }
            const uint64_t o = (uint64_t)lo + (uint64_t)hi;
            mid[g] = (int64_t)((uint64_t)mm - (o - outer));
            outer = o;
        }
        diag = dnext;
        if constexpr (SR) {
            lo += (int64_t)((uint32_t)nu & 0x3fffffffu);
            mid[0] += (int64_t)(nu >> 30);
        }
        constexpr int64_t M30 = (1 << 30) - 1;
        int64_t e = mid[0] + (lo >> 30), f = hi + (e >> 30);
#pragma unroll
        for (int g = 1; g < NG; ++g) {
            e = (e & M30) + mid[g];
            f += e >> 30;
        }
        const uint64_t *c = row + (RW - KB_CONV_TAIL);
        uint64_t L = (uint64_t)(e & M30) << 30 | (uint64_t)(lo & M30), H = (uint64_t)f;
        if (const int s = (int)c[6]; s != 60) {  // uniform
            H = (H << (60 - s)) + (L >> s);
            L &= (1ULL << s) - 1;
        }
        uint64_t r = kb_shoup4(H ^ (1ULL << 63), c[1], c[2], c[3]) + (L + c[0]);  // [0, 7p)
        r = kb_csub_sel(r, c[5]);
        r = kb_csub_sel(r, c[4]);
        r = kb_csub_sel(r, c[3]);
        yp[j * n] = r;
    }
}

struct conv_args {
    const uint64_t *x;
    long in_stride;
    uint64_t *y;
    long out_stride;
    const uint64_t *tab;
    const kb_conv_in *inp;
    const double *est;
    int in_n, out_n, polys, log_n;
    hipStream_t st;
};

template <bool SR, int IN = 1>
int launch(const conv_args &a, dim3 grid, int per, int log_bs) {
    if constexpr (IN <= KB_CONV_MAXROWS - (SR ? 1 : 0)) {
        if (a.in_n != IN) return launch<SR, IN + 1>(a, grid, per, log_bs);
        hipLaunchKernelGGL((k_rns_conv<IN, SR>), grid, dim3(1 << log_bs), 0, a.st, a.x, a.in_stride, a.y, a.out_stride,
                           a.tab, a.inp, a.est, a.out_n, per, a.log_n, log_bs);
        KB_LAUNCH_CHECK();
        return KBFV_OK;
    } else {
        kb_set_error("RNS conversion of %d limbs exceeds the register kernel", a.in_n);
        return KBFV_EINVAL;
    }
}

// Workgroups of one wave while that leaves compute units idle, of four otherwise.
// Where even single waves leave SIMDs idle, a coefficient's outputs are split over up
// to eight threads that each repeat the input part (about the work of two outputs):
// 28 primes, N=4096, Q -> R of 1 / 4 / 8 polynomials 26.5 / 26.9 / 29.8 us whole, 8.0 /
// 12.5 / 15.1 in 8 / 4 / 4 parts; 12 primes, 16 polynomials 11.0 whole, 8.0 in two, 32
// polynomials 11.0 whole, 11.5 in two; 30 primes of 45 bits, 32 polynomials 60 whole,
// 44 in two, 64 polynomials 67 whole, 78 in two.  Chains of up to 8 primes take the 7.3
// us of an empty call either way.
template <bool SR>
int launch_any(const conv_args &a) {
    const long coeffs = (long)a.polys << a.log_n, waves = coeffs / 64;
    const int lb = coeffs < 256L * 1024 ? 6 : 8;
    const long blocks = (long)a.polys << (a.log_n - lb);
    KB_REQUIRE(blocks < (1L << 31), "grid too large");
    int parts = 1;
    if (a.in_n > 8) parts = (int)std::min(8L, std::max(1L, (a.in_n > 16 && waves > 1024 ? 4096 : 2048) / waves));
    const int per = (a.out_n + parts - 1) / parts;
    return launch<SR>(a, dim3((unsigned)blocks, (a.out_n + per - 1) / per), per, lb);
}

}  // namespace

int kb_bconv_reg(const kbfv_context *c, bool q_to_r, const uint64_t *x, long in_stride, uint64_t *y, long out_stride,
                 int polys, hipStream_t st, bool noscale) {
    const kb_dev_tables &t = c->t;
    return launch_any<false>({x, in_stride, y, out_stride, q_to_r ? t.cv_qr : t.cv_rq,
                              q_to_r ? (noscale ? t.cv_in_qn : t.cv_in_q) : t.cv_in_r, q_to_r ? t.q_inv : t.r_inv,
                              q_to_r ? c->qn : c->rn, q_to_r ? c->rn : c->qn, polys, c->log_n, st});
}

int kb_scale_round_reg(const kbfv_context *c, const uint64_t *x, uint64_t *y, int polys, hipStream_t st) {
    const kb_dev_tables &t = c->t;
    return launch_any<true>({x, (long)(c->qn + c->rn) * c->n, y, (long)c->rn * c->n, t.cv_sr, nullptr, t.sr_frac, c->qn,
                             c->rn, polys, c->log_n, st});
}
