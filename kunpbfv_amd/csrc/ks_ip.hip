// Key-switch inner product on the VALU: the key streams past one to four ciphertexts
// (k_ip_stream) or stays in registers while more walk by (k_ip_hold, up to 32 digits).
//
// Replaces external_product_T_kernel and its _swk_reuse variant
// (include/ExternalProduct.cuh:11-177): for T limb k and coefficient n,
//     out[ct][h][b] = sum_{d < D} cin[ct][d] key[h][d][b]   mod t_k.
// In the stream a thread takes V coefficients of one key block b, both key halves h, and C
// ciphertexts at a time; a workgroup's waves take neighbouring blocks of the same
// coefficients, so the digits they share come through one L1.
//
// Products are Karatsuba on 30-bit halves with no carries: three
// v_mad_u64_u32 per 60 x 60-bit multiply-add into lo = sum x0 k0, hi = sum x1 k1 and
// mm = sum (x0 + x1)(k0 + k1).  Eight terms keep the middle sum mm - lo - hi below
// 2^64 (mm itself may wrap), so after every eight the middle is carried into
// the total sum = F 2^60 + e 2^30 + lo, e, lo < 2^30; beyond 16 terms F needs a
// carry word.  The reduction is one Shoup product by 2^s mod t.
//
// One ciphertext is bound by the key, read once: 28 digits, 15 blocks at N = 2^16
// (1.76 GB) take 372 us, 4.9 TB/s (745 us with 8-byte loads into LDS and 128-bit
// accumulators).
#include <type_traits>

#include "kbfv_internal.h"
#include "kbfv_ops.h"

namespace {

constexpr int IS_WAVES = 8;
constexpr int IS_STEP = 4;  // digits loaded together

template <int V>
__device__ __forceinline__ void load_v(const uint64_t *p, uint64_t (&o)[V]) {
    if constexpr (V == 1) {
        o[0] = *p;
    } else {
        const kb_u64x2 v = *(const kb_u64x2 *)p;
        o[0] = v.x, o[1] = v.y;
    }
}

// carries the middle sum mm - lo - hi of at most eight new terms into hi (WIDE:
// and hi into (top, F)), leaving lo and the middle below 2^30
template <bool WIDE>
__device__ __forceinline__ void carry_middle(uint64_t &lo, uint64_t &hi, uint64_t &mm, uint64_t &F, uint32_t &top) {
    constexpr uint64_t M = (1u << 30) - 1;
    const uint64_t e = mm - lo - hi + (lo >> 30);
    hi += e >> 30;
    lo &= M;
    if constexpr (WIDE) {
        F += hi;
        top += F < hi ? 1u : 0u;
        hi = 0;
    }
    mm = (e & M) + lo + hi;
}

// C ciphertexts at a time, V coefficients per thread; WIDE: more than 16 digits
template <int C, int V, bool WIDE>
__global__ void __launch_bounds__(64 * IS_WAVES)
    k_ip_stream(const uint64_t *__restrict__ cin, const uint64_t *__restrict__ key, uint64_t *__restrict__ out,
                const kb_fold *__restrict__ fold, int D, int B, int KD, int KB, int tn, int log_n, int batch) {
    const int lane = threadIdx.x & 63;
    const int waves = blockDim.x >> 6;
    const int bgroups = (B + waves - 1) / waves;
    // the groups of blocks of one tile are 8 workgroups apart: the same XCD
    const int tiles = (1 << log_n) / (64 * V);
    const int r = blockIdx.x / (8 * bgroups), q8 = blockIdx.x % (8 * bgroups);
    const int tg = r * 8 + q8 % 8;  // (T limb, tile); tiles is a multiple of 8
    const int b = (q8 / 8) * waves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (b >= B) return;
    const int kk = tg / tiles;
    const long N = 1L << log_n, TN = (long)tn << log_n;
    const long k = (long)kk * N + (long)(tg % tiles) * 64 * V + lane * V;
    const uint64_t *key0 = key + (long)b * TN + k, *key1 = key0 + (long)KD * KB * TN;
    const long ks = (long)KB * TN;  // digit stride in the key
    const kb_fold f = fold[kk];
    constexpr uint32_t M = (1u << 30) - 1;

    for (int c0 = 0; c0 < batch; c0 += C) {
        uint64_t lo[C][2][V], hi[C][2][V], mm[C][2][V], F[C][2][V];
        uint32_t top[C][2][V];
        const uint64_t *xp[C];
#pragma unroll
        for (int c = 0; c < C; ++c) {
            xp[c] = cin + (long)min(c0 + c, batch - 1) * D * TN + k;
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int v = 0; v < V; ++v) {
                    lo[c][h][v] = hi[c][h][v] = mm[c][h][v] = F[c][h][v] = 0;
                    top[c][h][v] = 0;
                }
        }
#pragma unroll 1
        for (int d0 = 0; d0 < D; d0 += IS_STEP) {
            uint64_t kv[IS_STEP][2][V], x[IS_STEP][C][V];
#pragma unroll
            for (int i = 0; i < IS_STEP; ++i) {
                const long d = min(d0 + i, D - 1);
                load_v<V>(key0 + d * ks, kv[i][0]);
                load_v<V>(key1 + d * ks, kv[i][1]);
#pragma unroll
                for (int c = 0; c < C; ++c) load_v<V>(xp[c] + d * TN, x[i][c]);
            }
#pragma unroll
            for (int i = 0; i < IS_STEP; ++i) {
                if (d0 + i >= D) break;  // uniform
#pragma unroll
                for (int v = 0; v < V; ++v) {
                    uint32_t k0[2], k1[2];
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        k0[h] = (uint32_t)kv[i][h][v] & M;
                        k1[h] = (uint32_t)(kv[i][h][v] >> 30);
                    }
#pragma unroll
                    for (int c = 0; c < C; ++c) {
                        const uint32_t x0 = (uint32_t)x[i][c][v] & M, x1 = (uint32_t)(x[i][c][v] >> 30);
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            kb_mad(lo[c][h][v], x0, k0[h]);
                            kb_mad(hi[c][h][v], x1, k1[h]);
                            kb_mad(mm[c][h][v], x0 + x1, k0[h] + k1[h]);
                        }
                    }
                }
            }
            if ((d0 & IS_STEP) || d0 + IS_STEP >= D) {  // eight terms: carry the middle
#pragma unroll
                for (int c = 0; c < C; ++c)
#pragma unroll
                    for (int h = 0; h < 2; ++h)
#pragma unroll
                        for (int v = 0; v < V; ++v)
                            carry_middle<WIDE>(lo[c][h][v], hi[c][h][v], mm[c][h][v], F[c][h][v], top[c][h][v]);
            }
        }
#pragma unroll
        for (int c = 0; c < C; ++c) {
            if (c0 + c >= batch) break;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                uint64_t o[V];
#pragma unroll
                for (int v = 0; v < V; ++v) {
                    const uint64_t l = lo[c][h][v], u = hi[c][h][v];
                    const uint64_t L = (mm[c][h][v] - l - u) << 30 | l;
                    o[v] = kb_fold_reduce<WIDE>(WIDE ? F[c][h][v] : u, top[c][h][v], L, f);
                }
                uint64_t *op = out + ((long)(c0 + c) * 2 * B + (long)h * B + b) * TN + k;
                if constexpr (V == 1)
                    *op = o[0];
                else
                    *(kb_u64x2 *)op = kb_u64x2{o[0], o[1]};
            }
        }
    }
}

// Larger batches: the key stays.  A thread keeps its coefficient's key values
// of one block, both halves, as 30-bit pairs in registers and walks the batch,
// two ciphertexts at a time; their digits are split once per workgroup and pass
// through a double-buffered LDS tile that all the blocks' waves read.  Bound by
// VALU issue (four instructions per product, about 80 per output).  15 digits, 8
// blocks, 7 ciphertexts at N = 2^15: 126 us (250 with 128-bit accumulators); 13
// digits, 64 ciphertexts: 729 us (1230 on the matrix cores, 401 for the bytes at 5
// TB/s); 28 digits, 16 ciphertexts at N = 2^16: 1.85 ms (2.54).
template <int MAXD>
__global__ void __launch_bounds__(64 * IS_WAVES)
    k_ip_hold(const uint64_t *__restrict__ cin, const uint64_t *__restrict__ key, uint64_t *__restrict__ out,
              const kb_fold *__restrict__ fold, int D, int B, int KD, int KB, int tn, int log_n, int batch) {
    constexpr bool WIDE = MAXD > 16;
    __shared__ uint4 xs[2][MAXD][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int waves = blockDim.x >> 6;
    const int bgroups = (B + waves - 1) / waves;
    const int tiles = 1 << (log_n - 6);
    const int r8 = blockIdx.x / (8 * bgroups), q8 = blockIdx.x % (8 * bgroups);
    const int tg = r8 * 8 + q8 % 8;
    const int b = min((q8 / 8) * waves + wave, B - 1);  // a wave past the last block repeats it
    const int kk = tg / tiles;
    const long N = 1L << log_n, TN = (long)tn << log_n;
    const long k = (long)kk * N + (long)(tg % tiles) * 64 + lane;
    const kb_fold f = fold[kk];
    constexpr uint32_t M = (1u << 30) - 1;

    uint32_t k0[MAXD][2], k1[MAXD][2];
    {
        const uint64_t *kp = key + (long)b * TN + k;
        const long ks = (long)KB * TN;
#pragma unroll
        for (int i = 0; i < MAXD; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint64_t v = kp[(long)(h * KD + min(i, D - 1)) * ks];
                k0[i][h] = (uint32_t)v & M;
                k1[i][h] = (uint32_t)(v >> 30);
            }
    }
    // the workgroup's rows of a ciphertext pair, row i of ciphertext c being number
    // 2 i + c, four loads of a wave in flight at a time
    auto stage = [&](int ct, int buf) {
        const uint64_t *xp = cin + k;
        for (int j0 = wave; j0 < 2 * D; j0 += 4 * waves) {
            uint64_t v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int j = min(j0 + u * waves, 2 * D - 1);
                v[u] = xp[((long)min(ct + (j & 1), batch - 1) * D + (j >> 1)) * TN];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int j = min(j0 + u * waves, 2 * D - 1);
                ((uint2 *)&xs[buf][j >> 1][lane])[j & 1] = make_uint2((uint32_t)v[u] & M, (uint32_t)(v[u] >> 30));
            }
        }
    };
    stage(0, 0);
    __syncthreads();
    for (int ct = 0, buf = 0; ct < batch; ct += 2, buf ^= 1) {
        if (ct + 2 < batch) stage(ct + 2, buf ^ 1);
        uint64_t lo[2][2], hi[2][2], mm[2][2], F[2][2];
        uint32_t top[2][2];
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int h = 0; h < 2; ++h) lo[c][h] = hi[c][h] = mm[c][h] = F[c][h] = 0, top[c][h] = 0;
#pragma unroll
        for (int i = 0; i < MAXD; ++i) {
            if (i < D) {  // uniform
                const uint4 x = xs[buf][i][lane];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    kb_pin(k0[i][h]), kb_pin(k1[i][h]);  // and their sum is formed here, not kept
                    const uint32_t ks = k0[i][h] + k1[i][h];
                    kb_mad(lo[0][h], x.x, k0[i][h]);
                    kb_mad(lo[1][h], x.z, k0[i][h]);
                    kb_mad(hi[0][h], x.y, k1[i][h]);
                    kb_mad(hi[1][h], x.w, k1[i][h]);
                    kb_mad(mm[0][h], x.x + x.y, ks);
                    kb_mad(mm[1][h], x.z + x.w, ks);
                }
            }
            if (i % 8 == 7 || i == MAXD - 1) {
#pragma unroll
                for (int c = 0; c < 2; ++c)
#pragma unroll
                    for (int h = 0; h < 2; ++h) carry_middle<WIDE>(lo[c][h], hi[c][h], mm[c][h], F[c][h], top[c][h]);
            }
        }
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            if (ct + c >= batch) break;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint64_t l = lo[c][h], u = hi[c][h];
                const uint64_t L = (mm[c][h] - l - u) << 30 | l;
                out[((long)(ct + c) * 2 * B + (long)h * B + b) * TN + k] =
                    kb_fold_reduce<WIDE>(WIDE ? F[c][h] : u, top[c][h], L, f);
            }
        }
        __syncthreads();
    }
}

}  // namespace

int kb_inner_product_stream(const kbfv_context *c, const uint64_t *cin, const uint64_t *key, uint64_t *out, int batch,
                            hipStream_t st) {
    const int D = c->dnum, B = c->ri_blocks;
    const int groups = (B + IS_WAVES - 1) / IS_WAVES, waves = (B + groups - 1) / groups;
    auto go = [&](auto tag) -> int {
        constexpr int C = decltype(tag)::value, V = C <= 2 ? 2 : 1;
        const long blocks = (long)groups * c->tn * (c->n / (64 * V));
        KB_REQUIRE(blocks < (1L << 31), "inner product grid too large");
        if (D > 16)
            hipLaunchKernelGGL((k_ip_stream<C, V, true>), dim3((unsigned)blocks), dim3(64 * waves), 0, st, cin, key, out,
                               c->t.t_fold, D, B, c->key_dnum, c->key_blocks, c->tn, c->log_n, batch);
        else
            hipLaunchKernelGGL((k_ip_stream<C, V, false>), dim3((unsigned)blocks), dim3(64 * waves), 0, st, cin, key, out,
                               c->t.t_fold, D, B, c->key_dnum, c->key_blocks, c->tn, c->log_n, batch);
        KB_LAUNCH_CHECK();
        return KBFV_OK;
    };
    // two ciphertexts and fewer: the key's bytes bound both kernels, and the stream
    // reads 16 per lane (28 digits, N = 2^16: 411 us for two, against 700).  Keys of more
    // than 16 digits leave the holding kernel two waves per SIMD, so it starts later:
    // 672 against 733 us for four, 1257 against 1103 for eight
    if (batch > (D > 16 ? 4 : 2) && D <= 32) {
        const long blocks = (long)groups * c->tn * (c->n / 64);
        KB_REQUIRE(blocks < (1L << 31), "inner product grid too large");
#define KB_IH(MD)                                                                                                   \
    if (D <= MD) {                                                                                                  \
        hipLaunchKernelGGL(k_ip_hold<MD>, dim3((unsigned)blocks), dim3(64 * waves), 0, st, cin, key, out, c->t.t_fold, \
                           D, B, c->key_dnum, c->key_blocks, c->tn, c->log_n, batch);                               \
        KB_LAUNCH_CHECK();                                                                                          \
        return KBFV_OK;                                                                                             \
    }
        KB_IH(2)
        KB_IH(4)
        KB_IH(8)
        KB_IH(12)
        KB_IH(16)
        KB_IH(24)
        KB_IH(32)
#undef KB_IH
    }
    if (batch == 1) return go(std::integral_constant<int, 1>{});
    if (batch == 2) return go(std::integral_constant<int, 2>{});
    return go(std::integral_constant<int, 4>{});
}
