// nnrh_qgemm_small.hip -- int8 GEMM / implicit-GEMM convolution for grids that
// leave most of the chip idle: small output tiles, K split over the waves of
// a block, fragments straight from global memory into registers.
//
// Same arithmetic as qgemm_kernel (nnrh_qgemm.hip) and qgemm_dma_kernel
// (nnrh_qgemm_dma.hip): exact int32 sums of i8 MFMA 16x16x64, the zero-point
// terms, one of NNR's requantize epilogues. int32 addition is associative
// modulo 2^32, so splitting K changes no bit.
//
// What bounds these shapes is not bytes or operations but the chain of one
// block: with 128 x 128 tiles a 49 x 512 output is 4 blocks, each walking all
// of K = 4608 in 36 dependent steps of load, barrier and MFMA (26 us). Here it
// is 128 blocks of 16 waves whose every load is in flight at once (5.2 us; an
// empty kernel takes 1.7). In a graph of one layer after another, weights from
// the Infinity Cache, rows x columns x K: 196x256x2304 16.1 -> 3.7 us, 37x768x3072
// 18.5 -> 5.0, 784x512x128 4.6 -> 2.9, 1x3072x768 7.7 -> 3.7, 1024x768x3072 19.7 ->
// 12.0.
// What is left is the L1's line rate on the operands, (1 / BM + 1 / BN) bytes
// a multiply, and about 2.5 us of launch, first latency and drain.
#include <cstdio>

#include "nnrh_internal.h"
#include "nnrh_rq.h"

namespace nnrh {

typedef int v4i __attribute__((ext_vector_type(4)));

namespace {

// epilogue of an instantiation: those whole networks run on, each without the
// branches of the others (with every mode in one kernel the encoder's 37 x 768
// x 768 projection takes 4.2 us instead of 2.8), and one for the rest
enum SmallEpi : int {
    SE_RQB = 0,       // RQ-B, constants in c0 / os, NHWC or row-major 8-bit output
    SE_RQB_ADD = 1,   // then QLinearAdd of a residual (uint8)
    SE_DQ = 2,        // RQ-D or EPI_I32S with their fused chains, row-major output
    SE_I32 = 3,       // int32 output, the zero-point sums formed here (sums_inline)
    SE_GEN = 4,       // any unfused 8-bit mode: scalar tails, NCHW output, row sums
};

// What the kernel reads before its first operand load sits in the first
// cache lines of the argument block: each line is a memory latency of its own.
struct SmallArgs {
    const uint8_t* a;
    const int8_t* b;
    long long a_bstride, b_bstride;
    int M, N, K, Kp;
    uint32_t div_t_mul, div_t_shift;   // tile index / (nbm or nbn)
    int nbm, nbn;
    // (64 bytes)
    int n_major;                       // tiles of one column block are neighbours
    int lda;                           // dense row stride
    uint32_t xmask;
    int nunits;                        // K in units of two MFMA steps
    // convolution
    int H, W, C, Cs, kW, sH, sW, dH, dW, pad_t, pad_l, oW;
    // (128 bytes)
    int sp_out;
    uint32_t padw;
    uint32_t div_sp_mul, div_sp_shift, div_ow_mul, div_ow_shift, div_c_mul, div_c_shift, div_kw_mul, div_kw_shift;
    // per-column arrays, all readable (an unused one repeats another)
    const int32_t* c;                  // c0, or colsum when the zero point comes with the call
    const float *p0, *p1;
    // (192 bytes)
    const int32_t* beta_col;
    long long param_bstride;
    void* y;
    long long ldy, y_bstride;
    int y_zp, lo, hi;
    int pairs;                         // (min, max) pairs mm_parts holds
};

// 16 zero bytes: the weights of a K step past the end
__device__ const uint32_t kZero16[4] = {0u, 0u, 0u, 0u};

// 16 bytes at any alignment
__device__ __forceinline__ v4i load16(const uint8_t* p) {
    v4i v;
    __builtin_memcpy(&v, p, 16);
    return v;
}

}  // namespace

// Block: one output tile of 16 MT rows x 16 NT columns, W = blockDim.x / 64
// waves. Wave w takes K in units of two MFMA steps (128 bytes of a row: a
// whole cache line), units w, w + W, ...; a unit's loads are issued while the
// unit before it multiplies. The W partial tiles meet in LDS and each thread
// finishes 4 consecutive columns of a row.
template <int MT, int NT, int AMODE, int VEC, int EP, int MAXW>
__global__ __launch_bounds__(MAXW * 64) void qgemm_small_kernel(SmallArgs s, GemmArgs g) {
    constexpr int BM = 16 * MT, BN = 16 * NT;
    constexpr int RS = BN + 4;              // LDS row stride in dwords: 16 rows spread over the banks
    constexpr int CH = BM * BN / 4;         // 4-column chunks of the tile
    extern __shared__ __attribute__((aligned(16))) int red[];   // [W][BM][RS]
    const int tid = threadIdx.x, nthr = blockDim.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), W = nthr >> 6;
    const int frow = lane & 15, fchunk = lane >> 4;

    // XCD x takes the x-th contiguous eighth of the tile list, ordered so
    // that neighbours share the operand with more bytes
    const int total = s.nbm * s.nbn;
    const int per_xcd = (total + 7) >> 3;
    const int t = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per_xcd || t >= total) return;
    const int z = blockIdx.z;
    const int tq = (int)fast_div((uint32_t)t, s.div_t_mul, s.div_t_shift);
    const int tr = t - tq * (s.n_major ? s.nbm : s.nbn);
    const int m0 = (s.n_major ? tr : tq) * BM, n0 = (s.n_major ? tq : tr) * BN;

    // ---- operand rows of this lane (rows past M read row M - 1 and are not
    // stored)
    const uint8_t* abase = s.a + (long long)z * s.a_bstride;
    const int8_t* bbase = s.b + (long long)z * s.b_bstride;
    const uint8_t* a_ptr[MT];
    int a_ih0[MT], a_iw0[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        int m = m0 + 16 * mt + frow;
        m = m < s.M ? m : s.M - 1;
        if constexpr (AMODE == A_DENSE) {
            a_ptr[mt] = abase + (long long)m * s.lda;
        } else {
            const int img = (int)fast_div((uint32_t)m, s.div_sp_mul, s.div_sp_shift);
            const int p = m - img * s.sp_out;
            const int oh = (int)fast_div((uint32_t)p, s.div_ow_mul, s.div_ow_shift);
            a_ptr[mt] = abase + (long long)img * s.H * s.W * s.Cs;
            a_ih0[mt] = oh * s.sH - s.pad_t;
            a_iw0[mt] = (p - oh * s.oW) * s.sW - s.pad_l;
        }
    }
    const int8_t* b_row[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
        b_row[nt] = bbase + piece_off(n0 + 16 * nt + frow, fchunk * 16, s.Kp);

    // ---- K loop
    auto load_a = [&](int k, v4i (&xf)[MT]) {
        if constexpr (AMODE == A_DENSE) {
            if constexpr (VEC == 16) {
                // K padding meets zero weights: any bytes do (where rows are
                // summed, those that the shift makes 0)
                const int kk = k < s.K ? k : 0;
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    xf[mt] = *(const v4i*)(a_ptr[mt] + kk);
                    if constexpr (EP == SE_I32) {
                        const int xw = (int)s.xmask;
                        if (k >= s.K) xf[mt] = v4i{xw, xw, xw, xw};
                    }
                }
            } else if constexpr (VEC == 8) {
                const int k0 = k < s.K ? k : 0, k1 = k + 8 < s.K ? k + 8 : 0;
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    const uint2 v0 = *(const uint2*)(a_ptr[mt] + k0), v1 = *(const uint2*)(a_ptr[mt] + k1);
                    xf[mt] = v4i{(int)v0.x, (int)v0.y, (int)v1.x, (int)v1.y};
                }
            } else {
                // rows of any length: whole chunks unaligned, the row's last
                // chunk byte by byte (it may end the matrix)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    if (k + 16 <= s.K) {
                        xf[mt] = load16(a_ptr[mt] + k);
                    } else {
                        uint32_t w[4] = {0u, 0u, 0u, 0u};
#pragma unroll
                        for (int i = 0; i < 16; ++i)
                            w[i >> 2] |= (k + i < s.K ? (uint32_t)a_ptr[mt][k + i] : s.xmask & 0xffu) << (8 * (i & 3));
                        xf[mt] = v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
                    }
                }
            }
        } else {
#pragma unroll
            for (int sb = 0; sb < 16 / VEC; ++sb) {
                const int kv = k + sb * VEC;
                const int kp = (int)fast_div((uint32_t)kv, s.div_c_mul, s.div_c_shift);
                const int ic = kv - kp * s.C;
                const int kh = (int)fast_div((uint32_t)kp, s.div_kw_mul, s.div_kw_shift);
                const int kw = kp - kh * s.kW;
                const int dh = kh * s.dH, dw = kw * s.dW;
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    const int ih = a_ih0[mt] + dh, iw = a_iw0[mt] + dw;
                    // a padded tap reads the image's first bytes and takes the
                    // pad byte; K padding meets zero weights
                    const bool in = (unsigned)ih < (unsigned)s.H && (unsigned)iw < (unsigned)s.W && kv < s.K;
                    const uint8_t* p = a_ptr[mt] + (in ? (long long)(ih * s.W + iw) * s.Cs + ic : 0LL);
                    if constexpr (VEC == 16) {
                        const v4i v = *(const v4i*)p;
                        const int pw = (int)s.padw;
                        xf[mt] = v4i{in ? v.x : pw, in ? v.y : pw, in ? v.z : pw, in ? v.w : pw};
                    } else if constexpr (VEC == 8) {
                        const uint2 v = *(const uint2*)p;
                        xf[mt][2 * sb] = (int)(in ? v.x : s.padw);
                        xf[mt][2 * sb + 1] = (int)(in ? v.y : s.padw);
                    } else if constexpr (VEC == 4) {
                        const uint32_t v = *(const uint32_t*)p;
                        xf[mt][sb] = (int)(in ? v : s.padw);
                    } else {
                        const uint32_t v = in ? (uint32_t)*p : (s.padw & 0xffu);
                        if ((sb & 3) == 0) xf[mt][sb >> 2] = 0;
                        xf[mt][sb >> 2] = (int)((uint32_t)xf[mt][sb >> 2] | v << (8 * (sb & 3)));
                    }
                }
            }
        }
    };
    v4i acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = v4i{0, 0, 0, 0};
    // the two halves of a 128-byte line come with two loads; odd rows take
    // theirs in the other order, so that each load asks for both kinds of half
    // (16 rows' equal halves cost the L1 twice the time: 512 rows, 768 columns,
    // K = 3072 in 32x64 tiles 7.7 -> 6.8 us)
    const int odd = (frow & 1) * 64;
    struct Unit { v4i x[2][MT], w[2][NT]; };
    auto load_unit = [&](int u, Unit& d) {
        // the second step of the last unit may lie past Kp: zero weights
        // (every load is unconditional, so that a wait counts only what it needs)
        const bool two = 128 * u + 64 < s.Kp;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const int8_t* p = b_row[nt] + (long long)u * 2048;
            d.w[0][nt] = *(const v4i*)p;
            d.w[1][nt] = *(const v4i*)(two ? p + 1024 : (const int8_t*)kZero16);
        }
        const int ka = 128 * u + 16 * fchunk;
        load_a(two ? ka + odd : ka, d.x[0]);
        load_a(two ? ka + (64 - odd) : (EP == SE_I32 ? s.Kp : ka), d.x[1]);
        if constexpr (EP == SE_I32)
            if (!two && odd) {   // (a row's one step is its first load)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    const v4i t = d.x[0][mt];
                    d.x[0][mt] = d.x[1][mt];
                    d.x[1][mt] = t;
                }
            }
    };
    // EPI_I32: this lane's part of the sums of its rows (a - a_sub) and
    // columns (b - b_sub), from the operands on their way to the MFMAs
    int rsum[MT], csum[NT];
    if constexpr (EP == SE_I32) {
#pragma unroll
        for (int i = 0; i < MT; ++i) rsum[i] = 0;
#pragma unroll
        for (int i = 0; i < NT; ++i) csum[i] = 0;
    }
    auto sum16 = [](const v4i& v, int acc0) {
        acc0 = __builtin_amdgcn_sdot4(v.x, 0x01010101, acc0, false);
        acc0 = __builtin_amdgcn_sdot4(v.y, 0x01010101, acc0, false);
        acc0 = __builtin_amdgcn_sdot4(v.z, 0x01010101, acc0, false);
        return __builtin_amdgcn_sdot4(v.w, 0x01010101, acc0, false);
    };
    auto mma_unit = [&](const Unit& d) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                v4i x;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    x[r] = (int)((uint32_t)(odd ? d.x[h ^ 1][mt][r] : d.x[h][mt][r]) ^ s.xmask);
                if constexpr (EP == SE_I32) {
                    rsum[mt] = sum16(x, rsum[mt]);
                    if (mt == 0) {
#pragma unroll
                        for (int nt = 0; nt < NT; ++nt) csum[nt] = sum16(d.w[h][nt], csum[nt]);
                    }
                }
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
                    acc[mt][nt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(d.w[h][nt], x, acc[mt][nt], 0, 0, 0);
            }
    };
    Unit ua, ub;
    // (W <= nunits: every wave has a unit)
    int u = wave;
    load_unit(u, ua);

    // ---- this thread's first chunk: its constants, behind the first operands
    // (NCHW stores run along the pixels, the others along the columns)
    const bool nchw = EP == SE_GEN && g.y_nchw;
    auto chunk_m = [&](int c) { return nchw ? c % BM : c / (BN / 4); };
    auto chunk_n = [&](int c) { return 4 * (nchw ? c / BM : c % (BN / 4)); };
    // (a row-major thread keeps its columns: its chunks are nthr apart, a
    // multiple of BN / 4)
    struct Cols { v4i c, p0, p1, beta; };
    auto load_cols = [&](int n, Cols& e) {
        // per-column arrays are padded to Np
        const long long po = (long long)z * s.param_bstride + n;
        e.c = *(const v4i*)(s.c + po);
        e.p0 = *(const v4i*)(s.p0 + po);
        if constexpr (EP == SE_DQ || EP == SE_GEN) e.p1 = *(const v4i*)(s.p1 + po);
        if constexpr (EP == SE_GEN) e.beta = *(const v4i*)(s.beta_col + po);
    };
    // what a chunk needs of its row: the residual bytes of a fused add (N %
    // 16 == 0 and rows 16-byte aligned), the zero-point sum
    auto load_row = [&](int m, int n) -> uint32_t {
        if (m >= s.M || n >= s.N) return 0u;
        if constexpr (EP == SE_RQB_ADD) return *(const uint32_t*)(g.add_other + (long long)m * s.ldy + n);
        if constexpr (EP == SE_GEN)
            if (g.rowsum) return (uint32_t)g.rowsum[(long long)z * g.rowsum_bstride + m];
        return 0u;
    };
    Cols e0;
    if (EP != SE_I32 && n0 + chunk_n(tid) < s.N && tid < CH) load_cols(n0 + chunk_n(tid), e0);
    uint32_t row_next = EP != SE_RQB_ADD && EP != SE_GEN ? 0u : load_row(m0 + chunk_m(tid), n0 + chunk_n(tid));

    for (; u + 2 * W < s.nunits; u += 2 * W) {
        load_unit(u + W, ub);
        mma_unit(ua);
        load_unit(u + 2 * W, ua);
        mma_unit(ub);
    }
    if (u + W < s.nunits) {
        load_unit(u + W, ub);
        mma_unit(ua);
        mma_unit(ub);
    } else {
        mma_unit(ua);
    }

    // ---- partial tiles to LDS: lane holds columns 16 nt + 4 fchunk .. + 3 of
    // row 16 mt + frow
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
            *(v4i*)(red + (wave * BM + 16 * mt + frow) * RS + 16 * nt + 4 * fchunk) = acc[mt][nt];
    int* const sums = red + W * BM * RS;   // SE_I32: [W][BM + BN]
    if constexpr (EP == SE_I32) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            int v = rsum[mt];
            v += __shfl_xor(v, 16, 64);
            v += __shfl_xor(v, 32, 64);
            if (fchunk == 0) sums[wave * (BM + BN) + 16 * mt + frow] = v;
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            int v = csum[nt];
            v += __shfl_xor(v, 16, 64);
            v += __shfl_xor(v, 32, 64);
            if (fchunk == 0) sums[wave * (BM + BN) + BM + 16 * nt + frow] = v;
        }
    }
    __syncthreads();

    // scalars of the call: with a device zero point array c is colsum and the
    // constant -alpha * colsum
    int alpha = 0, yzp = s.y_zp;
    float cm = 0.0f, dqs = 0.0f;
    constexpr bool LATE_ZP = EP == SE_DQ || EP == SE_I32 || EP == SE_GEN;
    if constexpr (LATE_ZP) {
        alpha = g.alpha;
        if (g.alpha_zp_dev)
            alpha = (g.a_xor ? (int)*(const uint8_t*)g.alpha_zp_dev : (int)*(const int8_t*)g.alpha_zp_dev) - g.a_sub;
        cm = g.cm;
        float cm_b = g.cm_b, cm_y = g.cm_y;
        if constexpr (EP == SE_DQ) {
            dqs = g.dq_scale;
            if (g.ngrp) {
                cm = g.grp_cm[z];
                yzp = g.grp_y_zp[z];
                dqs = g.grp_dq_scale[z];
                cm_b = g.grp_cm_b[z];
                cm_y = g.grp_cm_y[z];
            }
        }
        if (g.cm_a_scale_dev) {
            const float as = *g.cm_a_scale_dev;
            const float t1 = as * cm_b;
            cm = g.epi == EPI_I32S ? as : t1 / cm_y;
        }
    }
    float mm_mn = 0.0f, mm_mx = 0.0f;
    for (int c = tid; c < CH; c += nthr) {
        const int lm = chunk_m(c), ln = chunk_n(c);
        const int m = m0 + lm, n = n0 + ln;
        const uint32_t row_c = row_next;
        if ((EP == SE_RQB_ADD || EP == SE_GEN) && c + nthr < CH) row_next = load_row(m0 + chunk_m(c + nthr), n0 + chunk_n(c + nthr));
        if (m >= s.M || n >= s.N) continue;
        if (nchw && c != tid) load_cols(n, e0);
        v4i v = *(const v4i*)(red + lm * RS + ln);
        for (int w = 1; w < W; ++w) {
            const v4i p = *(const v4i*)(red + (w * BM + lm) * RS + ln);
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = wrap_add(v[r], p[r]);
        }
        const int nv = s.N - n < 4 ? s.N - n : 4;   // columns of this chunk
        long long yo = (long long)z * s.y_bstride + (long long)m * s.ldy + n;
        uint32_t word = 0;
        if constexpr (EP == SE_I32) {
            // sum (a - a_zp)(b - b_zp) = acc - alpha colsum - beta rowsum', the
            // row's sum of a - a_zp (a row's Kp - K padded bytes add 0)
            int row = 0;
            v4i col = v4i{0, 0, 0, 0};
            for (int w = 0; w < W; ++w) {
                row = wrap_add(row, sums[w * (BM + BN) + lm]);
                const v4i p = *(const v4i*)(sums + w * (BM + BN) + BM + ln);
#pragma unroll
                for (int r = 0; r < 4; ++r) col[r] = wrap_add(col[r], p[r]);
            }
            row = wrap_add(row, -wrap_mul(s.K, alpha));
#pragma unroll
            for (int r = 0; r < 4; ++r)
                v[r] = wrap_add(v[r], -wrap_add(wrap_mul(alpha, col[r]), wrap_mul(g.beta, row)));
            int32_t* y = (int32_t*)s.y + yo;
            if (nv == 4 && ((uintptr_t)y & 15) == 0) {
                *(v4i*)y = v;
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (r < nv) y[r] = v[r];
            }
            continue;
        }
        if constexpr (LATE_ZP) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                v[r] = wrap_add(v[r], g.c0 ? e0.c[r] : -wrap_mul(alpha, e0.c[r]));
                if (EP == SE_GEN && g.rowsum)
                    v[r] = wrap_add(v[r], -wrap_mul(g.beta_col ? e0.beta[r] : g.beta, (int32_t)row_c));
            }
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = wrap_add(v[r], e0.c[r]);
        }
        uint8_t* yb = (uint8_t*)s.y;
        if constexpr (EP == SE_RQB || EP == SE_RQB_ADD) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                word |= (rqb_fast(v[r], __int_as_float(e0.p0[r]), yzp, s.lo, s.hi) & 0xffu) << (8 * r);
        }
        if constexpr (EP == SE_RQB_ADD) {
            // QLinearAdd of the residual: RQ-E's body expression, or its
            // scalar tail from flat element add_body on
            uint32_t out = 0;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int q = (int)((word >> (8 * r)) & 0xffu), x = (int)((row_c >> (8 * r)) & 0xffu);
                const int a = g.add_conv_is_a ? q : x, b = g.add_conv_is_a ? x : q;
                float f;
                if (yo + r < g.add_body) {
                    f = __builtin_fmaf((float)b, g.add_sb, g.add_fixed);
                    f = __builtin_fmaf((float)a, g.add_sa, f);
                } else {
                    const float t1 = g.add_sa * (float)(a - g.add_a_zp);
                    const float t2 = g.add_sb * (float)(b - g.add_b_zp);
                    f = (t1 + t2) + (float)g.add_y_zp;
                }
                out |= (uint32_t)(clampi(x86_f2i(__builtin_rintf(f)), s.lo, s.hi) & 0xff) << (8 * r);
            }
            word = out;
        }
        if constexpr (EP == SE_DQ) {
            if (g.ngrp) {
                yb = (uint8_t*)g.grp_y[z];
                yo = (long long)m * s.ldy + n;
            }
            float o[4];
            const bool i32s = g.epi == EPI_I32S;
            if (i32s) {
                // MatMulInteger -> Cast -> Mul by fl(a_s * w_s[n]) -> Add(bias)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float f = (float)v[r] * (cm * __int_as_float(e0.p0[r]));
                    o[r] = g.dq_nobias ? f : f + __int_as_float(e0.p1[r]);
                }
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const uint32_t b = rqd_fast(v[r], cm, yzp, s.lo, s.hi) & 0xffu;
                    word |= b << (8 * r);
                    // DequantizeLinear, then the fp32 Add of the column bias
                    const float d = ((float)b - (float)yzp) * dqs;
                    o[r] = d + __int_as_float(e0.p1[r]);
                }
            }
            const bool f32_out = i32s || (g.dq_bias && !g.dq_codes);
            if (f32_out || g.mm_parts) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (g.dq_gelu) o[r] = gelu_erf(o[r]);
                    if (r < nv) {
                        mm_mn = fminf(mm_mn, o[r]);
                        mm_mx = fmaxf(mm_mx, o[r]);
                    }
                }
            }
            if (f32_out) {
                float* y = (float*)yb + yo;
                if (nv == 4 && ((uintptr_t)y & 15) == 0) {
                    *(float4*)y = make_float4(o[0], o[1], o[2], o[3]);
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (r < nv) y[r] = o[r];
                }
                continue;
            }
        }
        if constexpr (EP == SE_GEN) {
            // scalar-tail rows (TailMode)
            bool tail = false;
            if (g.tail != TAIL_NONE) {
                const int p = m - (int)fast_div((uint32_t)m, s.div_sp_mul, s.div_sp_shift) * s.sp_out;
                if (g.tail == TAIL_SPATIAL) {
                    tail = p >= (s.sp_out & ~15);
                } else {
                    const int oh = (int)fast_div((uint32_t)p, s.div_ow_mul, s.div_ow_shift);
                    const int oh0 = (oh / g.tile_h) * g.tile_h;
                    const int th = g.oH - oh0 < g.tile_h ? g.oH - oh0 : g.tile_h;
                    tail = p - oh0 * s.oW >= ((th * s.oW) & ~15);
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float q0 = __int_as_float(e0.p0[r]), q1 = __int_as_float(e0.p1[r]);
                uint32_t b;
                if (g.epi == EPI_RQB)
                    b = n + r >= g.bprime_from ? (uint32_t)rq_b_roundf(v[r], q0, yzp, s.lo, s.hi)
                                               : rqb_fast(v[r], q0, yzp, s.lo, s.hi);
                else if (g.epi == EPI_RQD)
                    b = rqd_fast(v[r], cm, yzp, s.lo, s.hi);
                else if (tail)
                    b = (uint32_t)rq_a_tail(v[r], q0, q1, g.inv_y, yzp, g.L, s.hi);
                else
                    b = rqa_fast(v[r], q0, q1, g.inv_y, yzp, g.L, s.hi);
                word |= (b & 0xffu) << (8 * r);
            }
            if (nchw) {
                const int img = (int)fast_div((uint32_t)m, s.div_sp_mul, s.div_sp_shift), p = m - img * s.sp_out;
                uint8_t* y = yb + (long long)z * s.y_bstride + ((long long)img * s.ldy + n) * s.sp_out + p;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (r < nv) y[(long long)r * s.sp_out] = (uint8_t)(word >> (8 * r));
                continue;
            }
        }
        uint8_t* y = yb + yo;
        if (nv == 4 && ((uintptr_t)y & 3) == 0) {
            *(uint32_t*)y = word;
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (r < nv) y[r] = (uint8_t)(word >> (8 * r));
        }
    }
    if constexpr (EP == SE_DQ) {
        if (g.mm_parts) {
            // one (min, max) pair per block; the pairs past the blocks get
            // (0, 0), which a range that includes 0 ignores
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) {
                mm_mn = fminf(mm_mn, __shfl_xor(mm_mn, off, 64));
                mm_mx = fmaxf(mm_mx, __shfl_xor(mm_mx, off, 64));
            }
            __syncthreads();   // every partial sum has been read
            float2* pr = (float2*)red;
            if (lane == 0) pr[wave] = make_float2(mm_mn, mm_mx);
            __syncthreads();
            if (tid == 0) {
                for (int w = 1; w < W; ++w) {
                    mm_mn = fminf(mm_mn, pr[w].x);
                    mm_mx = fmaxf(mm_mx, pr[w].y);
                }
                *(float2*)(g.mm_parts + 2 * (z * total + t)) = make_float2(mm_mn, mm_mx);
            }
            if (z == 0 && t == 0)
                for (int i = total * gridDim.z + tid; i < s.pairs; i += nthr)
                    *(float2*)(g.mm_parts + 2 * i) = make_float2(0.0f, 0.0f);
        }
    }
}

namespace {

// launch one instantiation with W waves a block
template <int MT, int NT, int AMODE, int VEC, int EP, int MAXW>
hipError_t launch_small(const GemmArgs& g, int batch, int W, hipStream_t st) {
    constexpr int BM = 16 * MT, BN = 16 * NT;
    SmallArgs s{};
    s.a = g.a; s.b = g.b_pieces; s.a_bstride = g.a_bstride; s.b_bstride = g.b_bstride;
    s.M = g.M; s.N = g.N; s.K = g.K; s.Kp = g.Kp;
    s.nbm = (g.M + BM - 1) / BM;
    s.nbn = (g.N + BN - 1) / BN;
    s.n_major = g.N >= g.M ? 1 : 0;
    fast_div_consts((uint32_t)(s.n_major ? s.nbm : s.nbn), &s.div_t_mul, &s.div_t_shift);
    s.lda = (int)g.lda;
    s.xmask = (uint32_t)g.a_xor * 0x01010101u;
    s.nunits = (g.Kp + 127) / 128;
    if (g.H > 0) {
        s.H = g.H; s.W = g.W; s.C = g.C; s.Cs = g.Cs; s.kW = g.kW; s.sH = g.sH; s.sW = g.sW; s.dH = g.dH; s.dW = g.dW;
        s.pad_t = g.pad_t; s.pad_l = g.pad_l;
        s.padw = (uint32_t)(g.pad_byte & 0xff) * 0x01010101u;
        fast_div_consts((uint32_t)g.C, &s.div_c_mul, &s.div_c_shift);
        fast_div_consts((uint32_t)g.kW, &s.div_kw_mul, &s.div_kw_shift);
    }
    if (g.oH > 0) {   // a convolution, 1x1 ones as dense GEMMs included
        s.oW = g.oW;
        s.sp_out = g.oH * g.oW;
        fast_div_consts((uint32_t)s.sp_out, &s.div_sp_mul, &s.div_sp_shift);
        fast_div_consts((uint32_t)g.oW, &s.div_ow_mul, &s.div_ow_shift);
    }
    s.c = g.c0 ? g.c0 : g.colsum;
    const float* any = (const float*)s.c;
    s.p0 = g.epi == EPI_RQB ? g.os : (g.cs ? g.cs : any);
    s.p1 = g.dq_bias ? g.dq_bias : (g.bf ? g.bf : any);
    s.beta_col = g.beta_col ? g.beta_col : s.c;
    s.param_bstride = g.param_bstride;
    s.y = g.y; s.ldy = g.ldy; s.y_bstride = g.y_bstride;
    s.y_zp = g.y_zp; s.lo = g.lo; s.hi = g.hi;
    s.pairs = (int)qgemm_pairs(g, batch);
    if (W > s.nunits) W = s.nunits;
    if (W > MAXW) W = MAXW;
    const long long tiles = (long long)s.nbm * s.nbn;
    if (tiles > 0x7ffffff0LL) return hipErrorInvalidValue;
    const dim3 grid((unsigned)(8 * ((tiles + 7) / 8)), 1, (unsigned)batch);
    const size_t lds = sizeof(int) * (size_t)W * (BM * (BN + 4) + (EP == SE_I32 ? BM + BN : 0));
    hipLaunchKernelGGL((qgemm_small_kernel<MT, NT, AMODE, VEC, EP, MAXW>), grid, dim3(W * 64), lds, st, s, g);
    return hipGetLastError();
}

// Tile and waves of a shape: the largest tile that still gives 190 blocks (of
// 256 CUs) and 760 waves, 16 x 16 if none does. Up to K = 256 no more than 32
// x 32: with one or two units of K the epilogue is most of the work, and its
// lanes are the block's. As many waves as K has units for, up to about 8 a CU.
// max_tiles: the (min, max) pairs of a launch that writes them, one a block;
// 64 x 64 tiles are never more than those pairs (4 per 128 x 128 or 256 x 64).
struct SmallPlan { int mt, nt, waves; };
SmallPlan small_plan(int M, int N, int Kp, int batch, long long max_tiles) {
    static const int T[5][3] = {{4, 4, 4}, {2, 4, 8}, {2, 2, 16}, {1, 2, 16}, {1, 1, 16}};
    const int units = (Kp + 127) / 128;
    SmallPlan p{};
    for (int i = max_tiles ? 0 : 1; i < 5; ++i) {
        const int mt = T[i][0], nt = T[i][1];
        const long long tiles = (long long)((M + 16 * mt - 1) / (16 * mt)) * ((N + 16 * nt - 1) / (16 * nt)) * batch;
        if (max_tiles) {
            if (tiles > max_tiles) break;
        } else if ((nt == 4 && units <= 2) || 8 * nt >= N + (nt == 1 ? 8 : 0)) {
            continue;
        }
        int w = 1;
        while (2 * w <= T[i][2] && 2 * w <= units && tiles * 2 * w <= 2500) w *= 2;
        p = SmallPlan{mt, nt, w};
        if (tiles >= 190 && tiles * w >= 760) break;
    }
    return p;
}

template <int AMODE, int VEC, int EP>
hipError_t launch_small_tile(const GemmArgs& g, int batch, hipStream_t s) {
    const SmallPlan p = small_plan(g.M, g.N, g.Kp, batch, g.mm_parts ? qgemm_pairs(g, batch) : 0);
    if (prof_enabled()) {
        char nm[96];
        snprintf(nm, sizeof(nm), "variant:small<%d,%d,%d,%d,%d>", p.mt, p.nt, AMODE, VEC, EP);
        prof_count(nm);
    }
    switch (p.mt * 8 + p.nt) {
    case 4 * 8 + 4:
        if constexpr (EP == SE_DQ) return launch_small<4, 4, AMODE, VEC, EP, 4>(g, batch, p.waves, s);
        return hipErrorInvalidValue;
    case 2 * 8 + 4: return launch_small<2, 4, AMODE, VEC, EP, 8>(g, batch, p.waves, s);
    case 2 * 8 + 2: return launch_small<2, 2, AMODE, VEC, EP, 16>(g, batch, p.waves, s);
    case 1 * 8 + 2: return launch_small<1, 2, AMODE, VEC, EP, 16>(g, batch, p.waves, s);
    default: return launch_small<1, 1, AMODE, VEC, EP, 16>(g, batch, p.waves, s);
    }
}

// Outputs up to which this kernel is the faster one, as its time over the other
// kernel's at thousands of outputs (graphs of calls whose operands come from the
// Infinity Cache, as a layer's do; N = 16 .. 3072, 7 .. 56 pixels). Against the
// register-staged kernel at any K up to 3.3 M: NCHW 3x3 0.34 at 1000, 0.67 at
// 3250, K % 16 != 0 0.35, 0.5; with a weight zero point 0.90 at 2800, 1.04 at 3250.
constexpr long long SMALL_MAX_OUT_REG = 3300000, SMALL_MAX_OUT_ROWSUM = 2800000;

// Against the pipelined and direct kernels:
long long small_max_out(const GemmArgs& g, int batch) {
    const int K = g.Kp;
    if (g.epi == EPI_I32) return 1650000;   // 0.77 at 1600 with its pass over B
    if (g.mm_parts) {
        // the (min, max) pairs allow few tiles smaller than 64 x 64. With Gelu K =
        // 64 and 128 1.25 at any size; 192 0.80 and 256 0.85 to 1600, 1.45 at 2200;
        // 768 0.53 at 1000, 0.95 at 1600, 1.3 at 2200. Without, the epilogue does
        // not cover a second round of blocks on the 256 CUs: K = 512 and more 0.70
        // up to one, 1.2 past it (3072 0.94); 320 and 384 0.95, 1.04; 192 and 256 1.0
        // +- 0.1
        if (g.dq_gelu) return K < 192 ? 0 : 1650000;
        return K < 320 ? 0 : K < 2048 ? 256 * 64 * 64 : 1650000;
    }
    if (g.dq_bias) return 1650000;   // fp32 chains 0.85 at 1600, K = 32 .. 3072
    // convolution groups of 64 channels, 3x3 0.67 at 1000, 1.02 at 1250; 1x1 of
    // K = 128 0.87 at 600, 1.16 at 800; of 32 0.92 at 1250, 1.2 at 1600; of 16
    // 0.84 at 1600
    if (batch > 1 && g.oH > 0) return g.N <= 16 ? 1650000 : g.N <= 32 ? 1300000 : K < 256 ? 700000 : 1220000;
    if (g.epi == EPI_RQD) {
        if (g.N < 64) return K <= 64 ? 1350000 : 1650000;   // 0.95 at 1250, 1.02 at 1600; 256 0.8
        // K = 64 0.96 at 600, 1.12 at 800; 128 0.93 at 800, 1.07 at 1000; 256 0.95
        // at 1000, 1.0 at 1250; 320 and 384 (three units of K on two waves) 0.86
        // at 600, 1.02 at 800; 512 .. 3072 0.92 at 1250, 1.10 at 1600
        return K <= 64 ? 650000 : K <= 128 ? 850000 : K <= 256 ? 1200000 : K <= 384 ? 750000 : 1350000;
    }
    if (g.add_other) {
        // K = 64 0.97 at 800, 1.05 at 1200, but 0.76 at 1600 where theirs holds the
        // weights in registers; 128 0.92 at 800, 1.0 at 1200; 192 and 256 0.82 at
        // 1250, 1.0 at 1600; 320 and 384 0.93 at 1000, 1.0 at 1250; 512 .. 2048 0.90
        // at 1600
        if (K == 64 && g.N > 64 && g.M > 128 * 31) return 1650000;
        return K <= 64 ? 1000000 : K <= 128 ? 1250000 : K <= 256 ? 1500000 : K < 512 ? 1250000 : 1650000;
    }
    // K = 64 0.95 at 1200, 1.0 .. 1.1 at 1600 (16 channels 0.9); 128 0.74, 256 0.86,
    // 1152 0.92 at 1600; 2048, 2304 and 4608 0.92 at 1250, 1.03 at 1600
    return K <= 64 ? (g.N <= 16 ? 1650000 : 1200000) : K < 2048 ? 1650000 : 1450000;
}

}  // namespace

// (a fused epilogue is refused where the pipelined kernel refuses it)
static bool small_modes(const GemmArgs& g, int batch, bool pipelined) {
    if (!g.b_pieces || g.kWp > 0 || g.row_coef || g.epi == EPI_RQC || g.tail == TAIL_OW) return false;
    if (g.epi == EPI_I32 ? !g.sums_inline || g.H > 0 : g.c0 == nullptr && g.colsum == nullptr) return false;
    if ((g.add_other || g.dq_bias) && !pipelined) return false;
    if (batch > 65535 || g.lda > 0x7fffffffLL) return false;
    if (!pipelined)
        return (long long)g.M * g.N * batch <=
               (g.rowsum && g.epi != EPI_I32 ? SMALL_MAX_OUT_ROWSUM : SMALL_MAX_OUT_REG);
    // (a count of 64 x 64 blocks decides there)
    const bool blocks = g.mm_parts && !g.dq_gelu;
    const long long m = blocks ? (g.M + 63) & ~63 : g.M, n = blocks ? (g.N + 63) & ~63 : g.N;
    return m * n * batch <= small_max_out(g, batch);
}

bool qgemm_small_size(long long outputs) { return outputs <= SMALL_MAX_OUT_REG; }

bool qgemm_small_eligible(const GemmArgs& g, int batch, int vec) {
    return small_modes(g, batch, qgemm_dma_eligible(g, vec) || qgemm_direct_eligible(g, batch));
}

hipError_t launch_qgemm_small(const GemmArgs& g, int batch, int vec, hipStream_t s) {
    const bool rqb = g.epi == EPI_RQB && g.c0 && !g.rowsum && g.tail == TAIL_NONE && !g.y_nchw && g.bprime_from >= g.N;
    const bool rqd = (g.epi == EPI_RQD && !g.rowsum) || g.epi == EPI_I32S;
    if (g.H > 0) {
        switch (vec) {
        case 16:
            if (g.add_other) return launch_small_tile<A_CONV, 16, SE_RQB_ADD>(g, batch, s);
            return rqb ? launch_small_tile<A_CONV, 16, SE_RQB>(g, batch, s)
                       : launch_small_tile<A_CONV, 16, SE_GEN>(g, batch, s);
        case 8: return launch_small_tile<A_CONV, 8, SE_GEN>(g, batch, s);
        case 4: return launch_small_tile<A_CONV, 4, SE_GEN>(g, batch, s);
        default: return launch_small_tile<A_CONV, 1, SE_GEN>(g, batch, s);
        }
    }
    if (g.epi == EPI_I32)
        return vec == 16 ? launch_small_tile<A_DENSE, 16, SE_I32>(g, batch, s)
                         : launch_small_tile<A_DENSE, 1, SE_I32>(g, batch, s);
    if (vec == 16) {
        if (g.add_other) return launch_small_tile<A_DENSE, 16, SE_RQB_ADD>(g, batch, s);
        if (rqd) return launch_small_tile<A_DENSE, 16, SE_DQ>(g, batch, s);
        return rqb ? launch_small_tile<A_DENSE, 16, SE_RQB>(g, batch, s)
                   : launch_small_tile<A_DENSE, 16, SE_GEN>(g, batch, s);
    }
    if (vec == 8)
        return rqb ? launch_small_tile<A_DENSE, 8, SE_RQB>(g, batch, s)
                   : launch_small_tile<A_DENSE, 8, SE_GEN>(g, batch, s);
    return launch_small_tile<A_DENSE, 1, SE_GEN>(g, batch, s);
}

}  // namespace nnrh
