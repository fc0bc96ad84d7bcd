// The dense side of a GAT layer around its one large product (feat @ W: fgnn_tall.hip where the scores come out of it as columns, a
// library product and gat_score_kernel elsewhere): the score weights folded out
// of W and the attention vectors, the scores of all nodes, and the gradients unfolded again
// (layers/gatconv_layer.py:50-55 of the reference: h = feat @ W, attn_row = (attn_l * h).sum(-1), attn_col = (attn_r * h).sum(-1)).
// The scores are taken as feat @ ((W * attn).sum(-1)), the same sums in another order: `feat` is read instead of the
// wider h.  Composed from tensor operations this was 11 launches before the sparse operator and 9 after it.
#include "fgnn_common.h"

typedef float gd_f4 __attribute__((ext_vector_type(4)));
typedef float gd_f4u __attribute__((ext_vector_type(4), aligned(4)));        // four floats at any float: one 128-bit load all the same

// One workgroup per input feature i.  score_wt [2H, fin] gets sum_f W[i,h,f] * attn_l[h,f], then the same for attn_r (transposed, so that
// the score kernel reads four consecutive k of a column at once); proj [fin, H*Fp] (NULL: not wanted) W with `pad` zero columns per
// head; all [fin, H*Fp + 2H] (NULL) the two side by side, the operand of the input's gradient.  Bound by its launch (W is a few
// hundred kilobytes), so the sums are free to run in 64 bits: whatever the order, they are no further off than a reduction
// of the products.
__global__ __launch_bounds__(256) void gat_fold_kernel(int fin, int H, int F, int pad, const float *__restrict__ W, const float *__restrict__ al,
                                                       const float *__restrict__ ar, float *__restrict__ score_wt, float *__restrict__ proj,
                                                       float *__restrict__ all)
{
    const int i = (int)blockIdx.x, Fp = F + pad, lda = H * Fp + 2 * H;
    const float *w = W + (size_t)i * H * F;
    for (int c = (int)threadIdx.x; c < H * Fp; c += 256) {
        const int h = c / Fp, f = c - h * Fp;
        const float v = f < F ? w[h * F + f] : 0.f;
        if (proj) proj[(size_t)i * H * Fp + c] = v;
        if (all) all[(size_t)i * lda + c] = v;
    }
    for (int h = fg_wave(); h < H; h += 4) {
        double dl = 0., dr = 0.;
        for (int f = fg_lane(); f < F; f += 64) {
            const double v = w[h * F + f];
            dl = fma(v, (double)al[h * F + f], dl);
            dr = fma(v, (double)ar[h * F + f], dr);
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) { dl += __shfl_xor(dl, off); dr += __shfl_xor(dr, off); }
        if (fg_lane() == 0) {
            const float l = (float)dl, r = (float)dr;
            score_wt[(size_t)h * fin + i] = l;
            score_wt[(size_t)(H + h) * fin + i] = r;
            if (all) { all[(size_t)i * lda + H * Fp + h] = l; all[(size_t)i * lda + H * Fp + H + h] = r; }
        }
    }
}

extern "C" int fgnn_gat_fold_weights(int fin, int H, int F, int pad, const float *W, const float *attn_l, const float *attn_r, float *score_wt,
                                     float *proj, float *all, void *stream)
{
    FGNN_REQUIRE(fin >= 0 && H >= 1 && F >= 1 && pad >= 0 && (int64_t)H * (F + pad + 2) <= (1 << 28), FGNN_ERR_SHAPE,
                 "fgnn_gat_fold_weights: bad sizes fin=%d H=%d F=%d pad=%d", fin, H, F, pad);
    FGNN_REQUIRE(fin == 0 || (W && attn_l && attn_r && score_wt), FGNN_ERR_NULL, "fgnn_gat_fold_weights: NULL argument");
    if (fin == 0) return 0;
    hipLaunchKernelGGL(gat_fold_kernel, dim3((unsigned)fin), dim3(256), 0, (hipStream_t)stream, fin, H, F, pad, W, attn_l, attn_r, score_wt, proj, all);
    return fgnn_launch_status("gat_fold_kernel");
}

// attn_row [n, H] and attn_col [n, H] = feat [n, K] @ score_wt^T: a thin product, bound by reading feat once.  16 x 16 x 4 matrix
// instructions, rows = nodes, columns = 2H scores in NT tiles of 16; lane (r, q) of a chunk of 16 dimensions reads four
// consecutive floats of node r and of score column r, and the chunk's four instructions take the first to fourth of them (both operands
// permuted alike).  KS waves share a tile's dimensions and add up in LDS: 4 where the
// nodes alone would leave compute units idle, else 1.  Against the library product and the two copies
// that split it: 2.45 M nodes x 100, 8 heads 430 -> 310 us (196 us to read feat at 5 TB/s); 233 k x 602 217 -> 174; 2708 x 1433, 1 head 32 -> 14;
// with more than 8 heads the weights' loads weigh in: 100 k x 64, 32 heads 39 -> 24, 30 k x 602, 16 heads 32 -> 37 us.
// Every 64 dimensions form a sum of their own: one chain over all of them was up to twice as far from the float64 scores as
// the library product (100 k x 602, 8 heads: 4.4e-7 against 2.2e-7; 1433, 2 heads: 6.8e-7 against 3.4e-7).
template <int NT, int KS>
__global__ __launch_bounds__(256) void gat_score_kernel(int64_t n, int K, int H, const float *__restrict__ feat, const float *__restrict__ wt,
                                                        float *__restrict__ arow, float *__restrict__ acol)
{
    __shared__ gd_f4 part[KS > 1 ? 3 * NT * 64 : 1];
    const int lane = fg_lane(), wave = fg_uni(fg_wave()), r16 = lane & 15, kq = lane >> 4;
    const int64_t tile = KS > 1 ? (int64_t)blockIdx.x : (int64_t)blockIdx.x * 4 + wave;
    if (tile * 16 >= n) return;                 // KS > 1: the whole workgroup (and the grid has no such workgroup)
    const int64_t node = tile * 16 + r16 < n ? tile * 16 + r16 : n - 1;
    const float *a_row = feat + (size_t)node * K;
    auto frag = [&](const float *p, int k, bool ok) {           // elements k .. k + 3, zero past the end
        gd_f4 v = {0.f, 0.f, 0.f, 0.f};
        if (ok && k + 4 <= K) v = *reinterpret_cast<const gd_f4u *>(p + k);
        else if (ok && k < K) {
#pragma unroll
            for (int u = 0; u < 3; ++u) if (k + u < K) v[u] = p[k + u];
        }
        return v;
    };
    gd_f4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = gd_f4{0.f, 0.f, 0.f, 0.f};
    constexpr int U = 4;                        // chunks in flight
    for (int c0 = (KS > 1 ? wave : 0) * 16; c0 < K; c0 += 16 * KS * U) {
        gd_f4 a[U], b[U][NT];
#pragma unroll
        for (int u = 0; u < U; ++u) a[u] = frag(a_row, c0 + 16 * KS * u + 4 * kq, true);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int col = t * 16 + r16;
                b[u][t] = frag(wt + (size_t)(col < 2 * H ? col : 0) * K, c0 + 16 * KS * u + 4 * kq, col < 2 * H);
            }
        gd_f4 sum[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) sum[t] = gd_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int t = 0; t < NT; ++t) sum[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][e], b[u][t][e], sum[t], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] += sum[t];
    }
    if constexpr (KS > 1) {
        if (wave) {
#pragma unroll
            for (int t = 0; t < NT; ++t) part[((wave - 1) * NT + t) * 64 + lane] = acc[t];
        }
        __syncthreads();
        if (wave) return;
#pragma unroll
        for (int w = 0; w < 3; ++w)
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[t] += part[(w * NT + t) * 64 + lane];
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int col = t * 16 + r16;           // the product's column; its rows are 4 kq .. 4 kq + 3
        if (col >= 2 * H) continue;
        float *dst = col < H ? arow + col : acol + (col - H);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int64_t m = tile * 16 + 4 * kq + r;
            if (m < n) dst[(size_t)m * H] = acc[t][r];
        }
    }
}

extern "C" int fgnn_gat_scores(int64_t n, int K, int H, const float *feat, const float *score_wt, float *attn_row, float *attn_col, void *stream)
{
    FGNN_REQUIRE(n >= 0 && K >= 0 && H >= 1, FGNN_ERR_SHAPE, "fgnn_gat_scores: bad sizes n=%lld K=%d H=%d", (long long)n, K, H);
    FGNN_REQUIRE(H <= 32 && K <= (1 << 28), FGNN_ERR_LIMIT, "fgnn_gat_scores: H=%d K=%d unsupported (at most 32 heads)", H, K);
    FGNN_REQUIRE(n == 0 || (attn_row && attn_col && (K == 0 || (feat && score_wt))), FGNN_ERR_NULL, "fgnn_gat_scores: NULL argument");
    if (n == 0) return 0;
    const int64_t tiles = (n + 15) / 16;
    FGNN_REQUIRE(tiles <= 2147483647LL, FGNN_ERR_LIMIT, "fgnn_gat_scores: too many rows");
    const bool split = tiles < 16 * 256 && K >= 64;      // under four waves per SIMD from the nodes alone
    const unsigned grid = (unsigned)(split ? tiles : (tiles + 3) / 4);
    hipStream_t st = (hipStream_t)stream;
    auto go = [&]<int NT>() {
        if (split) hipLaunchKernelGGL((gat_score_kernel<NT, 4>), dim3(grid), dim3(256), 0, st, n, K, H, feat, score_wt, attn_row, attn_col);
        else hipLaunchKernelGGL((gat_score_kernel<NT, 1>), dim3(grid), dim3(256), 0, st, n, K, H, feat, score_wt, attn_row, attn_col);
    };
    if (H <= 8) go.template operator()<1>();
    else if (H <= 16) go.template operator()<2>();
    else go.template operator()<4>();
    return fgnn_launch_status("gat_score_kernel");
}

// The gradients of W, attn_l and attn_r from that of the padded projection (dproj, rows ldp floats apart) and of the score weights
// (dscore [fin, 2H], rows lds apart):
//   dW[i,h,f] = dproj[i,h,f] + dscore[i,h] * attn_l[h,f] + dscore[i,H+h] * attn_r[h,f],   dattn_l[h,f] = sum_i W[i,h,f] * dscore[i,h]  (r alike).
// One launch: the first row_blocks workgroups write dW, each of the others sums 64 columns over the rows, 16 waves side by side in a
// fixed order and in 64 bits: in 32, the chain of fin / 16 terms was further from the float64 sums than the reduction that it
// replaced (fin = 1433: 1.8e-7 against 0.9e-7, 3703: 2.7e-7 against 1.0e-7), and nothing here waits for the arithmetic.
#define GU_TPB 1024
__global__ __launch_bounds__(GU_TPB) void gat_unfold_kernel(int fin, int H, int F, int pad, int row_blocks, const float *__restrict__ W, const float *__restrict__ al,
                                                            const float *__restrict__ ar, const float *__restrict__ dproj, int ldp,
                                                            const float *__restrict__ dscore, int lds, float *__restrict__ dW, float *__restrict__ dal,
                                                            float *__restrict__ dar)
{
    __shared__ double sl[GU_TPB], sr[GU_TPB];
    const int HF = H * F, Fp = F + pad;
    if ((int)blockIdx.x < row_blocks) {
        const int64_t total = (int64_t)fin * HF;
        for (int64_t t = (int64_t)blockIdx.x * GU_TPB + threadIdx.x; t < total; t += (int64_t)row_blocks * GU_TPB) {
            const int i = (int)(t / HF), c = (int)(t - (int64_t)i * HF), h = c / F;
            const float *s = dscore + (size_t)i * lds;
            dW[t] = fmaf(s[H + h], ar[c], fmaf(s[h], al[c], dproj[(size_t)i * ldp + h * Fp + (c - h * F)]));
        }
        return;
    }
    const int lane = fg_lane(), wave = fg_wave(), c = ((int)blockIdx.x - row_blocks) * 64 + lane;
    const int h = c < HF ? c / F : 0;
    double l = 0., r = 0.;
    if (c < HF) {
#pragma unroll 4
        for (int i = wave; i < fin; i += GU_TPB / 64) {
            const double w = W[(size_t)i * HF + c];
            l = fma(w, (double)dscore[(size_t)i * lds + h], l);
            r = fma(w, (double)dscore[(size_t)i * lds + H + h], r);
        }
    }
    sl[wave * 64 + lane] = l;
    sr[wave * 64 + lane] = r;
    __syncthreads();
    if (wave || c >= HF) return;
    for (int w = 1; w < GU_TPB / 64; ++w) { l += sl[w * 64 + lane]; r += sr[w * 64 + lane]; }
    dal[c] = (float)l;
    dar[c] = (float)r;
}

extern "C" int fgnn_gat_unfold_grads(int fin, int H, int F, int pad, const float *W, const float *attn_l, const float *attn_r, const float *dproj, int ldp,
                                     const float *dscore, int lds, float *dW, float *dattn_l, float *dattn_r, void *stream)
{
    FGNN_REQUIRE(fin >= 0 && H >= 1 && F >= 1 && pad >= 0 && (int64_t)H * (F + pad + 2) <= (1 << 28) && ldp >= H * (F + pad) && lds >= 2 * H, FGNN_ERR_SHAPE,
                 "fgnn_gat_unfold_grads: bad sizes fin=%d H=%d F=%d pad=%d ldp=%d lds=%d", fin, H, F, pad, ldp, lds);
    FGNN_REQUIRE(dattn_l && dattn_r && attn_l && attn_r && (fin == 0 || (W && dproj && dscore && dW)), FGNN_ERR_NULL, "fgnn_gat_unfold_grads: NULL argument");
    const int64_t need = ((int64_t)fin * H * F + GU_TPB - 1) / GU_TPB;
    const int row_blocks = (int)(need < 512 ? need : 512), col_blocks = (H * F + 63) / 64;
    hipLaunchKernelGGL(gat_unfold_kernel, dim3((unsigned)(row_blocks + col_blocks)), dim3(GU_TPB), 0, (hipStream_t)stream, fin, H, F, pad, row_blocks, W, attn_l,
                       attn_r, dproj, ldp, dscore, lds, dW, dattn_l, dattn_r);
    return fgnn_launch_status("gat_unfold_kernel");
}
