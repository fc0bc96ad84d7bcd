// Brute-force k-nearest-neighbour graph builder for batched point clouds (the graph the fused
// EdgeConv consumes).  The reference builds it with DGL's KNNGraph on every layer of its DGCNN
// loop (script/train/train_edgeconv_our.py:51-55): per cloud, for every point the k nearest points
// of the same cloud, the point itself included, grouped by destination.
//
//
// A wave owns KNN_QW query points at a time and all 64 lanes share them: lane l holds the running
// squared distances from each of the queries to 4*RG candidate points in registers (candidates
// 4l..4l+3 of every 256-point group of the tile).  The candidate coordinates of a tile stream
// through LDS in slices of KNN_DC dimensions, transposed ([dimension][point]) so that a lane
// fetches its 4 candidates with one 128-bit LDS read and uses them for all KNN_QW queries; the
// query coordinates are wave-uniform and come through scalar registers.  Distances accumulate
// dimension by dimension in ascending order with one subtract and one fma each, so a point is at
// distance exactly 0 from itself.
//
// Selection (k <= 64): a threshold that at least k candidates pass, the k-th smallest of lane minima; the candidates under it
// (usually k to 1.3 k of the 1024) are compacted into LDS with ballots and ordered by a merge sort over the wave, whose exchanges
// stay on the vector ALU.  When more than 128 pass, mostly candidates at equal distances, the list takes those below the threshold and the
// k smallest ids of those at it.  Where even that is too long, and for 64 < k <= 128, the selection runs k extraction rounds
// instead: wave-wide minimum (DPP butterfly), holder with the smallest node id by ballots, retire it.  Either way the order is
// total (smaller distance first, smaller node id on equal distance), so the result is deterministic.  Clouds with more points than
// one tile keep the best k of the tiles seen so far in registers and run them through the next tile's selection, where they win ties
// because their ids are smaller.  65536 queries on 1024 points of 3 dimensions: 187 -> 120 us at k = 20 (sorts by ds_bpermute
// before), 406 -> 135 us at k = 40 (a list of 64 entries before, which a third of the queries overran into the rounds); k = 64 in
// 64 dimensions 1135 -> 436 us.
#include "fgnn_common.h"
#include <float.h>
#include <type_traits>

#define KNN_QW 4         // queries a wave processes together
#define KNN_WAVES 4      // waves per workgroup
#define KNN_DC 8         // dimensions per LDS slice
#define KNN_MAX_K 128    // KR = 2 result registers per lane
#define KNN_CAP 128      // candidates a selection orders without extraction rounds
#define KNN_ONE_GROUP 32 // up to this k the threshold comes from one minimum per lane, above it from two

// Takes the k best of {prior list (pd, pi), the tile's distances} in order; the new list replaces
// the prior one.  List position p lives in lane p % 64 of register p / 64.
template <int NR, int KR>
__device__ __forceinline__ void knn_select_rounds(float (&dist)[NR], int tile0, float (&pd)[KR], int (&pi)[KR], int k, int lane, int fallback_id)
{
    float nd[KR];
    int ni[KR];
#pragma unroll
    for (int t = 0; t < KR; ++t) { nd[t] = INFINITY; ni[t] = fallback_id; }
    for (int j = 0; j < k; ++j) {
        float lm = dist[0];
#pragma unroll
        for (int r = 1; r < NR; ++r) lm = fminf(lm, dist[r]);
#pragma unroll
        for (int t = 0; t < KR; ++t) lm = fminf(lm, pd[t]);
        const float m = -fg_wave_max(-lm);
        int id = fallback_id;
        bool found = false;
#pragma unroll
        for (int t = 0; t < KR; ++t) {
            if (!found) {
                unsigned long long b = __ballot(pd[t] == m);
                if (b) {
                    int L = __builtin_ctzll(b);
                    id = __builtin_amdgcn_readlane(pi[t], L);
                    if (lane == L) pd[t] = INFINITY;
                    found = true;
                }
            }
        }
#pragma unroll
        for (int g = 0; g < NR / 4; ++g) {
            if (!found) {
                unsigned long long b0 = __ballot(dist[4 * g] == m), b1 = __ballot(dist[4 * g + 1] == m);
                unsigned long long b2 = __ballot(dist[4 * g + 2] == m), b3 = __ballot(dist[4 * g + 3] == m);
                unsigned long long any = b0 | b1 | b2 | b3;
                if (any) {
                    int L = __builtin_ctzll(any);
                    int i = ((b0 >> L) & 1) ? 0 : ((b1 >> L) & 1) ? 1 : ((b2 >> L) & 1) ? 2 : 3;
                    id = tile0 + g * 256 + L * 4 + i;
                    if (lane == L) {
#pragma unroll
                        for (int u = 0; u < 4; ++u) if (i == u) dist[4 * g + u] = INFINITY;
                    }
                    found = true;
                }
            }
        }
#pragma unroll
        for (int t = 0; t < KR; ++t)
            if ((j >> 6) == t && lane == (j & 63)) { nd[t] = m; ni[t] = id; }
    }
#pragma unroll
    for (int t = 0; t < KR; ++t) { pd[t] = nd[t]; pi[t] = ni[t]; }
}

// Value of lane ^ X.  Inside a row of 16 lanes the exchange is one or two DPP moves; rows and halves of the wave change places
// through the row swap instructions, so nothing here waits for the LDS pipe (as ds_bpermute does).
template <int X>
__device__ __forceinline__ unsigned knn_xor(unsigned v, int lane)
{
    if constexpr (X == 1) return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xf, 0xf, true);
    else if constexpr (X == 2) return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xf, 0xf, true);
    else if constexpr (X == 3) return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x1B, 0xf, 0xf, true);
    else if constexpr (X == 7) return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xf, 0xf, true);
    else if constexpr (X == 8) return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xf, 0xf, true);
    else if constexpr (X == 15) return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xf, 0xf, true);
    else if constexpr (X == 4) return knn_xor<3>(knn_xor<7>(v, lane), lane);
    else if constexpr (X == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);      // [0]: the even rows twice, [1]: the odd rows twice
        return (lane & 16) ? r[0] : r[1];
    } else if constexpr (X == 32) {
        const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);      // [0]: the lower half twice, [1]: the upper half twice
        return (lane & 32) ? r[0] : r[1];
    } else if constexpr (X == 31) return knn_xor<16>(knn_xor<15>(v, lane), lane);
    else return knn_xor<32>(knn_xor<31>(v, lane), lane);        // 63
}

// One step of a merge sort: lanes l and l ^ X compare, the lane without the highest bit of X keeps the smaller.
template <int X>
__device__ __forceinline__ void knn_step(float &d, int lane)
{
    const float o = __uint_as_float(knn_xor<X>(__float_as_uint(d), lane));
    constexpr int top = X >= 32 ? 32 : X >= 16 ? 16 : X >= 8 ? 8 : X >= 4 ? 4 : X >= 2 ? 2 : 1;
    d = (lane & top) ? fmaxf(d, o) : fminf(d, o);
}
template <int X>
__device__ __forceinline__ void knn_step(float &d, int &i, int lane)
{
    const float od = __uint_as_float(knn_xor<X>(__float_as_uint(d), lane));
    const int oi = (int)knn_xor<X>((unsigned)i, lane);
    constexpr int top = X >= 32 ? 32 : X >= 16 ? 16 : X >= 8 ? 8 : X >= 4 ? 4 : X >= 2 ? 2 : 1;
    const bool other_smaller = od < d || (od == d && oi < i);
    if (((lane & top) == 0) == other_smaller) { d = od; i = oi; }
}
// Sorts one value (or one (distance, id) pair) per lane over the wave, ascending.  The first step of every doubling compares
// with the mirrored lane, so all steps sort the same way.
#define KNN_MERGE_64(...) knn_step<16>(__VA_ARGS__); knn_step<8>(__VA_ARGS__); knn_step<4>(__VA_ARGS__); knn_step<2>(__VA_ARGS__); knn_step<1>(__VA_ARGS__)
#define KNN_SORT_64(...)                                                                                                         \
    knn_step<1>(__VA_ARGS__);                                                                                                    \
    knn_step<3>(__VA_ARGS__); knn_step<1>(__VA_ARGS__);                                                                          \
    knn_step<7>(__VA_ARGS__); knn_step<2>(__VA_ARGS__); knn_step<1>(__VA_ARGS__);                                                \
    knn_step<15>(__VA_ARGS__); knn_step<4>(__VA_ARGS__); knn_step<2>(__VA_ARGS__); knn_step<1>(__VA_ARGS__);                     \
    knn_step<31>(__VA_ARGS__); knn_step<8>(__VA_ARGS__); knn_step<4>(__VA_ARGS__); knn_step<2>(__VA_ARGS__); knn_step<1>(__VA_ARGS__); \
    knn_step<63>(__VA_ARGS__); KNN_MERGE_64(__VA_ARGS__)

// The k-th smallest of the minima of 64 lanes (or of 128 half lanes): at least k candidates pass it.  The more groups the minima
// come from, the fewer candidates pass beyond k: of 1024 candidates 24 pass 64 groups at k = 20 and 61 at k = 40, where 128
// groups leave 47.  minimum(from, to) is the lane's minimum over its registers [from, to).
template <int NR, typename Min>
__device__ __forceinline__ float knn_threshold(float prior, int k, int lane, Min minimum)
{
    float a = fminf(minimum(0, NR / 2), prior), b = minimum(NR / 2, NR);
    if (k <= KNN_ONE_GROUP) {
        a = fminf(a, b);
        KNN_SORT_64(a, lane);
        return fg_readlane(a, k - 1);
    }
    KNN_SORT_64(a, lane);
    KNN_SORT_64(b, lane);
    a = fminf(a, __uint_as_float(knn_xor<63>(__float_as_uint(b), lane)));       // the 64 smallest of both, as one bitonic sequence
    knn_step<32>(a, lane);
    KNN_MERGE_64(a, lane);
    return fg_readlane(a, k - 1);
}

// Orders the cnt <= KNN_CAP entries of a wave's list in LDS and leaves the first 64 of them in (d, i), ascending by (d, i).
__device__ __forceinline__ void knn_order(const float2 *list, int cnt, int lane, float &d, int &i)
{
    const float2 e = lane < cnt ? list[lane] : make_float2(INFINITY, __int_as_float(0x7fffffff));
    d = e.x; i = __float_as_int(e.y);
    KNN_SORT_64(d, i, lane);
    if (cnt > 64) {
        const float2 f = lane + 64 < cnt ? list[lane + 64] : make_float2(INFINITY, __int_as_float(0x7fffffff));
        float d2 = f.x;
        int i2 = __float_as_int(f.y);
        KNN_SORT_64(d2, i2, lane);
        const float od = __uint_as_float(knn_xor<63>(__float_as_uint(d2), lane));
        const int oi = (int)knn_xor<63>((unsigned)i2, lane);
        if (od < d || (od == d && oi < i)) { d = od; i = oi; }
        knn_step<32>(d, i, lane);
        KNN_MERGE_64(d, i, lane);
    }
}

// The k best of {prior list, tile} for k <= 64: (1) a threshold that at least k candidates pass; (2) the candidates under it
// (usually k to 1.3 k) are compacted into wave-private LDS with ballots; (3) a merge sort over the wave orders them.  More than KNN_CAP
// candidates under the threshold are thinned to those below it and the k smallest ids at it; more than KNN_CAP - 64 below it, or fewer
// than k groups with a candidate, fall back to the extraction rounds.  list: KNN_CAP entries of LDS owned by this wave.
template <int NR>
__device__ __forceinline__ void knn_select(float (&dist)[NR], int tile0, float (&pd)[1], int (&pi)[1], int k, int lane, int fallback_id, float2 *list)
{
    const float tau = knn_threshold<NR>(pd[0], k, lane, [&](int from, int to) {
        float m = dist[from];
#pragma unroll
        for (int r = 0; r < NR; ++r) if (r > from && r < to) m = fminf(m, dist[r]);
        return m;
    });
    int cnt = 0;
    auto put = [&](bool in, float d, int i) {
        const unsigned long long m = __ballot(in);
        const int pos = cnt + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
        if (in && pos < KNN_CAP) list[pos] = make_float2(d, __int_as_float(i));
        cnt += __popcll(m);
    };
    if (tile0) put(pd[0] <= tau, pd[0], pi[0]);
#pragma unroll
    for (int r = 0; r < NR; ++r) put(dist[r] <= tau, dist[r], tile0 + (r / 4) * 256 + lane * 4 + (r % 4));
    if (cnt > KNN_CAP && tau < INFINITY) {
        // mostly equal distances: whoever is below tau, and of those at tau the k smallest ids (the prior list's first, which are smaller
        // than the tile's and in order; then by group of 256, lane and register)
        fg_wave_lds_sync();
        cnt = 0;
        if (tile0) put(pd[0] < tau, pd[0], pi[0]);
#pragma unroll
        for (int r = 0; r < NR; ++r) put(dist[r] < tau, dist[r], tile0 + (r / 4) * 256 + lane * 4 + (r % 4));
        if (cnt <= KNN_CAP - 64) {
            const int end = cnt + k;
            if (tile0) put(pd[0] == tau, pd[0], pi[0]);
            const unsigned long long below = (1ull << lane) - 1ull;
#pragma unroll
            for (int g = 0; g < NR / 4; ++g) {
                int pos = cnt;
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const unsigned long long m = __ballot(dist[4 * g + u] == tau);
                    pos += __popcll(m & below);
                    cnt += __popcll(m);
                }
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (dist[4 * g + u] == tau) {
                        if (pos < end) list[pos] = make_float2(tau, __int_as_float(tile0 + g * 256 + lane * 4 + u));
                        ++pos;
                    }
            }
            cnt = min(cnt, end);
        } else cnt = KNN_CAP + 1;
    }
    if (cnt > KNN_CAP || !(tau < INFINITY)) {
        knn_select_rounds<NR, 1>(dist, tile0, pd, pi, k, lane, fallback_id);
        return;
    }
    fg_wave_lds_sync();
    float cd;
    int ci;
    knn_order(list, cnt, lane, cd, ci);
    fg_wave_lds_sync();
    pd[0] = lane < k ? cd : INFINITY;
    pi[0] = lane < k ? ci : fallback_id;
}
template <int NR>
__device__ __forceinline__ void knn_select(float (&dist)[NR], int tile0, float (&pd)[2], int (&pi)[2], int k, int lane, int fallback_id, float2 *)
{
    knn_select_rounds<NR, 2>(dist, tile0, pd, pi, k, lane, fallback_id);       // 64 < k <= 128
}

template <int RG, int KR>
__global__ __launch_bounds__(KNN_WAVES * 64) void knn_kernel(int P, int D, int k, int rows_aligned, const float *__restrict__ pts, int *__restrict__ out)
{
    constexpr int NR = 4 * RG;                  // distances per lane and query
    constexpr int TILE = 256 * RG;              // candidate points per tile
    __shared__ __attribute__((aligned(16))) float cs[KNN_DC * TILE];        // [dimension of the slice][point of the tile]
    __shared__ float2 sel[KNN_WAVES * KNN_CAP];                             // selection scratch
    const int tid = (int)threadIdx.x;
    const int lane = fg_lane();
    const int cloud = (int)blockIdx.y;
    const float *cp = pts + (size_t)cloud * P * D;
    const int qbase = fg_uni(((int)blockIdx.x * KNN_WAVES + fg_wave()) * KNN_QW);
    int qrow[KNN_QW];                           // clamped query rows (wave-uniform)
#pragma unroll
    for (int a = 0; a < KNN_QW; ++a) qrow[a] = min(qbase + a, P - 1);
    float pd[KNN_QW][KR];
    int pi[KNN_QW][KR];
#pragma unroll
    for (int a = 0; a < KNN_QW; ++a)
#pragma unroll
        for (int t = 0; t < KR; ++t) { pd[a][t] = INFINITY; pi[a][t] = qrow[a]; }

    for (int tile0 = 0; tile0 < P; tile0 += TILE) {
        float acc[KNN_QW][NR];
#pragma unroll
        for (int a = 0; a < KNN_QW; ++a)
#pragma unroll
            for (int r = 0; r < NR; ++r) acc[a][r] = 0.f;
        for (int d0 = 0; d0 < D; d0 += KNN_DC) {
            const int dn = min(KNN_DC, D - d0);
            __syncthreads();                    // the previous slice has been consumed
#pragma unroll
            for (int i = 0; i < RG; ++i) {
                const int c = tid + 256 * i;
                const bool ok = tile0 + c < P;
                const float *src = cp + (size_t)(ok ? tile0 + c : 0) * D + d0;
                if (dn == KNN_DC && rows_aligned) {              // every row starts on 16 bytes: two 128-bit loads
                    const float4 lo = *reinterpret_cast<const float4 *>(src), hi = *reinterpret_cast<const float4 *>(src + 4);
                    const float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
                    for (int dd = 0; dd < KNN_DC; ++dd) cs[dd * TILE + c] = ok ? v[dd] : 0.f;
                } else {
                    for (int dd = 0; dd < dn; ++dd) cs[dd * TILE + c] = ok ? src[dd] : 0.f;
                }
            }
            __syncthreads();
            auto step = [&](int dd) {
                float qv[KNN_QW];
#pragma unroll
                for (int a = 0; a < KNN_QW; ++a) qv[a] = cp[(size_t)qrow[a] * D + d0 + dd];
#pragma unroll
                for (int g = 0; g < RG; ++g) {
                    const float4 c4 = *reinterpret_cast<const float4 *>(&cs[dd * TILE + g * 256 + lane * 4]);
                    const float cv[4] = {c4.x, c4.y, c4.z, c4.w};
#pragma unroll
                    for (int a = 0; a < KNN_QW; ++a)
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            float df = qv[a] - cv[u];
                            acc[a][4 * g + u] = fmaf(df, df, acc[a][4 * g + u]);
                        }
                }
            };
            if (dn == KNN_DC) {
#pragma unroll
                for (int dd = 0; dd < KNN_DC; ++dd) step(dd);
            } else {
                for (int dd = 0; dd < dn; ++dd) step(dd);
            }
        }
        // points past the end of the cloud never win; NaN distances sort last among the real ones
#pragma unroll
        for (int g = 0; g < RG; ++g)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const bool ok = tile0 + g * 256 + lane * 4 + u < P;
#pragma unroll
                for (int a = 0; a < KNN_QW; ++a) acc[a][4 * g + u] = ok ? fminf(acc[a][4 * g + u], FLT_MAX) : INFINITY;
            }
#pragma unroll
        for (int a = 0; a < KNN_QW; ++a) knn_select<NR>(acc[a], tile0, pd[a], pi[a], k, lane, qrow[a], sel + fg_wave() * KNN_CAP);
    }
#pragma unroll
    for (int a = 0; a < KNN_QW; ++a) {
        const int q = qbase + a;
        if (q < P) {
            int *o = out + ((size_t)cloud * P + q) * k;
#pragma unroll
            for (int t = 0; t < KR; ++t) {
                const int j = t * 64 + lane;
                if (j < k) o[j] = cloud * P + pi[a][t];
            }
        }
    }
}

// Larger clouds of many dimensions: the distances come from the matrix cores as a filter, and only what the filter leaves open
// is computed exactly.
//
// A workgroup of 8 waves takes 32 queries; wave w multiplies its eighth of the tile's candidates (16 x 16 x 4 products, rows =
// candidates, columns = queries) straight out of global memory: lane (r, q) reads 4 consecutive floats of row r, and the 4
// products of a chunk take the first, second, third and fourth of them, a permutation of the dimensions that both operands share.
// The median, dimension by dimension, of three of the workgroup's queries is taken off all points, so a common offset costs no
// precision and one far point among the three does no harm.
// |c - q|^2 = |c|^2 - 2 c.q + |q|^2 then goes through LDS, 16 queries at a time, to the wave that selects.
//
// With u = 2^-24, S = |q|^2 + max |c|^2 (of the shifted points) the product form is within u S (2 D + 11) of the true distance and the
// exact path's own sum, one subtract and one fma per dimension, within 2 u S (D + 3); E = 2 u S (4 D + 32) covers both twice.  tau, the
// threshold that at least k approximations pass, thus bounds the k-th smallest exact distance by tau + E, and every candidate
// that can be among the k best has an approximation of at most tau + 2 E (few more than pass tau).  Sorted by approximation, two
// neighbours in the list more than 2 E apart are in order; those closer are computed by the exact path's operations in the
// exact path's order, and the list is sorted once more.  (All 47 candidates of a query at k = 40 cost 24 KB of gathered rows, and
// the L2 rate was the bound.)  With more candidates than lanes, or more points than a tile, all candidates are computed.  The graph is
// bit for bit the one of the kernel above.
//
// E holds for the farthest point of the tile.  Where more than KNN_CAP candidates pass because a few points are far out, the query
// is tried again with every candidate's own bound, E(c) = 2 u (|q|^2 + |c|^2) (4 D + 32): the k-th smallest of approximation + E(c) bounds
// the k-th smallest exact distance, and whoever's approximation - E(c) is not above it stays.  What is still open then (hundreds of points
// at one place, norms that overflow or are no numbers) takes the direct kernel's way: the workgroup streams the tile through LDS
// and the waves with open queries form all their distances.
//
// Bound by the fp32 matrix rate (1.4 us per dimension of 64 clouds x 1024 points, 95 TFLOP/s) and the selection, 140 us there.
// Before and after at k = 40: 64 dimensions 634 (379 with the present selection) -> 243 us, 128 dimensions 904 (642) -> 344 us.
#define KNN_MQ 32        // queries per workgroup
#define KNN_MW 8         // waves per workgroup
typedef float knn_f4 __attribute__((ext_vector_type(4)));

// The exact distance of point c from the wave-uniform query q: dimensions in ascending order, NaN last among the real ones.
__device__ __forceinline__ float knn_exact(const float *cp, int D, int q, int c, int rows_aligned)
{
    const float *qr = cp + (size_t)q * D, *cr = cp + (size_t)c * D;
    float acc = 0.f;
    int d = 0;
    if (rows_aligned)
        for (; d + 32 <= D; d += 32) {              // 8 loads in flight
            knn_f4 v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = *reinterpret_cast<const knn_f4 *>(cr + d + 4 * u);
#pragma unroll
            for (int u = 0; u < 32; ++u) { const float df = qr[d + u] - v[u / 4][u % 4]; acc = fmaf(df, df, acc); }
        }
#pragma unroll 4
    for (; d < D; ++d) { const float df = qr[d] - cr[d]; acc = fmaf(df, df, acc); }
    return fminf(acc, FLT_MAX);
}

// The open queries of a workgroup (bits of `any`; of the wave: `open`) against one tile, by the direct kernel's operations in their order: the
// tile streams through LDS (cs, KNN_DC x TILE floats) and the waves with open queries form all their distances, 2 x 8 waves at a time.
struct knn_best { float d[4]; int i[4]; };
template <int RG>
__device__ __forceinline__ knn_best knn_exact_tile(int P, int D, int k, int rows_aligned, const float *cp, int q0, int tile0, unsigned any, unsigned open,
                                                   float *cs, float2 *list, knn_best best)
{
    constexpr int NR = 4 * RG, TILE = 256 * RG;
    const int lane = fg_lane(), wave = fg_uni(fg_wave());
#pragma unroll 1
    for (int gq = 0; gq < 2; ++gq) {
        if (!((any >> (2 * gq)) & 3)) continue;         // uniform over the workgroup
        const unsigned mine = (open >> (2 * gq)) & 3;
        const int q = q0 + gq * 16 + 2 * wave, qa = min(q, P - 1), qb = min(q + 1, P - 1);
        float ex[2][NR];
#pragma unroll
        for (int r = 0; r < NR; ++r) ex[0][r] = ex[1][r] = 0.f;
        for (int d0 = 0; d0 < D; d0 += KNN_DC) {
            const int dn = min(KNN_DC, D - d0);
            __syncthreads();                            // the previous slice has been consumed
            for (int c = (int)threadIdx.x; c < TILE; c += KNN_MW * 64) {
                const bool ok = tile0 + c < P;
                const float *src = cp + (size_t)(ok ? tile0 + c : 0) * D + d0;
                if (dn == KNN_DC && rows_aligned) {
                    const knn_f4 lo = *reinterpret_cast<const knn_f4 *>(src), hi = *reinterpret_cast<const knn_f4 *>(src + 4);
#pragma unroll
                    for (int u = 0; u < 4; ++u) { cs[u * TILE + c] = ok ? lo[u] : 0.f; cs[(4 + u) * TILE + c] = ok ? hi[u] : 0.f; }
                } else {
                    for (int dd = 0; dd < dn; ++dd) cs[dd * TILE + c] = ok ? src[dd] : 0.f;
                }
            }
            __syncthreads();
            if (mine) {
#pragma unroll 2
                for (int dd = 0; dd < dn; ++dd) {
                    const float v0 = cp[(size_t)qa * D + d0 + dd], v1 = cp[(size_t)qb * D + d0 + dd];
#pragma unroll
                    for (int g = 0; g < RG; ++g) {
                        const knn_f4 c4 = *reinterpret_cast<const knn_f4 *>(&cs[dd * TILE + g * 256 + lane * 4]);
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const float f0 = v0 - c4[u], f1 = v1 - c4[u];
                            ex[0][4 * g + u] = fmaf(f0, f0, ex[0][4 * g + u]);
                            ex[1][4 * g + u] = fmaf(f1, f1, ex[1][4 * g + u]);
                        }
                    }
                }
            }
        }
#pragma unroll 1
        for (int j = 0; j < 2; ++j) {
            if (!((mine >> j) & 1)) continue;           // uniform over the wave
            float dist[NR];
#pragma unroll
            for (int r = 0; r < NR; ++r)
                dist[r] = tile0 + (r / 4) * 256 + lane * 4 + (r % 4) < P ? fminf(j ? ex[1][r] : ex[0][r], FLT_MAX) : INFINITY;
            float hd[1] = {gq ? (j ? best.d[3] : best.d[2]) : (j ? best.d[1] : best.d[0])};
            int hi[1] = {gq ? (j ? best.i[3] : best.i[2]) : (j ? best.i[1] : best.i[0])};
            knn_select<NR>(dist, tile0, hd, hi, k, lane, j ? qb : qa, list);
#pragma unroll
            for (int a = 0; a < 4; ++a) if (a == 2 * gq + j) { best.d[a] = hd[0]; best.i[a] = hi[0]; }
        }
    }
    __syncthreads();                                    // the last slice has been read
    return best;
}
// The same as a function of its own.  Its pointers name their memory: plain ones would be accessed by flat instructions, of which the
// ordering that fg_wave_lds_sync counts on (LDS instructions of a wave execute in order) is not known.
typedef __attribute__((address_space(3))) float *knn_lds_floats;
typedef __attribute__((address_space(3))) float2 *knn_lds_pairs;
typedef const __attribute__((address_space(1))) float *knn_global_floats;
template <int RG>
__device__ __attribute__((noinline)) knn_best knn_exact_tile_call(int P, int D, int k, int rows_aligned, knn_global_floats cp, int q0, int tile0, unsigned any,
                                                                  unsigned open, knn_lds_floats cs, knn_lds_pairs list, knn_best best)
{
    return knn_exact_tile<RG>(P, D, k, rows_aligned, (const float *)cp, q0, tile0, any, open, (float *)cs, (float2 *)list, best);
}

template <int RG, bool MULTI>
__global__ __launch_bounds__(KNN_MW * 64, 4) void knn_mfma_kernel(int P, int D, int k, int rows_aligned, unsigned per_xcd, unsigned q_blocks, unsigned n_blocks,
                                                                  const float *__restrict__ pts, int *__restrict__ out)
{
    constexpr int NR = 4 * RG, TILE = 256 * RG, NT = 2 * RG, NH = NT < 4 ? NT : 4, ROW = TILE + 4;      // rows 4 banks apart: 16 lanes write 16 rows at once
    __shared__ __attribute__((aligned(16))) float buf[16 * ROW];
    __shared__ __attribute__((aligned(16))) float cn[TILE];
    __shared__ float2 lists[KNN_MW * KNN_CAP];
    __shared__ float wmax[KNN_MW];
    __shared__ unsigned open_of[KNN_MW];
    const unsigned b = per_xcd ? (blockIdx.x % FGNN_NUM_XCD) * per_xcd + blockIdx.x / FGNN_NUM_XCD : blockIdx.x;
    if (b >= n_blocks) return;                  // the whole workgroup
    const int cloud = (int)(b / q_blocks), q0 = (int)(b % q_blocks) * KNN_MQ;
    const float *cp = pts + (size_t)cloud * P * D;
    const int lane = fg_lane(), wave = fg_uni(fg_wave()), r16 = lane & 15, kq = lane >> 4;
    float2 *list = lists + wave * KNN_CAP;
    // MULTI (more points than a tile): the best of the tiles seen so far, for the wave's queries q0 + 16 (a / 2) + 2 wave + a % 2
    float pd[4] = {INFINITY, INFINITY, INFINITY, INFINITY};
    int pi[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) pi[a] = min(q0 + (a / 2) * 16 + 2 * wave + a % 2, P - 1);
    auto finish = [&](int q, int i) { if (q < P && lane < k) out[((size_t)cloud * P + q) * k + lane] = cloud * P + i; };

    // 4 floats of a row from dimension d0 + 4 kq on: one load that checks the cloud's bounds (rows past its end read as zero).  TAIL, the last
    // chunk where D is no multiple of 16: zero past the row's end, too, and floats one by one where four could straddle the cloud's.
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(cp), 0, P * D * 4, 0x00027000);
    const unsigned lane_off = (unsigned)(r16 * D + 4 * kq) * 4u;
    auto frag = [&](int row0, bool one_row, int d0, auto tail) {          // row row0 + r16, or row row0 in all lanes
        const int off = (int)((one_row ? 16u * kq : lane_off) + ((unsigned)row0 * D + d0) * 4u);
        knn_f4 v;
        if constexpr (!decltype(tail)::value) v = __builtin_bit_cast(knn_f4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, 0, 0));
        else {
            if (D % 4 == 0) v = __builtin_bit_cast(knn_f4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, 0, 0));
            else {
#pragma unroll
                for (int u = 0; u < 4; ++u) v[u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, off + 4 * u, 0, 0));
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = d0 + 4 * kq + u < D ? v[u] : 0.f;
        }
        return v;
    };
    for (int tile0 = 0; tile0 < (MULTI ? P : 1); tile0 += TILE) {
        knn_f4 acc[NT][2];
        float nrm[NT], qn[2] = {0.f, 0.f};
        const int crow = tile0 + wave * NT * 16;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            acc[t][0] = acc[t][1] = knn_f4{0.f, 0.f, 0.f, 0.f};
            nrm[t] = 0.f;
        }
        auto chunk = [&](int d0, auto tail) {
            const knn_f4 m0 = frag(q0, true, d0, tail), m1 = frag(q0 + 10, true, d0, tail), m2 = frag(q0 + 21, true, d0, tail);
            knn_f4 m;
#pragma unroll
            for (int u = 0; u < 4; ++u) m[u] = __builtin_amdgcn_fmed3f(m0[u], m1[u], m2[u]);
            const knn_f4 b0 = frag(q0, false, d0, tail) - m, b1 = frag(q0 + 16, false, d0, tail) - m;
#pragma unroll
            for (int u = 0; u < 4; ++u) { qn[0] = fmaf(b0[u], b0[u], qn[0]); qn[1] = fmaf(b1[u], b1[u], qn[1]); }
#pragma unroll
            for (int h = 0; h < NT; h += NH) {          // at most 4 tiles of operands in registers
                knn_f4 a[NH];
#pragma unroll
                for (int t = 0; t < NH; ++t) a[t] = frag(crow + (h + t) * 16, false, d0, tail);
#pragma unroll
                for (int t = 0; t < NH; ++t) {
                    a[t] -= m;
#pragma unroll
                    for (int u = 0; u < 4; ++u) nrm[h + t] = fmaf(a[t][u], a[t][u], nrm[h + t]);
                }
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int t = 0; t < NH; ++t) {
                        acc[h + t][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t][u], b0[u], acc[h + t][0], 0, 0, 0);
                        acc[h + t][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t][u], b1[u], acc[h + t][1], 0, 0, 0);
                    }
            }
        };
        int d0 = 0;
        for (; d0 + 16 <= D; d0 += 16) chunk(d0, std::false_type());
        if (d0 < D) chunk(d0, std::true_type());
        // lane (r, q) holds a quarter of the norms of row r: add the quarters up
        auto quarters = [&](float v) {
            v += __uint_as_float(knn_xor<16>(__float_as_uint(v), lane));
            return v + __uint_as_float(knn_xor<32>(__float_as_uint(v), lane));
        };
        auto sane = [](float v) { return v < 1e37f ? v : INFINITY; };             // overflow or NaN: the bound becomes infinite
        qn[0] = quarters(qn[0]);
        qn[1] = quarters(qn[1]);
        float mx = 0.f;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const float n = quarters(nrm[t]);
            if (crow + t * 16 + r16 < P) mx = fmaxf(mx, sane(n));
            if (kq == 0) cn[(wave * NT + t) * 16 + r16] = n;
        }
        mx = fg_wave_max(mx);
        if (lane == 0) wmax[wave] = mx;
        unsigned open = 0;                      // the wave's queries that the filter leaves open, bit a as in pd[a] (uniform)
        fg_wave_lds_sync();                     // a wave reads only the norms that it wrote
        auto select16 = [&](auto group) {
            constexpr int gq = decltype(group)::value;
            const float qg = qn[gq];
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int c = (wave * NT + t) * 16 + 4 * kq;                      // the product's rows 4 kq .. 4 kq + 3, column r16
                const knn_f4 n4 = *reinterpret_cast<const knn_f4 *>(&cn[c]);
                *reinterpret_cast<knn_f4 *>(&buf[r16 * ROW + c]) = (n4 - 2.f * acc[t][gq]) + qg;
            }
            __syncthreads();
            float cmax = wmax[0];
#pragma unroll
            for (int w = 1; w < KNN_MW; ++w) cmax = fmaxf(cmax, wmax[w]);
#pragma unroll 1
            for (int j = 0; j < 2; ++j) {
                const int ql = 2 * wave + j, q = min(q0 + gq * 16 + ql, P - 1);
                float hd = INFINITY;
                int hi = q;
                if constexpr (MULTI) { hd = j ? pd[2 * gq + 1] : pd[2 * gq]; hi = j ? pi[2 * gq + 1] : pi[2 * gq]; }
                float *row = &buf[ql * ROW + lane * 4];
                float dist[NR];
                auto fetch = [&]() {
#pragma unroll
                    for (int g = 0; g < RG; ++g) {
                        const knn_f4 v = *reinterpret_cast<const knn_f4 *>(row + g * 256);
#pragma unroll
                        for (int u = 0; u < 4; ++u) dist[4 * g + u] = tile0 + g * 256 + lane * 4 + u < P ? v[u] : INFINITY;
                    }
                };
                fetch();
                const float qn2 = sane(fg_readlane(qg, ql)), rel = (float)(4 * D + 32) * 0x1p-23f, tiny = (float)(D + 1) * 1e-36f;
                float E = rel * (qn2 + cmax) + tiny;
                auto least = [&](int from, int to) {
                    float m = dist[from];
#pragma unroll
                    for (int r = 0; r < NR; ++r) if (r > from && r < to) m = fminf(m, dist[r]);
                    return m;
                };
                int cnt = 0;
                auto put = [&](bool in, float d, int i) {
                    const unsigned long long m = __ballot(in);
                    const int pos = cnt + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
                    if (in && pos < KNN_CAP) list[pos] = make_float2(d, __int_as_float(i));
                    cnt += __popcll(m);
                };
                const float lim = knn_threshold<NR>(hd, k, lane, least) + 2.f * E;
                bool bounded = lim < INFINITY;              // false, too, where E is infinite or the threshold no number
                if (MULTI && tile0) put(hd <= lim, hd, hi);
#pragma unroll
                for (int r = 0; r < NR; ++r) put(dist[r] <= lim, dist[r], tile0 + (r / 4) * 256 + lane * 4 + (r % 4));
                // once more with every candidate's own bound, where half of a sample have a good deal less than the farthest
                if (bounded && cnt > KNN_CAP && __popcll(__ballot(16.f * cn[lane * 4] < cmax)) >= 32) {
                    fg_wave_lds_sync();
                    auto own = [&](int g) {                 // E(c) of the lane's four candidates of group g
                        knn_f4 e = *reinterpret_cast<const knn_f4 *>(&cn[g * 256 + lane * 4]);
#pragma unroll
                        for (int u = 0; u < 4; ++u) e[u] = rel * (qn2 + e[u]) + tiny;
                        return e;
                    };
#pragma unroll
                    for (int g = 0; g < RG; ++g) {
                        const knn_f4 e = own(g);
#pragma unroll
                        for (int u = 0; u < 4; ++u) dist[4 * g + u] = dist[4 * g + u] < INFINITY ? dist[4 * g + u] + e[u] : INFINITY;
                    }
                    const float tau = knn_threshold<NR>(hd, k, lane, least);
                    bounded = tau < INFINITY;
                    cnt = 0;
                    E = 0.f;                                // the largest bound of those that stay
                    if (MULTI && tile0) put(hd <= tau, hd, hi);
#pragma unroll
                    for (int g = 0; g < RG; ++g) {
                        const knn_f4 e = own(g);
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const bool in = dist[4 * g + u] - 2.f * e[u] <= tau && dist[4 * g + u] < INFINITY;
                            if (in) E = fmaxf(E, e[u]);
                            put(in, dist[4 * g + u] - e[u], tile0 + g * 256 + lane * 4 + u);
                        }
                    }
                    E = fg_wave_max(E);
                }
                fg_wave_lds_sync();
                if (bounded && cnt <= 64 && !MULTI) {
                    const float2 e = lane < cnt ? list[lane] : make_float2(INFINITY, __int_as_float(0x7fffffff));
                    float cd = e.x;
                    int ci = __float_as_int(e.y);
                    KNN_SORT_64(cd, ci, lane);
                    const float before = fg_bperm(cd, lane ? lane - 1 : 0), after = fg_bperm(cd, lane < 63 ? lane + 1 : 63);
                    const bool near = lane < cnt && ((lane && cd - before <= 2.f * E) || (lane + 1 < cnt && after - cd <= 2.f * E));
                    if (__ballot(near)) {
                        if (near) cd = knn_exact(cp, D, q, ci, rows_aligned);
                        KNN_SORT_64(cd, ci, lane);
                    }
                    hd = lane < k ? cd : INFINITY;
                    hi = lane < k ? ci : q;
                } else if (bounded && cnt <= KNN_CAP) {
                    for (int e = lane; e < cnt; e += 64) list[e].x = knn_exact(cp, D, q, __float_as_int(list[e].y), rows_aligned);
                    fg_wave_lds_sync();
                    float cd;
                    int ci;
                    knn_order(list, cnt, lane, cd, ci);
                    hd = lane < k ? cd : INFINITY;
                    hi = lane < k ? ci : q;
                } else {
                    open |= 1u << (2 * gq + j);
                }
                if constexpr (MULTI) {
                    if (j) { pd[2 * gq + 1] = hd; pi[2 * gq + 1] = hi; }
                    else { pd[2 * gq] = hd; pi[2 * gq] = hi; }
                } else if (!((open >> (2 * gq + j)) & 1)) finish(q0 + gq * 16 + ql, hi);
                fg_wave_lds_sync();
            }
            __syncthreads();                    // the rows have been read
        };
        select16(std::integral_constant<int, 0>());
        select16(std::integral_constant<int, 1>());

        // the queries that are still open (the rows of buf have been read)
        if (lane == 0) open_of[wave] = open;
        __syncthreads();
        unsigned any = 0;
#pragma unroll
        for (int w = 0; w < KNN_MW; ++w) any |= open_of[w];
        static_assert(KNN_DC * TILE <= 16 * ROW, "the slices go where the approximations were");
        if (any) {
            knn_best best;
#pragma unroll
            for (int a = 0; a < 4; ++a) { best.d[a] = pd[a]; best.i[a] = pi[a]; }
            if constexpr (MULTI) best = knn_exact_tile_call<RG>(P, D, k, rows_aligned, (knn_global_floats)cp, q0, tile0, any, open, (knn_lds_floats)buf, (knn_lds_pairs)list, best);
            else best = knn_exact_tile<RG>(P, D, k, rows_aligned, cp, q0, tile0, any, open, buf, list, best);
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                if constexpr (MULTI) { pd[a] = best.d[a]; pi[a] = best.i[a]; }
                else if ((open >> a) & 1) finish(q0 + (a / 2) * 16 + 2 * wave + a % 2, best.i[a]);
            }
        }
    }
    if constexpr (MULTI) {
#pragma unroll
        for (int a = 0; a < 4; ++a) finish(q0 + (a / 2) * 16 + 2 * wave + a % 2, pi[a]);
    }
}

template <int RG, bool MULTI>
static void knn_mfma_launch(int n_clouds, int P, int D, int k, const float *points, int32_t *src_ind, hipStream_t st)
{
    const unsigned q_blocks = (unsigned)((P + KNN_MQ - 1) / KNN_MQ), n_blocks = q_blocks * (unsigned)n_clouds;
    unsigned grid = n_blocks, per_xcd = 0;
    if (grid >= 8 * FGNN_NUM_XCD && fgnn_current_device_has_xcd_mapping()) {      // a cloud is read through one XCD's L2
        per_xcd = (grid + FGNN_NUM_XCD - 1) / FGNN_NUM_XCD;
        grid = per_xcd * FGNN_NUM_XCD;
    }
    hipLaunchKernelGGL((knn_mfma_kernel<RG, MULTI>), dim3(grid), dim3(KNN_MW * 64), 0, st, P, D, k, D % 4 == 0 && fgnn_aligned16(points) ? 1 : 0, per_xcd,
                       q_blocks, n_blocks, points, src_ind);
}

template <int RG, int KR>
static void knn_launch(int n_clouds, int P, int D, int k, const float *points, int32_t *src_ind, hipStream_t st)
{
    const int qwg = KNN_WAVES * KNN_QW;
    dim3 grid((unsigned)((P + qwg - 1) / qwg), (unsigned)n_clouds);
    hipLaunchKernelGGL((knn_kernel<RG, KR>), grid, dim3(KNN_WAVES * 64), 0, st, P, D, k,
                       (D % 4 == 0 && fgnn_aligned16(points)) ? 1 : 0, points, src_ind);
}

extern "C" int fgnn_knn_graph(int n_clouds, int P, int D, int k, const float *points, int32_t *src_ind, void *stream)
{
    FGNN_REQUIRE(n_clouds >= 0 && P >= 1 && D >= 1 && k >= 1, FGNN_ERR_SHAPE, "fgnn_knn_graph: bad sizes clouds=%d P=%d D=%d k=%d", n_clouds, P, D, k);
    FGNN_REQUIRE(k <= P, FGNN_ERR_SHAPE, "fgnn_knn_graph: k=%d exceeds the %d points of a cloud", k, P);
    FGNN_REQUIRE(k <= KNN_MAX_K, FGNN_ERR_LIMIT, "fgnn_knn_graph: k=%d exceeds the limit of %d neighbours", k, KNN_MAX_K);
    FGNN_REQUIRE((int64_t)n_clouds * P * k <= 2147483647LL, FGNN_ERR_LIMIT, "fgnn_knn_graph: more than 2^31 edges");
    FGNN_REQUIRE(points && src_ind, FGNN_ERR_NULL, "fgnn_knn_graph: NULL argument");
    FGNN_REQUIRE(n_clouds <= 65535, FGNN_ERR_LIMIT, "fgnn_knn_graph: more than 65535 clouds");
    if (n_clouds == 0) return 0;
    hipStream_t st = (hipStream_t)stream;
    const int rg = P <= 256 ? 1 : P <= 512 ? 2 : 4;     // tile = 256 * rg candidate points
    // A launch holds fewer than 2^32 threads in one dimension: 2^23 workgroups of the matrix form, whose grid has only one.
    // A cloud's bytes are counted in 31 bits by the loads that check its bounds.
    const int64_t blocks = (int64_t)n_clouds * ((P + KNN_MQ - 1) / KNN_MQ);
    const bool fits = blocks <= (1 << 23) - FGNN_NUM_XCD && (int64_t)P * D * 4 <= 0x7fffffff;
    // The matrix form costs less per dimension (64 clouds: 1.5 against 4.2 us at 1024 points, 0.5 against 0.85 at 512) and at 512 points more
    // per query, where the two meet at 48 dimensions (67 against 66 us; 32: 55 against 59).  With more points it wins from 16 on where
    // its 32 queries a workgroup still fill the chip twice (64 x 1024: 158 against 117 us at 16; 8 x 2048: 80 against 68); with
    // fewer workgroups the meeting point moves up (8 x 1024: 22 against 26 at 16, 40 against 34 at 48; 1 x 1024: 32 against 33 at 48).  At
    // 256 points it loses up to 128 dimensions (46 against 44 us; 34 against 29 at 64).
    if (k <= 64 && fits && rg >= 2 && D >= (rg == 4 && blocks >= 512 ? 16 : 48)) {
        if (rg == 2) knn_mfma_launch<2, false>(n_clouds, P, D, k, points, src_ind, st);
        else if (P <= 1024) knn_mfma_launch<4, false>(n_clouds, P, D, k, points, src_ind, st);
        else knn_mfma_launch<4, true>(n_clouds, P, D, k, points, src_ind, st);
    } else if (k <= 64) {
        if (rg == 1) knn_launch<1, 1>(n_clouds, P, D, k, points, src_ind, st);
        else if (rg == 2) knn_launch<2, 1>(n_clouds, P, D, k, points, src_ind, st);
        else knn_launch<4, 1>(n_clouds, P, D, k, points, src_ind, st);
    } else {
        if (rg == 1) knn_launch<1, 2>(n_clouds, P, D, k, points, src_ind, st);
        else if (rg == 2) knn_launch<2, 2>(n_clouds, P, D, k, points, src_ind, st);
        else knn_launch<4, 2>(n_clouds, P, D, k, points, src_ind, st);
    }
    return fgnn_launch_status("knn_kernel");
}
