// Dense products over very many rows (one per node, point or edge) with a small matrix on the other side, on the fp32 matrix
// instructions (v_mfma_f32_16x16x4_f32):
//   tall product    y [n, m] = x [n, k] @ b [k, m] (+ bias)            the projections of the layers and their input gradients
//   tall reduction  c [ka, kb] = x [n, ka]^T @ g [n, kb]                the weight gradients
// Both take a few extra columns out of two more arrays of h columns each (the attention scores of a GAT layer and their gradients),
// so that the scores fall out of the projection and nothing is stacked or cropped in memory.
#include <algorithm>
#include "fgnn_common.h"

typedef float tl_f4 __attribute__((ext_vector_type(4)));
typedef float tl_f2 __attribute__((ext_vector_type(2)));

#define TL_LDS_MAX (160 * 1024)
#define TL_WAVES(NT) ((NT) <= 9 ? 16 : 12)  // most waves of a workgroup (one per compute unit) that the registers of the accumulators leave room for

struct TallP {
    int64_t n;
    int k, m;                               // columns of x, columns of y
    const float *x; int64_t ldx;
    const float *b; int64_t ldb; int trans; // b[r][c] at b[r * ldb + c], trans: at b[c * ldb + r]; (k + 2 hin) x (m + 2 hout)
    const float *bias;
    float *y; int64_t ldy;
    int hin; const float *xe0, *xe1;        // input columns k .. k + 2 hin: xe0 [n, hin], xe1 [n, hin]
    int hout; float *ye0, *ye1;             // output columns m .. m + 2 hout
    int kk, kkm;                            // chunks of 16 input columns, those of x among them
    int waves;                              // of a workgroup
    int splits;                             // column ranges of y, a workgroup works on one of them
    int vecy;                               // rows of y start at 16 bytes
};

// Four consecutive floats, VEC of them a load.
template <int VEC>
__device__ __forceinline__ tl_f4 tl_load4(const float *__restrict__ q)
{
    if constexpr (VEC == 4) return *reinterpret_cast<const tl_f4 *>(q);
    else if constexpr (VEC == 2) {
        const tl_f2 a = *reinterpret_cast<const tl_f2 *>(q), b = *reinterpret_cast<const tl_f2 *>(q + 2);
        return tl_f4{a[0], a[1], b[0], b[1]};
    } else return tl_f4{q[0], q[1], q[2], q[3]};
}

// A workgroup keeps NT 16-column tiles of b in LDS for good, in operand order (one ds_read_b128 feeds four instructions), and walks
// over the rows; a wave computes 16 rows x NT tiles at a time.  The weights are the A operand, so that a lane ends up with four
// consecutive columns of one row (row lane % 16, columns 16 t + 4 (lane / 16) ..) and stores them as 128 bits; x goes
// straight from memory to registers, four consecutive floats per lane, 64 columns ahead of their use.  Column ranges of the same rows
// run side by side on one XCD, where the second finds x in the L2.
// Bound by the matrix unit (155 TFLOP/s in these instructions alone; the operand reads and the x loads beside them leave 100-110).
// us, library products and what stood around them / this kernel: 2.4 M x 100 -> 256 + 16 scores 1474 + 260 / 1285 (104 TFLOP/s), 256 -> 48 + 2
// 698 + 590 / 746 (3.4 TB/s of x), 2.4 M gradients 48 + 2 -> 256 1061 + 210 / 835; 169 k x 128 -> 256 + 8 125 + 28 / 152, 384 -> 64 178 / 107.
template <int NT, int VEC, bool HIN>
__global__ __launch_bounds__(64 * TL_WAVES(NT)) void tall_product_kernel(TallP p)
{
    extern __shared__ tl_f4 wl[];           // [chunk][NT][64]
    const int waves = p.waves;
    const int lane = fg_lane(), wave = fg_wave(), r16 = lane & 15, g = lane >> 4;
    const int KK = p.kk;
    const int64_t ntiles = (p.n + 15) / 16;
    // workgroup w runs on XCD w % 8: ranges of the same rows 8 workgroups apart
    const int split = ((int)blockIdx.x / FGNN_NUM_XCD) % p.splits;
    const int64_t block = (int64_t)((int)blockIdx.x / FGNN_NUM_XCD / p.splits) * FGNN_NUM_XCD + (int)blockIdx.x % FGNN_NUM_XCD;
    const int64_t blocks = (int64_t)gridDim.x / p.splits;
    const int col0 = split * 16 * NT;
    const bool extra_out = p.hout > 0 && split == p.splits - 1;        // the extra columns take the last tile of the last range

    // The input column that step s of a chunk takes from lane group g (-1: none).  A whole chunk: four consecutive columns a lane, one per
    // step.  A chunk of fewer than 16 columns (the last of x, the extra columns): the groups side by side, so that the steps past
    // the last column are left out.
    const int whole = p.k / 16;
    auto column_of = [&](int kc, int g, int s) {
        if (kc < whole) return 16 * kc + 4 * g + s;
        const int e = 4 * s + g;
        if (kc < p.kkm) return 16 * kc + e < p.k ? 16 * kc + e : -1;
        return e < 2 * p.hin ? p.k + e : -1;
    };
#pragma unroll 4
    for (int i = (int)threadIdx.x; i < KK * NT * 64; i += 64 * waves) {     // (loads without branches, those of four trips in flight)
        const int l = i & 63, q = i >> 6, kc = q / NT, t = q - kc * NT;
        const bool extra = extra_out && t == NT - 1;
        const int j = extra ? (l & 15) : col0 + 16 * t + (l & 15);
        const bool okc = extra ? j < 2 * p.hout : j < p.m;
        const int64_t col = okc ? (extra ? p.m + j : j) : 0;
        float v[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int64_t row = column_of(kc, l >> 4, s), r = row < 0 ? 0 : row;
            v[s] = p.b[p.trans ? col * p.ldb + r : r * p.ldb + col];
            if (!okc || row < 0) v[s] = 0.f;
        }
        wl[i] = tl_f4{v[0], v[1], v[2], v[3]};
    }
    __syncthreads();

    // whole chunks c0 .. c0 + 3 of a row (xr: the row at the lane's own columns)
    auto load = [&](tl_f4 (&v)[4], const float *xr, int c0) {
#pragma unroll
        for (int c = 0; c < 4; ++c) if (c0 + c < whole) v[c] = tl_load4<VEC>(xr + 16 * (c0 + c));
    };
    auto row_of = [&](int64_t tile) { return tile * 16 + r16 < p.n ? tile * 16 + r16 : p.n - 1; };

    const int64_t step = blocks * waves;
    int64_t tile = block * waves + wave;
    if (tile >= ntiles) return;
    int64_t node = row_of(tile);
    const float *xr = p.x + node * p.ldx + 4 * g;
    tl_f4 cur[4] = {};
    load(cur, xr, 0);
    for (; tile < ntiles; tile += step) {
        const int64_t next = row_of(tile + step);
        const float *xn = p.x + next * p.ldx + 4 * g;
        tl_f4 acc[NT], esum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = tl_f4{0.f, 0.f, 0.f, 0.f};
        tl_f4 rest[2] = {};                     // the chunks of fewer than 16 columns
        if (whole < p.kkm) {
#pragma unroll
            for (int s = 0; s < 4; ++s) if (16 * whole + 4 * s + g < p.k) rest[0][s] = xr[16 * whole + 4 * s - 3 * g];
        }
        if (HIN) {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int e = 4 * s + g;
                if (e < 2 * p.hin) rest[1][s] = (e < p.hin ? p.xe0 + e : p.xe1 + (e - p.hin))[node * p.hin];
            }
        }
#pragma unroll 1
        for (int c0 = 0; c0 < whole; c0 += 4) {
            tl_f4 nxt[4] = {cur[0], cur[1], cur[2], cur[3]};
            const bool last = c0 + 4 >= whole;
            load(nxt, last ? xn : xr, last ? 0 : c0 + 4);
            // operands in groups of four tiles, the next group's read while one is multiplied: no instruction waits for the
            // one before it, and no more than two groups are in registers
            constexpr int GP = (NT + 3) / 4;
            const tl_f4 *w = wl + (size_t)c0 * NT * 64 + lane;
            tl_f4 a[2][4];
#pragma unroll
            for (int u = 0; u < 4; ++u) if (u < NT) a[0][u] = w[u * 64];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                if (c0 + c >= whole) break;
#pragma unroll
                for (int i = 0; i < GP; ++i) {
                    const int at = (c * GP + i) & 1, nc = i + 1 < GP ? c : c + 1, nt = i + 1 < GP ? 4 * (i + 1) : 0;
                    if (nc == c || (nc < 4 && c0 + nc < whole)) {
#pragma unroll
                        for (int u = 0; u < 4; ++u) if (nt + u < NT) a[at ^ 1][u] = w[(nc * NT + nt + u) * 64];
                    }
#pragma unroll
                    for (int s = 0; s < 4; ++s)
#pragma unroll
                        for (int u = 0; u < 4; ++u)
                            if (4 * i + u < NT) acc[4 * i + u] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[at][u][s], cur[c][s], acc[4 * i + u], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            // the extra columns are sums over 64 input columns each, added up: nearer to the exact scores than one long chain
            if (extra_out) {
                esum += acc[NT - 1];
                acc[NT - 1] = tl_f4{0.f, 0.f, 0.f, 0.f};
                asm volatile("" : "+v"(esum));
            }
            // The next columns are waited for here, at the end of a group: a wait at its start would also be one for the stores of
            // the rows before (loads and stores share a counter).
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                asm volatile("" : "+v"(nxt[c]));
                cur[c] = nxt[c];
            }
        }
#pragma unroll 1
        for (int kc = whole; kc < KK; ++kc) {
            const tl_f4 xv = kc < p.kkm ? rest[0] : rest[1];
            const int cols = kc < p.kkm ? p.k - 16 * kc : 2 * p.hin;
            const float *ws = (const float *)(wl + (size_t)kc * NT * 64 + lane);
#pragma unroll 1
            for (int s = 0; 4 * s < cols; ++s) {
                const float x1 = s == 0 ? xv[0] : s == 1 ? xv[1] : s == 2 ? xv[2] : xv[3];
#pragma unroll
                for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(ws[t * 256 + s], x1, acc[t], 0, 0, 0);
            }
        }
        if (extra_out) esum += acc[NT - 1];
        if (tile * 16 + r16 < p.n) {
            // re-defined here, so that addresses, comparisons and loads of the bias stay here: hoisted out of the loop they take nine
            // registers a tile
            const float *bias = p.bias;
            int m = p.m, j4 = 4 * g;
            asm volatile("" : "+s"(bias), "+s"(m), "+v"(j4));
            float *yb = p.y + node * p.ldy + col0 + j4;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int j0 = col0 + 16 * t;
                if (j0 >= m) continue;
                tl_f4 v = acc[t];
                if (bias) {
#pragma unroll
                    for (int s = 0; s < 4; ++s) v[s] += bias[min(j0 + j4 + s, m - 1)];
                }
                if (p.vecy && j0 + 16 <= m) *reinterpret_cast<tl_f4 *>(yb + 16 * t) = v;
                else {
#pragma unroll
                    for (int s = 0; s < 4; ++s) if (j0 + j4 + s < m) yb[16 * t + s] = v[s];
                }
            }
            if (extra_out) {
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const int e = 4 * g + s;
                    if (e < p.hout) p.ye0[node * p.hout + e] = esum[s];
                    else if (e < 2 * p.hout) p.ye1[node * p.hout + e - p.hout] = esum[s];
                }
            }
        }
        node = next;
        xr = xn;
    }
}

static inline int tl_vec(const void *p, int64_t ld, int k)
{
    if (((uintptr_t)p & 15) == 0 && ld % 4 == 0 && k % 4 == 0) return 4;
    if (((uintptr_t)p & 7) == 0 && ld % 2 == 0 && k % 2 == 0) return 2;
    return 1;
}

// Numbers of 16-column tiles that kernels exist for: the next one up is taken (0: none).
static inline int tl_tiles(int t)
{
    for (int v : {1, 2, 3, 4, 5, 6, 8, 9, 12, 16, 17, 18}) if (t <= v) return v;
    return 0;
}
template <typename Fn>
static inline void tl_dispatch_tiles(int t, Fn &&f)
{
    switch (t) {
    case 1: f.template operator()<1>(); break;
    case 2: f.template operator()<2>(); break;
    case 3: f.template operator()<3>(); break;
    case 4: f.template operator()<4>(); break;
    case 5: f.template operator()<5>(); break;
    case 6: f.template operator()<6>(); break;
    case 8: f.template operator()<8>(); break;
    case 9: f.template operator()<9>(); break;
    case 12: f.template operator()<12>(); break;
    case 16: f.template operator()<16>(); break;
    case 17: f.template operator()<17>(); break;
    default: f.template operator()<18>(); break;
    }
}

struct TallPlan { int tiles, splits, waves; int64_t blocks; };   // blocks: workgroups of a column range
static bool tall_product_plan(int64_t n, int k, int m, int hin, int hout, int cus, TallPlan *pl)
{
    const int kk = (k + 15) / 16 + (hin ? 1 : 0), total = (m + 15) / 16 + (hout ? 1 : 0), fit = std::min(18, TL_LDS_MAX / (kk * 1024));
    if (fit < 1) return false;
    int splits = (total + fit - 1) / fit, tiles = tl_tiles((total + splits - 1) / splits);
    while ((size_t)tiles * kk * 1024 > TL_LDS_MAX) {                         // the next number of tiles that a kernel exists for does not fit
        ++splits;
        tiles = tl_tiles((total + splits - 1) / splits);
    }
    splits = (total + tiles - 1) / tiles;
    // One workgroup per compute unit, of as many waves (four SIMDs' worth at a time) as give the shortest way through the row tiles:
    // 4096 tiles are one and a third rounds for 12 waves on 256 units and two for 8, so 24 tile times against 16 (65 k x 64 -> 256: 54 -> 33 us).
    // A column range gets whole eighths of the units (its workgroups are dealt out by XCD), rounded down: of three ranges 80 on 256 units,
    // for with 88 eight workgroups of the 264 begin when the others have ended (us, 88 / 80, 180 -> 384 + 12 scores: 70 k rows 216 / 109,
    // 169 k 401 / 251, 500 k 1216 / 685; library product and score kernel 133, 265, 800).
    const int64_t rows = (n + 15) / 16, units = std::max(cus / splits / FGNN_NUM_XCD * FGNN_NUM_XCD, FGNN_NUM_XCD);
    int64_t best = INT64_MAX;
    for (int w = TL_WAVES(tiles); w >= 4; w -= 4) {
        const int64_t cost = (rows + units * w - 1) / (units * w) * w;
        if (cost < best) { best = cost; pl->waves = w; }
    }
    const int64_t need = (rows + pl->waves - 1) / pl->waves;
    pl->blocks = std::min(units, (need + FGNN_NUM_XCD - 1) / FGNN_NUM_XCD * FGNN_NUM_XCD);
    pl->tiles = tiles; pl->splits = splits;
    return true;
}

extern "C" int64_t fgnn_tall_product_workgroups(int64_t n, int k, int m, int hin, int hout, int compute_units)
{
    TallPlan pl;
    if (n < 1 || k < 1 || m < 1 || hin < 0 || hout < 0 || k > (1 << 20) || compute_units < 1 || !tall_product_plan(n, k, m, hin, hout, compute_units, &pl)) return 0;
    return pl.blocks * pl.splits;
}

extern "C" int fgnn_tall_product(int64_t n, int k, int m, const float *x, int64_t ldx, const float *b, int64_t ldb, int b_transposed, const float *bias,
                                 float *y, int64_t ldy, int hin, const float *xe0, const float *xe1, int hout, float *ye0, float *ye1, void *stream)
{
    FGNN_REQUIRE(n >= 0 && k >= 1 && m >= 1 && ldx >= k && ldy >= m && hin >= 0 && hout >= 0, FGNN_ERR_SHAPE,
                 "fgnn_tall_product: bad sizes n=%lld k=%d m=%d ldx=%lld ldy=%lld", (long long)n, k, m, (long long)ldx, (long long)ldy);
    FGNN_REQUIRE(hin <= 8 && hout <= 8 && k <= (1 << 20), FGNN_ERR_LIMIT, "fgnn_tall_product: more than 8 extra columns a side");
    FGNN_REQUIRE(ldb >= (b_transposed ? k + 2 * hin : m + 2 * hout), FGNN_ERR_SHAPE, "fgnn_tall_product: ldb=%lld", (long long)ldb);
    FGNN_REQUIRE(n == 0 || (x && b && y && (!hin || (xe0 && xe1)) && (!hout || (ye0 && ye1))), FGNN_ERR_NULL, "fgnn_tall_product: NULL argument");
    FGNN_REQUIRE(((uintptr_t)y & 15) == 0 || ldy % 4 != 0, FGNN_ERR_ALIGN, "fgnn_tall_product: y not 16-byte aligned");
    if (n == 0) return 0;
    const int vec = tl_vec(x, ldx, k);
    TallP p{};
    p.n = n; p.k = k; p.m = m; p.x = x; p.ldx = ldx; p.b = b; p.ldb = ldb; p.trans = b_transposed; p.bias = bias; p.y = y; p.ldy = ldy;
    p.hin = hin; p.xe0 = xe0; p.xe1 = xe1; p.hout = hout; p.ye0 = ye0; p.ye1 = ye1;
    p.kkm = (k + 15) / 16; p.kk = p.kkm + (hin ? 1 : 0);
    p.vecy = ldy % 4 == 0;
    const int cus = fgnn_current_device_compute_units();
    TallPlan pl;
    FGNN_REQUIRE(tall_product_plan(n, k, m, hin, hout, cus > 0 ? cus : 256, &pl), FGNN_ERR_LIMIT, "fgnn_tall_product: %d input columns unsupported", k);
    p.splits = pl.splits; p.waves = pl.waves;
    const size_t lds = (size_t)pl.tiles * p.kk * 1024;
    const unsigned grid = (unsigned)(pl.blocks * pl.splits);
    hipStream_t st = (hipStream_t)stream;
    FGNN_REQUIRE(hin == 0 || vec == 4, FGNN_ERR_ALIGN, "fgnn_tall_product: extra input columns need x in rows of 16-byte multiples");
    tl_dispatch_tiles(pl.tiles, [&]<int NT>() {
        const dim3 g(grid), w(64 * p.waves);
        if (hin) hipLaunchKernelGGL((tall_product_kernel<NT, 4, true>), g, w, lds, st, p);
        else if (vec == 4) hipLaunchKernelGGL((tall_product_kernel<NT, 4, false>), g, w, lds, st, p);
        else if (vec == 2) hipLaunchKernelGGL((tall_product_kernel<NT, 2, false>), g, w, lds, st, p);
        else hipLaunchKernelGGL((tall_product_kernel<NT, 1, false>), g, w, lds, st, p);
    });
    return fgnn_launch_status("tall_product_kernel");
}

// ------------------------------------------------------------------------------------------------ tall reduction
struct TallR {
    int64_t n, rows_per_block;
    int ka, kb, h;                          // columns of x, of g, and of each of the two extra arrays on g's side
    const float *x; int64_t ldx; const float *g; int64_t ldg; const float *ge0, *ge1;
    int vx, vg;                             // floats a load takes
    int ta, tb, tiles;                      // 16-column tiles of x; of g with its extra columns; of the result
    int rpp;                                // rows a load pass takes
    float *part;                            // [gridDim][ka][kb + 2 h]
};
#define TR_WAVES 16
#define TR_TPB (64 * TR_WAVES)
#define TR_SLOTS 5
#define TR_MAX_U 9                          // tiles a wave holds, a number that tl_tiles knows
#define TR_TILE(R) ((R) * 16 + 16)          // floats an operand tile of R rows takes in LDS; the 16 spread the tiles' rows over the banks

// A workgroup sums the whole result over a range of rows; its waves hold U 16 x 16 tiles of it each, dealt out one after the other, so
// that 7 x 17 tiles keep 16 waves busy as well as 8 x 16 do.  R rows of both operands
// are staged in LDS tile by tile (read from memory once, 128 bits per thread where the rows allow it, one stage ahead): the operand of
// four rows is then 64 consecutive floats, at an offset known when compiling, and an instruction costs two LDS reads and
// no vector arithmetic, which would take its time from the matrix unit (a vector instruction beside every matrix instruction: 11 % less).
// us, batched library product over chunks of rows, its sum and the stacked operand / this kernel and its sum: 2.4 M x 256, 48 + 2
// 638 + 460 / 918 (bound by reading x: 3.2 TB/s), 169 k x 256, 40 + 2 82 + 30 / 76, 33 k x 64, 128 32 / 23.  A second stage of LDS, so that rows are stored
// while the others are multiplied, spilled registers and was slower (2.4 M x 100, 272: 1.59 -> 1.65 to 2.2 ms).
template <int U, int R>
__global__ __launch_bounds__(TR_TPB) void tall_reduce_kernel(TallR p)
{
    extern __shared__ float sm[];
    const int tid = (int)threadIdx.x, lane = fg_lane(), wave = fg_wave(), r16 = lane & 15, q = lane >> 4;
    float *gs = sm + p.ta * TR_TILE(R);
    const int64_t r0 = (int64_t)blockIdx.x * p.rows_per_block, r1 = r0 + p.rows_per_block < p.n ? r0 + p.rows_per_block : p.n;

    // a thread's column of four floats, fixed over the loop: c < ca of x, else of g
    const int ca = (p.ka + 3) / 4, cols = ca + (p.kb + 3) / 4;
    const int c = tid % cols, lr = tid / cols;
    const bool isx = c < ca;
    const int rend = lr < p.rpp ? R : 0;
    const int col = isx ? 4 * c : 4 * (c - ca), width = isx ? p.ka : p.kb, vec = isx ? p.vx : p.vg;
    const float *src = (isx ? p.x : p.g) + col;
    const int64_t ld = isx ? p.ldx : p.ldg;
    float *dst = (isx ? sm : gs) + (col >> 4) * TR_TILE(R) + (col & 15) + lr * 16;
    const int er = tid >> 4, ee = tid & 15;                                                 // extra columns: one float per thread

    for (int i = tid; i < (p.ta + p.tb) * TR_TILE(R); i += TR_TPB) sm[i] = 0.f;             // the padding of the last tiles stays zero

    tl_f4 pre[TR_SLOTS];
    float pree = 0.f;
    auto fetch = [&](int64_t row0) {
#pragma unroll
        for (int i = 0; i < TR_SLOTS; ++i) {
            const int rr = lr + i * p.rpp;
            const int64_t row = row0 + rr;
            tl_f4 v = {0.f, 0.f, 0.f, 0.f};
            if (rr < rend && row < r1) {
                const float *s = src + row * ld;
                if (vec == 4) v = *reinterpret_cast<const tl_f4 *>(s);
                else if (vec == 2) {
                    const tl_f2 u = *reinterpret_cast<const tl_f2 *>(s);
                    v[0] = u[0]; v[1] = u[1];
                    if (col + 2 < width) { const tl_f2 w = *reinterpret_cast<const tl_f2 *>(s + 2); v[2] = w[0]; v[3] = w[1]; }
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) if (col + e < width) v[e] = s[e];
                }
            }
            pre[i] = v;
        }
        if (p.h) {
            const int64_t row = row0 + er;
            pree = 0.f;
            if (er < R && row < r1) {
                if (ee < p.h) pree = p.ge0[row * p.h + ee];
                else if (ee < 2 * p.h) pree = p.ge1[row * p.h + ee - p.h];
            }
        }
    };
    // operands of the wave's tiles (wave-uniform); past the last tile the last one again, results unused
    const int t0 = wave * U;
    int at[U], bt[U];
    const float *ap[U], *bp[U];
    tl_f4 acc[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int t = fg_uni(min(t0 + u, p.tiles - 1));
        at[u] = t / p.tb;
        bt[u] = t % p.tb;
        ap[u] = sm + at[u] * TR_TILE(R) + lane;
        bp[u] = gs + bt[u] * TR_TILE(R) + lane;
        acc[u] = tl_f4{0.f, 0.f, 0.f, 0.f};
    }
    const bool busy = t0 < p.tiles;

    fetch(r0);
#pragma unroll 1
    for (int64_t row0 = r0; row0 < r1; row0 += R) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < TR_SLOTS; ++i) {
            if (lr + i * p.rpp < rend) *reinterpret_cast<tl_f4 *>(dst + i * p.rpp * 16) = pre[i];
        }
        if (p.h && er < R) gs[(p.tb - 1) * TR_TILE(R) + er * 16 + ee] = pree;
        __syncthreads();
        if (row0 + R < r1) fetch(row0 + R);
        if (!busy) continue;
#pragma unroll
        for (int s = 0; s < R / 4; s += 2) {
            // a few tiles at a time, so that the operands of no more are in registers
            constexpr int G = U > 5 ? 3 : 6;
#pragma unroll
            for (int u0 = 0; u0 < U; u0 += G) {
                float xv[2][G], gv[2][G];
#pragma unroll
                for (int u = 0; u < G; ++u) {
                    if (u0 + u >= U) continue;
                    const float *a = ap[u0 + u], *b = bp[u0 + u];
                    xv[0][u] = a[64 * s]; xv[1][u] = a[64 * s + 64];
                    gv[0][u] = b[64 * s]; gv[1][u] = b[64 * s + 64];
                }
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int u = 0; u < G; ++u)
                        if (u0 + u < U) acc[u0 + u] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[h][u], gv[h][u], acc[u0 + u], 0, 0, 0);
                if (U > 4) __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    const int kb2 = p.kb + 2 * p.h;
    float *out = p.part + (size_t)blockIdx.x * p.ka * kb2;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        if (t0 + u >= p.tiles) continue;
        const bool extra = p.h > 0 && bt[u] == p.tb - 1;
        const int j = extra ? r16 : 16 * bt[u] + r16;
        if (extra ? j >= 2 * p.h : j >= p.kb) continue;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int i = 16 * at[u] + 4 * q + s;
            if (i < p.ka) out[(size_t)i * kb2 + (extra ? p.kb + j : j)] = acc[u][s];
        }
    }
}

// c[i] = sum over the partial results, in a fixed order and in 64 bits (the pass is bound by its launch and its reads)
__global__ __launch_bounds__(256) void tall_reduce_sum_kernel(int64_t total, int parts, const float *__restrict__ part, float *__restrict__ c)
{
    __shared__ double sh[8][33];
    const int o = (int)threadIdx.x & 31, w = (int)threadIdx.x >> 5;
    const int64_t i = (int64_t)blockIdx.x * 32 + o;
    double s = 0.;
    if (i < total) {
#pragma unroll 4
        for (int j = w; j < parts; j += 8) s += (double)part[(size_t)j * total + i];
    }
    sh[w][o] = s;
    __syncthreads();
    if (w || i >= total) return;
#pragma unroll
    for (int j = 1; j < 8; ++j) s += sh[j][o];
    c[i] = (float)s;
}

struct TallRPlan { int ta, tb, tiles, u, R, rpp, blocks; int64_t rows; size_t lds; };
static bool tall_reduce_plan(int64_t n, int ka, int kb, int h, TallRPlan *pl)
{
    const int cols = (ka + 3) / 4 + (kb + 3) / 4;
    if (cols > TR_TPB / 4) return false;
    pl->ta = (ka + 15) / 16;
    pl->tb = (kb + 15) / 16 + (h ? 1 : 0);
    pl->tiles = pl->ta * pl->tb;
    if (pl->tiles > TR_MAX_U * TR_WAVES) return false;
    pl->u = tl_tiles((pl->tiles + TR_WAVES - 1) / TR_WAVES);
    pl->rpp = std::min(TR_TPB / cols, 32);                                   // at least 4: TR_SLOTS passes take R rows
    pl->R = pl->rpp * TR_SLOTS >= 32 ? 32 : 16;
    pl->lds = (size_t)(pl->ta + pl->tb) * TR_TILE(pl->R) * sizeof(float);
    if (pl->lds > TL_LDS_MAX) return false;
    const int64_t want = std::min<int64_t>(256, (n + 255) / 256);
    const int64_t rows = (n + want - 1) / std::max<int64_t>(want, 1);
    pl->rows = (rows + pl->R - 1) / pl->R * pl->R;
    pl->blocks = (int)((n + pl->rows - 1) / pl->rows);
    return true;
}

extern "C" size_t fgnn_tall_reduce_workspace_bytes(int64_t n, int ka, int kb, int h)
{
    TallRPlan pl;
    if (n <= 0 || ka < 1 || kb < 1 || h < 0 || h > 8 || !tall_reduce_plan(n, ka, kb, h, &pl)) return 0;
    return (size_t)pl.blocks * (size_t)ka * (kb + 2 * h) * sizeof(float);
}

extern "C" int fgnn_tall_reduce(int64_t n, int ka, int kb, const float *x, int64_t ldx, const float *g, int64_t ldg, int h, const float *ge0, const float *ge1,
                                float *c, void *workspace, size_t workspace_bytes, void *stream)
{
    FGNN_REQUIRE(n >= 1 && ka >= 1 && kb >= 1 && ldx >= ka && ldg >= kb && h >= 0, FGNN_ERR_SHAPE, "fgnn_tall_reduce: bad sizes n=%lld ka=%d kb=%d ldx=%lld ldg=%lld",
                 (long long)n, ka, kb, (long long)ldx, (long long)ldg);
    TallRPlan pl;
    FGNN_REQUIRE(h <= 8 && tall_reduce_plan(n, ka, kb, h, &pl), FGNN_ERR_LIMIT, "fgnn_tall_reduce: ka=%d kb=%d h=%d unsupported", ka, kb, h);
    FGNN_REQUIRE(x && g && c && (!h || (ge0 && ge1)), FGNN_ERR_NULL, "fgnn_tall_reduce: NULL argument");
    const size_t need = fgnn_tall_reduce_workspace_bytes(n, ka, kb, h);
    FGNN_REQUIRE(workspace && workspace_bytes >= need, FGNN_ERR_WORKSPACE, "fgnn_tall_reduce: workspace %zu < %zu bytes", workspace_bytes, need);
    TallR p{};
    p.n = n; p.rows_per_block = pl.rows; p.ka = ka; p.kb = kb; p.h = h; p.x = x; p.ldx = ldx; p.g = g; p.ldg = ldg; p.ge0 = ge0; p.ge1 = ge1;
    p.vx = tl_vec(x, ldx, ka); p.vg = tl_vec(g, ldg, kb);
    p.ta = pl.ta; p.tb = pl.tb; p.tiles = pl.tiles; p.rpp = pl.rpp; p.part = (float *)workspace;
    hipStream_t st = (hipStream_t)stream;
    tl_dispatch_tiles(pl.u, [&]<int U>() {
        if constexpr (U <= TR_MAX_U) {
            if (pl.R == 32) hipLaunchKernelGGL((tall_reduce_kernel<U, 32>), dim3((unsigned)pl.blocks), dim3(TR_TPB), pl.lds, st, p);
            else hipLaunchKernelGGL((tall_reduce_kernel<U, 16>), dim3((unsigned)pl.blocks), dim3(TR_TPB), pl.lds, st, p);
        }
    });
    int rc = fgnn_launch_status("tall_reduce_kernel");
    if (rc) return rc;
    const int64_t total = (int64_t)ka * (kb + 2 * h);
    hipLaunchKernelGGL(tall_reduce_sum_kernel, dim3((unsigned)((total + 31) / 32)), dim3(256), 0, st, total, pl.blocks, p.part, c);
    return fgnn_launch_status("tall_reduce_sum_kernel");
}

// ------------------------------------------------------------------------------------------------ column sums
// A workgroup sums a range of rows; thread t takes every (1024 / columns)-th row of its column (VEC of them), four loads in flight, in 64
// bits, and the rows are added up in LDS.  Bound by reading x: us, torch's reduction (in chunks where the columns are no multiple of four) / this and
// its sum: 169 k x 64 20 / 13 (3.3 TB/s), 233 k x 41 39 / 12, 2.4 M x 64 142 / 110 (5.7 TB/s), x 41 135 / 94.
#define CS_TPB 1024
template <int VEC>
__global__ __launch_bounds__(CS_TPB) void column_sum_kernel(int64_t n, int64_t rows_per_block, int c, const float *__restrict__ x, int64_t ldx, float *__restrict__ part)
{
    __shared__ double sh[VEC][CS_TPB];
    const int tid = (int)threadIdx.x, cols = c / VEC, rpp = CS_TPB / cols, col = tid % cols, lr = tid / cols;
    const int64_t r0 = (int64_t)blockIdx.x * rows_per_block, r1 = r0 + rows_per_block < n ? r0 + rows_per_block : n;
    double s[VEC] = {};
    if (lr < rpp) {
        const float *q = x + col * VEC;
        for (int64_t r = r0 + lr; r < r1; r += 4 * rpp) {
            float v[4][VEC];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int64_t row = r + (int64_t)u * rpp;
                const float *src = q + (row < r1 ? row : r) * ldx;          // past the end: the first row again, not added
                if constexpr (VEC == 4) { const tl_f4 w = *reinterpret_cast<const tl_f4 *>(src); v[u][0] = w[0]; v[u][1] = w[1]; v[u][2] = w[2]; v[u][3] = w[3]; }
                else v[u][0] = *src;
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (r + (int64_t)u * rpp < r1) {
#pragma unroll
                    for (int e = 0; e < VEC; ++e) s[e] += (double)v[u][e];
                }
        }
    }
#pragma unroll
    for (int e = 0; e < VEC; ++e) sh[e][tid] = s[e];
    __syncthreads();
    // column i of the result: element i % VEC of the threads of quad i / VEC
    for (int i = tid; i < c; i += CS_TPB) {
        double t = 0.;
        for (int j = 0; j < rpp; ++j) t += sh[i % VEC][i / VEC + j * cols];
        part[(size_t)blockIdx.x * c + i] = (float)t;
    }
}

static int64_t column_sum_rows(int64_t n) { return (n + 255) / 256; }       // of a workgroup
static int column_sum_blocks(int64_t n) { return (int)((n + column_sum_rows(n) - 1) / column_sum_rows(n)); }

extern "C" size_t fgnn_column_sum_workspace_bytes(int64_t n, int c)
{
    return n >= 1 && c >= 1 && c <= CS_TPB ? (size_t)column_sum_blocks(n) * c * sizeof(float) : 0;
}

extern "C" int fgnn_column_sum(int64_t n, int c, const float *x, int64_t ldx, float *out, void *workspace, size_t workspace_bytes, void *stream)
{
    FGNN_REQUIRE(n >= 1 && c >= 1 && ldx >= c, FGNN_ERR_SHAPE, "fgnn_column_sum: bad sizes n=%lld c=%d ldx=%lld", (long long)n, c, (long long)ldx);
    FGNN_REQUIRE(c <= CS_TPB, FGNN_ERR_LIMIT, "fgnn_column_sum: %d columns unsupported", c);
    FGNN_REQUIRE(x && out, FGNN_ERR_NULL, "fgnn_column_sum: NULL argument");
    const size_t need = fgnn_column_sum_workspace_bytes(n, c);
    FGNN_REQUIRE(workspace && workspace_bytes >= need, FGNN_ERR_WORKSPACE, "fgnn_column_sum: workspace %zu < %zu bytes", workspace_bytes, need);
    hipStream_t st = (hipStream_t)stream;
    const dim3 grid((unsigned)column_sum_blocks(n));
    float *part = (float *)workspace;
    if (tl_vec(x, ldx, c) == 4) hipLaunchKernelGGL(column_sum_kernel<4>, grid, dim3(CS_TPB), 0, st, n, column_sum_rows(n), c, x, ldx, part);
    else hipLaunchKernelGGL(column_sum_kernel<1>, grid, dim3(CS_TPB), 0, st, n, column_sum_rows(n), c, x, ldx, part);
    int rc = fgnn_launch_status("column_sum_kernel");
    if (rc) return rc;
    hipLaunchKernelGGL(tall_reduce_sum_kernel, dim3((unsigned)((c + 31) / 32)), dim3(256), 0, st, (int64_t)c, column_sum_blocks(n), part, out);
    return fgnn_launch_status("tall_reduce_sum_kernel");
}
