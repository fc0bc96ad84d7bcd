// GPU CSR -> CSC transpose (stable), replacing the reference's cuSPARSE call
// (src/csr2csc/csr2csc.cu:10-23), and the COO -> CSR builder.
//
// Both are stable LSD radix sorts of small records with digits of up to 11 bits (22-bit ids: two passes of
// 11).  Each pass is histogram -> scan -> stable scatter: a workgroup owns a contiguous tile, each of its 16
// waves a contiguous sixteenth of it, and a wave walks its part 64 records at a time, ranking equal digits
// inside the wave with ballots, so equal keys keep their order.  Integer work only, bit-exact and deterministic.
//
// What bounds a pass is the scatter: 2048 digits leave about 4 consecutive records of a tile per digit, far
// less than a 128-byte line.  Two things keep the lines whole: the workgroups of one XCD take a contiguous
// eighth of the tiles (the next tile of a digit's run is written through the same L2 shortly after, so 2048
// open lines, 256 KB, complete in it), and a record's words travel together (8-byte stores).  64.3 M records of
// 8 bytes: the scatter of a pass takes 0.34-0.39 ms (1.03 GB, 2.6-3.0 TB/s) and the pass 0.51; with 8-bit digits,
// separate 4-byte key and payload streams and the tiles dealt round-robin it was 0.44 and 0.59 ms, and 44 bits took
// six passes instead of four.  COO -> CSR -> CSC of that graph: 10.3 -> 4.0 ms.
//
// A workgroup is 1024 threads with 8 records each: at 512 threads with 16 the records, ranks and counters held 128-168
// registers, one workgroup lived on a compute unit and the ranking chain had nothing to hide behind (0.67 ms).
#include "fgnn_common.h"

#define RS_TPB 1024
#define RS_WAVES 16
#define RS_MAX_BITS 11
#define RS_MAX_DIGITS (1 << RS_MAX_BITS)
#define RS_DPT (RS_MAX_DIGITS / RS_TPB)      // digits per thread in the per-tile scans
// Records per thread: tiles of 8192 keep the per-tile digit runs long; small inputs take tiles of 2048 so that they
// spread over the chip (1 M records: 512 workgroups instead of 128).  From 2 M records on the runs count for more: CSR -> CSC of 2.1 M
// entries in 2000 columns 57 us with the large tiles and 81 with the small ones, of 4 M in 131 k columns 86 and 126.
#define RS_SMALL_N (2 << 20)
static inline int rs_items(int64_t n) { return n < RS_SMALL_N ? 2 : 8; }
static inline int rs_num_tiles(int64_t n) { const int64_t t = (int64_t)RS_TPB * rs_items(n); return (int)((n + t - 1) / t); }
static __host__ __device__ inline int rs_hist_ld(int ntiles) { return (ntiles + 7) & ~7; }     // ints per digit of the count array
static inline unsigned rs_grid(int ntiles) { return (unsigned)(((ntiles + FGNN_NUM_XCD - 1) / FGNN_NUM_XCD) * FGNN_NUM_XCD); }
// Workgroup b -> tile: the workgroups of an XCD (b % 8) own a contiguous range of tiles.  May be >= ntiles: no work.
__device__ __forceinline__ int rs_tile_of(int b, int ntiles) { return (b % FGNN_NUM_XCD) * ((ntiles + FGNN_NUM_XCD - 1) / FGNN_NUM_XCD) + b / FGNN_NUM_XCD; }

// hist[d * rs_hist_ld(ntiles) + t] = records of tile t whose digit is d.  keys: every `stride`-th int.
template <int ITEMS>
__global__ __launch_bounds__(RS_TPB) void rs_hist_kernel(const int *__restrict__ keys, int stride, int64_t n, int shift, int mask, int ntiles, int *__restrict__ hist)
{
    __shared__ int cnt[2][RS_MAX_DIGITS];        // two sets of counters: half the collisions
    const int tile = rs_tile_of((int)blockIdx.x, ntiles);
    if (tile >= ntiles) return;
    for (int d = (int)threadIdx.x; d <= mask; d += RS_TPB) { cnt[0][d] = 0; cnt[1][d] = 0; }
    __syncthreads();
    const int64_t base = (int64_t)tile * (RS_TPB * ITEMS) + threadIdx.x;
    const int set = (int)threadIdx.x & 1;
    int key[ITEMS];
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
        const int64_t i = base + it * RS_TPB;
        key[it] = i < n ? keys[i * stride] : 0;
    }
#pragma unroll
    for (int it = 0; it < ITEMS; ++it)
        if (base + it * RS_TPB < n) atomicAdd(&cnt[set][(key[it] >> shift) & mask], 1);
    __syncthreads();
    for (int d = (int)threadIdx.x; d <= mask; d += RS_TPB) hist[(size_t)d * rs_hist_ld(ntiles) + tile] = cnt[0][d] + cnt[1][d];
}

// Inclusive sum over the lanes of a wave.
__device__ __forceinline__ int rs_wave_incl(int v, int lane)
{
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        int t = __shfl_up(v, off);
        if (lane >= off) v += t;
    }
    return v;
}

// One workgroup per digit: exclusive scan of that digit's per-tile counts in place.  The row is walked
// in chunks of 256 * 8 counts: every thread scans 8 consecutive counts serially, the 256 thread totals
// are scanned with wave shuffles and one exchange through LDS, and the chunk's total carries over.
#define RS_SCAN_TPB 256
__global__ __launch_bounds__(RS_SCAN_TPB) void rs_scan_kernel(int *__restrict__ hist, int ntiles, int *__restrict__ digit_total)
{
    constexpr int PER = 8;
    __shared__ int wave_tot[RS_SCAN_TPB / 64];
    int *row = hist + (size_t)blockIdx.x * rs_hist_ld(ntiles);
    const int lane = fg_lane(), wave = fg_wave();
    int carry = 0;
    for (int base = 0; base < ntiles; base += RS_SCAN_TPB * PER) {
        const int i0 = base + (int)threadIdx.x * PER;           // rows are padded to PER counts, whatever the padding holds
        int v[PER] = {0, 0, 0, 0, 0, 0, 0, 0}, tot = 0;
        if (i0 < ntiles) {
            *reinterpret_cast<int4 *>(v) = *reinterpret_cast<const int4 *>(row + i0);
            *reinterpret_cast<int4 *>(v + 4) = *reinterpret_cast<const int4 *>(row + i0 + 4);
        }
#pragma unroll
        for (int j = 0; j < PER; ++j) { if (i0 + j >= ntiles) v[j] = 0; tot += v[j]; }
        const int incl = rs_wave_incl(tot, lane);
        __syncthreads();                        // the previous chunk's wave totals have been read
        if (lane == 63) wave_tot[wave] = incl;
        __syncthreads();
        int run = carry + incl - tot;
        for (int w = 0; w < wave; ++w) run += wave_tot[w];
#pragma unroll
        for (int j = 0; j < PER; ++j) { const int t = v[j]; v[j] = run; run += t; }
        if (i0 < ntiles) {
            *reinterpret_cast<int4 *>(row + i0) = *reinterpret_cast<const int4 *>(v);
            *reinterpret_cast<int4 *>(row + i0 + 4) = *reinterpret_cast<const int4 *>(v + 4);
        }
        carry += wave_tot[0] + wave_tot[1] + wave_tot[2] + wave_tot[3];
    }
    if (threadIdx.x == 0) digit_total[blockIdx.x] = carry;
}

// Where the records of a pass come from.
//   RS_PAIR:     rec[i] = {x, y}; the key is x, or y with KEY_Y
//   RS_ARRAYS:   {a[i], b[i]} (b == NULL: {a[i], i}), likewise
//   RS_TRIPLE:   key[i] and rec[i]
//   RS_TRIPLE_SWAP: as RS_TRIPLE with key and rec.x exchanged (from here on the other id is sorted)
//   RS_EDGES:    key b[i], rec {a[i], i} (b: source, a: destination of input edge i)
//   RS_CSR:      key a[i], rec {i, row of position i}
enum rs_in { RS_PAIR, RS_ARRAYS, RS_TRIPLE, RS_TRIPLE_SWAP, RS_EDGES, RS_CSR };
// Where they go: RS_TO_PAIR rec_out[q]; RS_TO_ARRAYS {a_out[q], b_out[q]}; RS_TO_TRIPLE key_out[q], rec_out[q];
// RS_TO_ARRAYS3 key_out[q], {a_out[q], b_out[q]}.
enum rs_out { RS_TO_PAIR, RS_TO_ARRAYS, RS_TO_TRIPLE, RS_TO_ARRAYS3 };
struct rs_args {
    const int *a, *b;               // separate input arrays
    const int *key; const int2 *rec;
    int *a_out, *b_out, *key_out; int2 *rec_out;
    const int *row_ptr, *hint;      // RS_CSR
};

// hint[k] = row of position min(k << CSC_HINT_SHIFT, n - 1): a coarse inverse of row_ptr.  128 = the records a wave of a small
// tile owns, so that every wave of RS_CSR finds the row of its first record there.
#define CSC_HINT_SHIFT 7
// Up to this many rows per position of a tile their starts are scanned for the positions' rows; beyond, the positions are searched
// for.  Scanning costs one workgroup 1 us per thousand rows (100 M empty rows between two halves of 1 M entries: 16 ms, searched 0.08);
// where all tiles span such runs the two meet at about 10 rows per entry (8 M entries: scanned 365 us at 10 and 458 at 14, searched
// 423 at 18).
#define CSC_SCAN_ROWS 8
static int csc_num_hints(int64_t E) { return E > 0 ? (int)((E - 1) >> CSC_HINT_SHIFT) + 2 : 0; }
__global__ __launch_bounds__(256) void csc_row_hint_kernel(int64_t n, int n_rows, int n_hint, const int *__restrict__ row_ptr, int *__restrict__ hint)
{
    const int k = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (k >= n_hint) return;
    int64_t p = (int64_t)k << CSC_HINT_SHIFT;
    if (p > n - 1) p = n - 1;
    int lo = 0, hi = n_rows;                    // the last r with row_ptr[r] <= p
    while (hi - lo > 1) {
        const int mid = (int)(((unsigned)lo + (unsigned)hi) >> 1);
        if (row_ptr[mid] <= (int)p) lo = mid; else hi = mid;
    }
    hint[k] = lo;
}

// Stable scatter of one pass.  The tile is first sorted by digit inside LDS (local position = the digit's base inside
// the tile + rank among the tile's earlier records of that digit), then written out in local order: the records of a
// digit leave as one run.  The digit counters and the staged records share the same LDS (72 KB in all: two workgroups
// of 16 waves per compute unit), and the words of a three-word record are staged one part after the other.
template <int ITEMS, rs_in IN, rs_out OUT, bool KEY_Y>
__global__ __launch_bounds__(RS_TPB, 8) void rs_scatter_kernel(rs_args A, int64_t n, int shift, int mask, int ntiles, const int *__restrict__ hist,
                                                            const int *__restrict__ digit_total)
{
    constexpr int TILE = RS_TPB * ITEMS, SUB = 64 * ITEMS;
    constexpr bool TRIPLE = OUT == RS_TO_TRIPLE || OUT == RS_TO_ARRAYS3;
    constexpr size_t LDS = TILE * sizeof(int2) > RS_WAVES * RS_MAX_DIGITS * sizeof(uint16_t) ? TILE * sizeof(int2) : RS_WAVES * RS_MAX_DIGITS * sizeof(uint16_t);
    __shared__ __attribute__((aligned(16))) char buf[LDS];
    __shared__ int gofs[RS_MAX_DIGITS];          // per digit: global position of the tile's run minus its local base
    __shared__ int wave_tot[2][RS_WAVES];
    uint16_t (*wcnt)[RS_MAX_DIGITS] = reinterpret_cast<uint16_t (*)[RS_MAX_DIGITS]>(buf);   // per wave and digit: running count, then the local base
    const int wave = fg_wave(), lane = fg_lane(), tid = (int)threadIdx.x;
    const int tile = rs_tile_of((int)blockIdx.x, ntiles);
    if (tile >= ntiles) return;
    const int64_t tile0 = (int64_t)tile * TILE;
    const int64_t first = tile0 + wave * SUB;    // the wave's first record
    const int count = (int)((n - tile0) < (int64_t)TILE ? (n - tile0) : (int64_t)TILE);
    const int mine = count - wave * SUB - lane;  // record it * 64 of the lane exists when it lies below this
    int key[ITEMS];
    int2 rec[ITEMS];
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
        const int64_t i = tile0 + min(wave * SUB + it * 64 + lane, count - 1);     // past the end: a copy of the last record, never stored
        int2 r = make_int2(0, 0);
        int k = 0;
        if constexpr (IN == RS_PAIR) r = A.rec[i];
        else if constexpr (IN == RS_ARRAYS) { r.x = A.a[i]; r.y = A.b ? A.b[i] : (int)i; }
        else if constexpr (IN == RS_EDGES) { k = A.b[i]; r = make_int2(A.a[i], (int)i); }
        else if constexpr (IN == RS_CSR) { k = A.a[i]; r.x = (int)i; }
        else { k = A.key[i]; r = A.rec[i]; }
        if constexpr (IN == RS_TRIPLE_SWAP) { const int t = k; k = r.x; r.x = t; }
        if constexpr (IN == RS_PAIR || IN == RS_ARRAYS) k = KEY_Y ? r.y : r.x;
        key[it] = k;
        rec[it] = r;
    }
    if constexpr (IN == RS_CSR) {
        const int64_t last = tile0 + TILE < n ? tile0 + TILE : n - 1;      // rows up to the one that holds the next tile's first position
        const int r0 = A.hint[tile0 >> CSC_HINT_SHIFT], r1 = A.hint[(last + (1 << CSC_HINT_SHIFT) - 1) >> CSC_HINT_SHIFT];
        // row of every position of the tile, in LDS
        int *mark = reinterpret_cast<int *>(buf);
        if (r1 - r0 > CSC_SCAN_ROWS * TILE) {
            // the tile spans a long run of empty rows: each position is searched for between the two hints around it
#pragma unroll 1
            for (int i = tid; i < count; i += RS_TPB) {
                const int p = (int)(tile0 + i);
                int lo = A.hint[p >> CSC_HINT_SHIFT], hi = A.hint[(p >> CSC_HINT_SHIFT) + 1] + 1;
                while (hi - lo > 1) {
                    const int mid = (int)(((unsigned)lo + (unsigned)hi) >> 1);
                    if (A.row_ptr[mid] <= p) lo = mid; else hi = mid;
                }
                mark[i] = lo;
            }
            __syncthreads();
        } else {
            // the starts of the non-empty rows leave their number (several rows that start at one position are empty but for the
            // last, the largest number), then a running maximum over the positions
            for (int i = tid; i < TILE; i += RS_TPB) mark[i] = 0;
            __syncthreads();
            for (int64_t r = (int64_t)r0 + 1 + tid; r <= r1; r += RS_TPB) {
                const int64_t o = (int64_t)A.row_ptr[r] - tile0;
                if (o >= 0 && o < TILE) atomicMax(&mark[o], (int)r);
            }
            __syncthreads();
            // a lane takes ITEMS consecutive positions, the lanes of a wave the wave's SUB positions
            int m[ITEMS];
            int *own = mark + wave * SUB + lane * ITEMS;
            int top = 0;
#pragma unroll
            for (int it = 0; it < ITEMS; ++it) { m[it] = own[it]; top = max(top, m[it]); m[it] = top; }
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const int t = __shfl_up(top, off);
                if (lane >= off) top = max(top, t);
            }
            int run = __shfl_up(top, 1);
            run = max(lane == 0 ? 0 : run, first < n ? A.hint[first >> CSC_HINT_SHIFT] : 0);
#pragma unroll
            for (int it = 0; it < ITEMS; ++it) own[it] = max(m[it], run);
            fg_wave_lds_sync();
        }
#pragma unroll
        for (int it = 0; it < ITEMS; ++it) rec[it].y = mark[wave * SUB + it * 64 + lane];
        __syncthreads();
    }
    for (int d = tid; d < RS_WAVES * RS_MAX_DIGITS / 2; d += RS_TPB) reinterpret_cast<int *>(buf)[d] = 0;
    __syncthreads();
    const unsigned long long lt = (1ull << lane) - 1ull;
    int rank[ITEMS];
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
        const bool ok = it * 64 < mine;
        // opaque here: the ballots of later records stay behind this one (hoisted to the top they cost 60 registers and half the waves)
        const int d = (int)fg_pin((uint32_t)((key[it] >> shift) & mask));
        // lanes with the same digit: per bit a sign-extended bit field (0 or -1), its ballot, and peers &= ~(bit ^ ballot) on each half
        const unsigned long long valid = __builtin_amdgcn_ballot_w64(ok);
        uint32_t plo = (uint32_t)valid, phi = (uint32_t)(valid >> 32);
#pragma unroll
        for (int bit = 0; bit < RS_MAX_BITS; ++bit) {
            const uint32_t x = (uint32_t)__builtin_amdgcn_sbfe(d, bit, 1);
            const unsigned long long bal = __builtin_amdgcn_ballot_w64(x != 0);
            plo &= ~(x ^ (uint32_t)bal);
            phi &= ~(x ^ (uint32_t)(bal >> 32));
        }
        const unsigned long long peers = ((unsigned long long)phi << 32) | plo;
        const int base = wcnt[wave][d];
        rank[it] = base + __popcll(peers & lt);
        fg_wave_lds_sync();
        // the highest lane of every peer group advances the wave's counter of that digit
        if (ok && (peers >> lane) == 1ull) wcnt[wave][d] = (uint16_t)(base + __popcll(peers));
        fg_wave_lds_sync();
    }
    __syncthreads();
    {
        // thread t owns digits RS_DPT*t ..: exclusive scans of the tile's digit counts and of the digits' totals
        int c[RS_DPT], g[RS_DPT], ctot = 0, gtot = 0;
#pragma unroll
        for (int j = 0; j < RS_DPT; ++j) {
            const int d = RS_DPT * tid + j;
            c[j] = 0;
#pragma unroll 4
            for (int w = 0; w < RS_WAVES; ++w) c[j] += wcnt[w][d];
            g[j] = d <= mask ? digit_total[d] : 0;
            ctot += c[j];
            gtot += g[j];
        }
        const int ci = rs_wave_incl(ctot, lane), gi = rs_wave_incl(gtot, lane);
        if (lane == 63) { wave_tot[0][wave] = ci; wave_tot[1][wave] = gi; }
        __syncthreads();
        int lbase = ci - ctot, gbase = gi - gtot;
        for (int w = 0; w < wave; ++w) { lbase += wave_tot[0][w]; gbase += wave_tot[1][w]; }
#pragma unroll
        for (int j = 0; j < RS_DPT; ++j) {
            const int d = RS_DPT * tid + j;
            if (d <= mask) gofs[d] = gbase + hist[(size_t)d * rs_hist_ld(ntiles) + tile] - lbase;
            int run = lbase;
#pragma unroll 4
            for (int w = 0; w < RS_WAVES; ++w) { const int t = wcnt[w][d]; wcnt[w][d] = (uint16_t)run; run += t; }
            lbase += c[j];
            gbase += g[j];
        }
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) rank[it] += wcnt[wave][(key[it] >> shift) & mask];
    __syncthreads();                             // the counters have been read: the same LDS now stages the records
    int2 *stage = reinterpret_cast<int2 *>(buf);
    if constexpr (!TRIPLE) {
#pragma unroll
        for (int it = 0; it < ITEMS; ++it)
            if (it * 64 < mine) stage[rank[it]] = rec[it];
        __syncthreads();
#pragma unroll 4
        for (int i = tid; i < count; i += RS_TPB) {
            const int2 r = stage[i];
            const int q = gofs[((KEY_Y ? r.y : r.x) >> shift) & mask] + i;
            if constexpr (OUT == RS_TO_PAIR) A.rec_out[q] = r;
            else { A.a_out[q] = r.x; A.b_out[q] = r.y; }
        }
    } else {
        int *kstage = reinterpret_cast<int *>(buf);
#pragma unroll
        for (int it = 0; it < ITEMS; ++it)
            if (it * 64 < mine) kstage[rank[it]] = key[it];
        __syncthreads();
        int dst[ITEMS];
#pragma unroll
        for (int it = 0; it < ITEMS; ++it) {
            const int i = it * RS_TPB + tid;
            dst[it] = 0;
            if (i < count) {
                const int k = kstage[i];
                dst[it] = gofs[(k >> shift) & mask] + i;
                A.key_out[dst[it]] = k;
            }
        }
        __syncthreads();
#pragma unroll
        for (int it = 0; it < ITEMS; ++it)
            if (it * 64 < mine) stage[rank[it]] = rec[it];
        __syncthreads();
#pragma unroll
        for (int it = 0; it < ITEMS; ++it) {
            const int i = it * RS_TPB + tid;
            if (i < count) {
                const int2 r = stage[i];
                if constexpr (OUT == RS_TO_TRIPLE) A.rec_out[dst[it]] = r;
                else { A.a_out[dst[it]] = r.x; A.b_out[dst[it]] = r.y; }
            }
        }
    }
}

// col_ptr from the sorted columns.
__global__ __launch_bounds__(256) void csc_colptr_kernel(int64_t n, int n_cols, const int *__restrict__ sorted_keys, int *__restrict__ col_ptr)
{
    const int64_t q0 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (q0 >= n) return;
    int v[4], prev = q0 > 0 ? sorted_keys[q0 - 1] : -1;
    if (q0 + 4 <= n) *reinterpret_cast<int4 *>(v) = *reinterpret_cast<const int4 *>(sorted_keys + q0);
    else
        for (int j = 0; j < 4; ++j) v[j] = q0 + j < n ? sorted_keys[q0 + j] : 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int64_t q = q0 + j;
        if (q >= n) break;
        for (int c = prev + 1; c <= v[j]; ++c) col_ptr[c] = (int)q;
        if (q == n - 1)
            for (int c = v[j] + 1; c <= n_cols; ++c) col_ptr[c] = (int)n;
        prev = v[j];
    }
}

__global__ __launch_bounds__(256) void fill_i32_kernel(int *p, size_t n, int v)
{
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Key bits to sort for ids below n_cols.
static int rs_key_bits(int n_cols)
{
    int bits = 1;
    while (bits < 31 && (1LL << bits) < (long long)n_cols) ++bits;
    return bits;
}

// Passes of equal digit width for a key of `key_bits` bits (18 bits: 9 + 9 rather than 11 + 7: fewer digits mean longer runs).
struct rs_plan { int passes, bits; };
static rs_plan rs_plan_of(int key_bits)
{
    rs_plan p;
    p.passes = (key_bits + RS_MAX_BITS - 1) / RS_MAX_BITS;
    p.bits = (key_bits + p.passes - 1) / p.passes;
    return p;
}
static size_t rs_hist_bytes(int64_t n, int bits)
{
    return fgnn_align256(((size_t)rs_hist_ld(rs_num_tiles(n)) << bits) * sizeof(int)) + fgnn_align256(RS_MAX_DIGITS * sizeof(int));
}

// One pass: `keys` / `stride` name the same digits for the histogram that the scatter finds in its records.
template <rs_in IN, rs_out OUT, bool KEY_Y>
static int rs_pass(const rs_args &A, const int *keys, int stride, int64_t n, int shift, int bits, int *hist, hipStream_t st)
{
    const int ntiles = rs_num_tiles(n), mask = (1 << bits) - 1;
    int *digit_total = (int *)((char *)hist + fgnn_align256(((size_t)rs_hist_ld(ntiles) << bits) * sizeof(int)));
    const bool small = rs_items(n) == 2;
    if (small) hipLaunchKernelGGL(rs_hist_kernel<2>, dim3(rs_grid(ntiles)), dim3(RS_TPB), 0, st, keys, stride, n, shift, mask, ntiles, hist);
    else hipLaunchKernelGGL(rs_hist_kernel<8>, dim3(rs_grid(ntiles)), dim3(RS_TPB), 0, st, keys, stride, n, shift, mask, ntiles, hist);
    int rc = fgnn_launch_status("rs_hist_kernel");
    if (rc) return rc;
    hipLaunchKernelGGL(rs_scan_kernel, dim3(1 << bits), dim3(RS_SCAN_TPB), 0, st, hist, ntiles, digit_total);
    rc = fgnn_launch_status("rs_scan_kernel");
    if (rc) return rc;
    if (small) hipLaunchKernelGGL((rs_scatter_kernel<2, IN, OUT, KEY_Y>), dim3(rs_grid(ntiles)), dim3(RS_TPB), 0, st, A, n, shift, mask, ntiles, hist, digit_total);
    else hipLaunchKernelGGL((rs_scatter_kernel<8, IN, OUT, KEY_Y>), dim3(rs_grid(ntiles)), dim3(RS_TPB), 0, st, A, n, shift, mask, ntiles, hist, digit_total);
    return fgnn_launch_status("rs_scatter_kernel");
}

// Scratch of rs_sort_pairs: up to two record buffers, the sorted keys, the digit counts.
static size_t rs_sort_workspace(int64_t n, int key_bits)
{
    const rs_plan p = rs_plan_of(key_bits);
    const size_t nb = fgnn_align256((size_t)n * sizeof(int2));
    return (size_t)(p.passes > 2 ? 2 : p.passes - 1) * nb + fgnn_align256((size_t)n * sizeof(int)) + rs_hist_bytes(n, p.bits);
}

// Stable LSD radix sort of n pairs by the low `key_bits` key bits.  keys_in is not modified; pay_in == NULL sorts the element
// indices.  The sorted payload lands in pay_out; *sorted_keys points at the sorted keys (inside the workspace).
static int rs_sort_pairs(const int *keys_in, const int *pay_in, int64_t n, int key_bits, int *pay_out, const int **sorted_keys, void *workspace,
                         hipStream_t st)
{
    const rs_plan p = rs_plan_of(key_bits);
    char *w = (char *)workspace;
    int2 *rec[2] = {nullptr, nullptr};
    for (int i = 0; i < 2 && i < p.passes - 1; ++i) { rec[i] = (int2 *)w; w += fgnn_align256((size_t)n * sizeof(int2)); }
    int *keys = (int *)w; w += fgnn_align256((size_t)n * sizeof(int));
    int *hist = (int *)w;
    *sorted_keys = keys;
    for (int i = 0; i < p.passes; ++i) {
        const bool last = i == p.passes - 1;
        rs_args A = {};
        A.a = keys_in; A.b = pay_in; A.a_out = keys; A.b_out = pay_out;
        if (i > 0) A.rec = rec[(i - 1) & 1];
        if (!last) A.rec_out = rec[i & 1];
        int rc;
        if (i == 0) rc = last ? rs_pass<RS_ARRAYS, RS_TO_ARRAYS, false>(A, keys_in, 1, n, 0, p.bits, hist, st)
                              : rs_pass<RS_ARRAYS, RS_TO_PAIR, false>(A, keys_in, 1, n, 0, p.bits, hist, st);
        else rc = last ? rs_pass<RS_PAIR, RS_TO_ARRAYS, false>(A, (const int *)A.rec, 2, n, p.bits * i, p.bits, hist, st)
                       : rs_pass<RS_PAIR, RS_TO_PAIR, false>(A, (const int *)A.rec, 2, n, p.bits * i, p.bits, hist, st);
        if (rc) return rc;
    }
    return 0;
}

// Up to two buffers of (key, two words), the sorted columns, the digit counts, the row hints: 16 bytes per entry up to 22 bits of column
// ids (4 M columns) and 28 above, where the passes through an index payload held 12.
extern "C" size_t fgnn_csr2csc_workspace_bytes(int n_rows, int n_cols, int64_t E)
{
    (void)n_rows;
    const rs_plan p = rs_plan_of(rs_key_bits(n_cols));
    const size_t kb = fgnn_align256((size_t)E * sizeof(int)), rb = fgnn_align256((size_t)E * sizeof(int2));
    return (size_t)(p.passes > 2 ? 2 : p.passes - 1) * (kb + rb) + kb + rs_hist_bytes(E, p.bits) + fgnn_align256((size_t)csc_num_hints(E) * sizeof(int));
}

// The records are (column, position, row): the row of a position is known where the positions are still in order, in the
// first pass, and carrying it through the other passes costs 8 bytes per entry and pass; finding it at the end, position by
// position at random places of row_ptr, took 1.3 ms for 64.3 M entries, as much as two passes.
extern "C" int fgnn_csr2csc(int n_rows, int n_cols, int64_t E, const int32_t *row_ptr, const int32_t *col_ind, int32_t *col_ptr,
                            int32_t *row_ind, int32_t *permute, void *workspace, size_t workspace_bytes, void *stream)
{
    FGNN_REQUIRE(n_rows >= 0 && n_cols >= 0 && E >= 0, FGNN_ERR_SHAPE, "fgnn_csr2csc: bad sizes");
    FGNN_REQUIRE(E <= 2147483647LL - RS_TPB * 8, FGNN_ERR_LIMIT, "fgnn_csr2csc: E=%lld exceeds int32 positions", (long long)E);
    FGNN_REQUIRE(row_ptr && col_ptr && (E == 0 || (col_ind && row_ind && permute)), FGNN_ERR_NULL, "fgnn_csr2csc: NULL argument");
    hipStream_t st = (hipStream_t)stream;
    if (E == 0) {
        hipLaunchKernelGGL(fill_i32_kernel, dim3((unsigned)((n_cols + 1 + 255) / 256)), dim3(256), 0, st, col_ptr, (size_t)n_cols + 1, 0);
        return fgnn_launch_status("fill_i32_kernel");
    }
    FGNN_REQUIRE(n_cols >= 1 && n_rows >= 1, FGNN_ERR_SHAPE, "fgnn_csr2csc: edges without rows or columns");
    size_t need = fgnn_csr2csc_workspace_bytes(n_rows, n_cols, E);
    FGNN_REQUIRE(workspace && workspace_bytes >= need, FGNN_ERR_WORKSPACE, "fgnn_csr2csc: workspace %zu < %zu bytes", workspace_bytes, need);
    const rs_plan p = rs_plan_of(rs_key_bits(n_cols));
    const size_t kb = fgnn_align256((size_t)E * sizeof(int)), rb = fgnn_align256((size_t)E * sizeof(int2));
    char *w = (char *)workspace;
    int *key[2] = {nullptr, nullptr};
    int2 *rec[2] = {nullptr, nullptr};
    for (int i = 0; i < 2 && i < p.passes - 1; ++i) { key[i] = (int *)w; w += kb; rec[i] = (int2 *)w; w += rb; }
    int *sorted = (int *)w; w += kb;
    int *hist = (int *)w; w += rs_hist_bytes(E, p.bits);
    int *hint = (int *)w;
    const int n_hint = csc_num_hints(E);
    hipLaunchKernelGGL(csc_row_hint_kernel, dim3((unsigned)((n_hint + 255) / 256)), dim3(256), 0, st, E, n_rows, n_hint, row_ptr, hint);
    int rc = fgnn_launch_status("csc_row_hint_kernel");
    for (int i = 0; i < p.passes && !rc; ++i) {
        const bool last = i == p.passes - 1;
        rs_args A = {};
        A.a = col_ind; A.row_ptr = row_ptr; A.hint = hint;
        if (i > 0) { A.key = key[(i - 1) & 1]; A.rec = rec[(i - 1) & 1]; }
        A.key_out = last ? sorted : key[i & 1];
        A.rec_out = last ? nullptr : rec[i & 1];
        A.a_out = permute; A.b_out = row_ind;
        if (i == 0) rc = last ? rs_pass<RS_CSR, RS_TO_ARRAYS3, false>(A, col_ind, 1, E, 0, p.bits, hist, st)
                              : rs_pass<RS_CSR, RS_TO_TRIPLE, false>(A, col_ind, 1, E, 0, p.bits, hist, st);
        else rc = last ? rs_pass<RS_TRIPLE, RS_TO_ARRAYS3, false>(A, A.key, 1, E, p.bits * i, p.bits, hist, st)
                       : rs_pass<RS_TRIPLE, RS_TO_TRIPLE, false>(A, A.key, 1, E, p.bits * i, p.bits, hist, st);
    }
    if (rc) return rc;
    hipLaunchKernelGGL(csc_colptr_kernel, dim3((unsigned)((E + 1023) / 1024)), dim3(256), 0, st, E, n_cols, sorted, col_ptr);
    return fgnn_launch_status("csc_colptr_kernel");
}

// ------------------------------------------------------------------------------- COO -> CSR
// Edge list (dst[e], src[e]) -> CSR by destination with sources ascending inside a row, optionally
// merging duplicate edges: what the reference does on the host with scipy's csr_matrix
// (script/train/train_gatconv_our.py:87-91).  One LSD sort over the source's digits and then the
// destination's; both ids travel in the record, so nothing is gathered between the two (through an index
// payload the two gathers took 2.5 ms for 64.3 M edges).  Where the caller wants the position of every
// input edge, its index travels too.  The sorted records are then counted (duplicates) and written.

#define SC_ITEMS 16
#define SC_TILE (256 * SC_ITEMS)
// Inclusive scan in three steps: per-tile totals, scan of the totals (one workgroup), per-tile scan + offset.
__global__ __launch_bounds__(256) void scan_tile_sums_kernel(int64_t n, const int *__restrict__ in, int *__restrict__ sums)
{
    __shared__ int sh[256];
    int64_t base = (int64_t)blockIdx.x * SC_TILE + (int64_t)threadIdx.x * SC_ITEMS;
    int acc = 0;
#pragma unroll
    for (int k = 0; k < SC_ITEMS; ++k) acc += (base + k < n) ? in[base + k] : 0;
    sh[threadIdx.x] = acc;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) sums[blockIdx.x] = sh[0];
}
// 1024 threads x 8 sums per chunk (64.3 M records: 15.7 k sums in two chunks).
#define SC_SUMS_TPB 1024
__global__ __launch_bounds__(SC_SUMS_TPB) void scan_sums_kernel(int nt, int *__restrict__ sums, int *__restrict__ total)
{
    constexpr int PER = 8;
    __shared__ int wave_tot[SC_SUMS_TPB / 64];
    const int lane = fg_lane(), wave = fg_wave();
    int carry = 0;
    for (int base = 0; base < nt; base += SC_SUMS_TPB * PER) {
        const int i0 = base + (int)threadIdx.x * PER;
        int v[PER], tot = 0;
#pragma unroll
        for (int j = 0; j < PER; ++j) { v[j] = i0 + j < nt ? sums[i0 + j] : 0; tot += v[j]; }
        const int incl = rs_wave_incl(tot, lane);
        __syncthreads();                        // the previous chunk's wave totals have been read
        if (lane == 63) wave_tot[wave] = incl;
        __syncthreads();
        int run = carry + incl - tot;
        for (int w = 0; w < SC_SUMS_TPB / 64; ++w) {
            const int t = wave_tot[w];
            if (w < wave) run += t;
            carry += t;
        }
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            if (i0 + j < nt) sums[i0 + j] = run;          // exclusive offset of tile i0 + j
            run += v[j];
        }
    }
    if (threadIdx.x == 0) *total = carry;
}
__global__ __launch_bounds__(256) void scan_apply_kernel(int64_t n, const int *__restrict__ in, const int *__restrict__ sums, int *__restrict__ out)
{
    __shared__ int sh[256];
    int64_t base = (int64_t)blockIdx.x * SC_TILE + (int64_t)threadIdx.x * SC_ITEMS;
    int v[SC_ITEMS];
    int acc = 0;
#pragma unroll
    for (int k = 0; k < SC_ITEMS; ++k) { v[k] = (base + k < n) ? in[base + k] : 0; acc += v[k]; }
    sh[threadIdx.x] = acc;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
        int t = (int)threadIdx.x >= off ? sh[threadIdx.x - off] : 0;
        __syncthreads();
        sh[threadIdx.x] += t;
        __syncthreads();
    }
    int run = sums[blockIdx.x] + sh[threadIdx.x] - acc;
#pragma unroll
    for (int k = 0; k < SC_ITEMS; ++k) {
        run += v[k];
        if (base + k < n) out[base + k] = run;
    }
}

// Library-internal entry points to the sort and the scan (the schedule builder uses them too).
size_t fgnn_rs_sort_workspace(int64_t n, int key_bits) { return rs_sort_workspace(n, key_bits); }
int fgnn_rs_key_bits(int n_keys) { return rs_key_bits(n_keys); }
int fgnn_rs_sort_pairs(const int *keys_in, const int *pay_in, int64_t n, int key_bits, int *pay_out, const int **sorted_keys, void *workspace,
                       hipStream_t st)
{
    return rs_sort_pairs(keys_in, pay_in, n, key_bits, pay_out, sorted_keys, workspace, st);
}
size_t fgnn_scan_workspace(int64_t n) { return fgnn_align256(((size_t)((n + SC_TILE - 1) / SC_TILE) + 1) * sizeof(int)); }
// out[i] = in[0] + ... + in[i]; *total_dev = the sum of all.  tile_sums: fgnn_scan_workspace(n) bytes.
int fgnn_inclusive_scan_i32(const int *in, int64_t n, int *out, int *tile_sums, int *total_dev, hipStream_t st)
{
    const int nt = (int)((n + SC_TILE - 1) / SC_TILE);
    hipLaunchKernelGGL(scan_tile_sums_kernel, dim3(nt), dim3(256), 0, st, n, in, tile_sums);
    int rc = fgnn_launch_status("scan_tile_sums_kernel");
    if (rc) return rc;
    hipLaunchKernelGGL(scan_sums_kernel, dim3(1), dim3(SC_SUMS_TPB), 0, st, nt, tile_sums, total_dev);
    rc = fgnn_launch_status("scan_sums_kernel");
    if (rc) return rc;
    hipLaunchKernelGGL(scan_apply_kernel, dim3(nt), dim3(256), 0, st, n, in, tile_sums, out);
    return fgnn_launch_status("scan_apply_kernel");
}

// Tile sums of "record q starts a new (dst, src) group" over the sorted records {dst, src} (TRIPLE: key dst, rec {src, edge}).
template <bool TRIPLE>
__device__ __forceinline__ int2 coo_at(const int *__restrict__ key, const int2 *__restrict__ rec, int64_t q)
{
    if constexpr (TRIPLE) return make_int2(key[q], rec[q].x);
    else return rec[q];
}
template <bool TRIPLE>
__global__ __launch_bounds__(256) void coo_count_kernel(int64_t n, const int *__restrict__ key, const int2 *__restrict__ rec, int *__restrict__ sums)
{
    __shared__ int sh[4];
    const int64_t base = (int64_t)blockIdx.x * SC_TILE;
    int acc = 0;
#pragma unroll
    for (int k = 0; k < SC_ITEMS; ++k) {
        const int64_t q = base + k * 256 + (int)threadIdx.x;
        if (q < n) {
            const int2 r = coo_at<TRIPLE>(key, rec, q);
            const int2 b = q > 0 ? coo_at<TRIPLE>(key, rec, q - 1) : make_int2(-1, -1);
            acc += r.x != b.x || r.y != b.y;
        }
    }
    acc = rs_wave_incl(acc, fg_lane());
    if (fg_lane() == 63) sh[fg_wave()] = acc;
    __syncthreads();
    if (threadIdx.x == 0) sums[blockIdx.x] = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// row_ptr[from .. to] = v for every lane of a wave (all of them call it; to < from: nothing).  Runs of COO_LONG_RUN rows and more are
// written by the whole wave: one lane's stores to 10 M empty rows took half a second.  any_long (uniform): there may be such runs.
#define COO_LONG_RUN 16
__device__ __forceinline__ void coo_fill_rows(int *__restrict__ row_ptr, int from, int to, int v, bool any_long)
{
    const bool big = any_long && (int64_t)to - from >= COO_LONG_RUN;
    if (!big)
        for (int i = from; i <= to; ++i) row_ptr[i] = v;
    if (!any_long) return;
    for (unsigned long long m = __ballot(big); m; m &= m - 1) {
        const int l = __builtin_ctzll(m), a = __builtin_amdgcn_readlane(from, l), b = __builtin_amdgcn_readlane(to, l), x = __builtin_amdgcn_readlane(v, l);
        for (int64_t i = (int64_t)a + fg_lane(); i <= b; i += 64) row_ptr[i] = x;
    }
}

// The CSR from the sorted records: the first record of every group writes its source at the group's position and, where its
// destination is a new one, the row pointers up to it; every input edge learns the position of its group.  sums: exclusive
// tile offsets (NULL: no merging, record q is entry q).
template <bool TRIPLE>
__global__ __launch_bounds__(256) void coo_write_kernel(int64_t n, int n_rows, const int *__restrict__ key, const int2 *__restrict__ rec,
                                                        const int *__restrict__ sums, int *__restrict__ col_ind, int *__restrict__ row_ptr,
                                                        int64_t *__restrict__ n_out, int *__restrict__ edge_pos)
{
    __shared__ int wave_cnt[SC_ITEMS][4];
    const int lane = fg_lane(), wave = fg_wave();
    const int64_t base = (int64_t)blockIdx.x * SC_TILE;
    const unsigned long long le = lane == 63 ? ~0ull : (1ull << (lane + 1)) - 1ull;
    int2 r[SC_ITEMS];
    int before[SC_ITEMS], prev_dst[SC_ITEMS];       // groups started in the wave's 64 records up to and with this one
    unsigned fl = 0;
    int jump = 0;                                   // rows from record to record (never negative), or-ed: below COO_LONG_RUN where all are
#pragma unroll
    for (int k = 0; k < SC_ITEMS; ++k) {
        const int64_t q = base + k * 256 + (int)threadIdx.x;
        r[k] = make_int2(-1, -1);
        int2 b = make_int2(-1, -1);
        if (q < n) {
            r[k] = coo_at<TRIPLE>(key, rec, q);
            if (q > 0) b = coo_at<TRIPLE>(key, rec, q - 1);
        }
        const bool f = q < n && (!sums || r[k].x != b.x || r[k].y != b.y);
        prev_dst[k] = b.x;
        jump |= r[k].x - b.x;
        fl |= (unsigned)f << k;
        const unsigned long long m = __ballot(f);
        before[k] = __popcll(m & le);
        if (lane == 0) wave_cnt[k][wave] = __popcll(m);
    }
    __syncthreads();
    const bool any_long = __ballot(jump >= COO_LONG_RUN) != 0;
    int run = sums ? sums[blockIdx.x] : (int)base;
#pragma unroll
    for (int k = 0; k < SC_ITEMS; ++k) {
        const int64_t q = base + k * 256 + (int)threadIdx.x;
        int ofs = run;
        for (int w = 0; w < wave; ++w) ofs += wave_cnt[k][w];
        const int pos = ofs + before[k] - 1;
        run += (wave_cnt[k][0] + wave_cnt[k][1]) + (wave_cnt[k][2] + wave_cnt[k][3]);
        const bool head = (fl >> k) & 1, end = q == n - 1;
        if (q < n) {
            if (head) col_ind[pos] = r[k].y;
            if (end) *n_out = pos + 1;
            if constexpr (TRIPLE) edge_pos[rec[q].y] = pos;
        }
        coo_fill_rows(row_ptr, prev_dst[k] + 1, head ? r[k].x : prev_dst[k], pos, any_long);
        if (base + SC_TILE >= n) coo_fill_rows(row_ptr, r[k].x + 1, end ? n_rows : r[k].x, pos + 1, true);      // uniform: the last tile
    }
}

// With positions: two buffers of (key, two words); without: two of pairs.  The caller's edge_pos is not known here: room for both, 24 bytes
// per edge (through index payloads, 36).
extern "C" size_t fgnn_coo2csr_workspace_bytes(int n_rows, int n_cols, int64_t E)
{
    const rs_plan ps = rs_plan_of(rs_key_bits(n_cols)), pd = rs_plan_of(rs_key_bits(n_rows));
    const size_t nt = (size_t)((E + SC_TILE - 1) / SC_TILE);
    const size_t kb = fgnn_align256((size_t)E * sizeof(int)), rb = fgnn_align256((size_t)E * sizeof(int2));
    return 2 * (kb + rb) + rs_hist_bytes(E, ps.bits > pd.bits ? ps.bits : pd.bits) + fgnn_align256((nt + 1) * sizeof(int)) + 256;
}

extern "C" int fgnn_coo2csr(int n_rows, int n_cols, int64_t E, const int32_t *dst, const int32_t *src, int dedupe, int32_t *row_ptr,
                            int32_t *col_ind, int64_t *n_out, int32_t *edge_pos, void *workspace, size_t workspace_bytes, void *stream)
{
    FGNN_REQUIRE(n_rows >= 0 && n_cols >= 0 && E >= 0, FGNN_ERR_SHAPE, "fgnn_coo2csr: bad sizes");
    FGNN_REQUIRE(E <= 2147483647LL - RS_TPB * 8, FGNN_ERR_LIMIT, "fgnn_coo2csr: E=%lld exceeds int32 positions", (long long)E);
    FGNN_REQUIRE(row_ptr && n_out && (E == 0 || (dst && src && col_ind)), FGNN_ERR_NULL, "fgnn_coo2csr: NULL argument");
    hipStream_t st = (hipStream_t)stream;
    if (E == 0) {
        hipLaunchKernelGGL(fill_i32_kernel, dim3((unsigned)((n_rows + 1 + 255) / 256)), dim3(256), 0, st, row_ptr, (size_t)n_rows + 1, 0);
        int rc = fgnn_launch_status("fill_i32_kernel");
        if (rc) return rc;
        hipLaunchKernelGGL(fill_i32_kernel, dim3(1), dim3(256), 0, st, (int *)n_out, (size_t)2, 0);    // int64 zero, as a kernel
        return fgnn_launch_status("fill_i32_kernel");
    }
    FGNN_REQUIRE(n_cols >= 1 && n_rows >= 1, FGNN_ERR_SHAPE, "fgnn_coo2csr: edges without rows or columns");
    size_t need = fgnn_coo2csr_workspace_bytes(n_rows, n_cols, E);
    FGNN_REQUIRE(workspace && workspace_bytes >= need, FGNN_ERR_WORKSPACE, "fgnn_coo2csr: workspace %zu < %zu bytes", workspace_bytes, need);
    const rs_plan ps = rs_plan_of(rs_key_bits(n_cols)), pd = rs_plan_of(rs_key_bits(n_rows));
    const size_t kb = fgnn_align256((size_t)E * sizeof(int)), rb = fgnn_align256((size_t)E * sizeof(int2));
    char *w = (char *)workspace;
    int *key[2];
    int2 *rec[2];
    for (int i = 0; i < 2; ++i) { key[i] = (int *)w; w += kb; rec[i] = (int2 *)w; w += rb; }
    int *hist = (int *)w; w += rs_hist_bytes(E, ps.bits > pd.bits ? ps.bits : pd.bits);
    const int nt = (int)((E + SC_TILE - 1) / SC_TILE);
    int *sums = (int *)w; w += fgnn_align256(((size_t)nt + 1) * sizeof(int));
    int *total = (int *)w;

    const int passes = ps.passes + pd.passes;
    int rc = 0;
    for (int i = 0; i < passes && !rc; ++i) {
        const bool by_src = i < ps.passes;
        const int bits = by_src ? ps.bits : pd.bits, shift = bits * (by_src ? i : i - ps.passes);
        rs_args A = {};
        A.a = dst; A.b = src;
        A.key = key[(i - 1) & 1]; A.rec = rec[(i - 1) & 1];
        A.key_out = key[i & 1]; A.rec_out = rec[i & 1];
        if (!edge_pos) {                                    // records {dst, src}
            if (i == 0) rc = rs_pass<RS_ARRAYS, RS_TO_PAIR, true>(A, src, 1, E, shift, bits, hist, st);
            else if (by_src) rc = rs_pass<RS_PAIR, RS_TO_PAIR, true>(A, (const int *)A.rec + 1, 2, E, shift, bits, hist, st);
            else rc = rs_pass<RS_PAIR, RS_TO_PAIR, false>(A, (const int *)A.rec, 2, E, shift, bits, hist, st);
        } else {                                            // src, {dst, edge}; then dst, {src, edge}
            if (i == 0) rc = rs_pass<RS_EDGES, RS_TO_TRIPLE, false>(A, src, 1, E, shift, bits, hist, st);
            else if (i == ps.passes) rc = rs_pass<RS_TRIPLE_SWAP, RS_TO_TRIPLE, false>(A, (const int *)A.rec, 2, E, shift, bits, hist, st);
            else rc = rs_pass<RS_TRIPLE, RS_TO_TRIPLE, false>(A, A.key, 1, E, shift, bits, hist, st);
        }
    }
    if (rc) return rc;
    const int *skey = key[(passes - 1) & 1];
    const int2 *srec = rec[(passes - 1) & 1];
    if (dedupe) {
        if (edge_pos) hipLaunchKernelGGL(coo_count_kernel<true>, dim3(nt), dim3(256), 0, st, E, skey, srec, sums);
        else hipLaunchKernelGGL(coo_count_kernel<false>, dim3(nt), dim3(256), 0, st, E, skey, srec, sums);
        rc = fgnn_launch_status("coo_count_kernel");
        if (rc) return rc;
        hipLaunchKernelGGL(scan_sums_kernel, dim3(1), dim3(SC_SUMS_TPB), 0, st, nt, sums, total);
        rc = fgnn_launch_status("scan_sums_kernel");
        if (rc) return rc;
    }
    if (edge_pos) hipLaunchKernelGGL(coo_write_kernel<true>, dim3(nt), dim3(256), 0, st, E, n_rows, skey, srec, dedupe ? sums : nullptr, col_ind, row_ptr, n_out, edge_pos);
    else hipLaunchKernelGGL(coo_write_kernel<false>, dim3(nt), dim3(256), 0, st, E, n_rows, skey, srec, dedupe ? sums : nullptr, col_ind, row_ptr, n_out, nullptr);
    return fgnn_launch_status("coo_write_kernel");
}
