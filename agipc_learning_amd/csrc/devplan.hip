// Structure analysis of one MAS system on the device (see devplan.hpp).
// Integer work: counting, stable sorts and scans over the matrix structure,
// bound by memory latency; every output is a pure function of the inputs (no
// order of atomics reaches an output: atomics only count or take a maximum).
#include "devplan.hpp"

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include "device.hpp"
#include "spmv_layout.hpp"
#include "wave_prefix.hpp"

namespace masx
{
namespace
{
constexpr int kThreads = 256;

inline int grid_for(long long n, int per = kThreads)
{
    const long long g = (n + per - 1) / per;
    return (int)(g < 1 ? 1 : (g > 65536 ? 65536 : g));
}

__device__ __forceinline__ int packed_index(int bank, int r, int c) { return bank * r - r * (r + 1) / 2 + c; }

// first entry of row r whose column is >= c (columns sorted within a row)
__device__ __forceinline__ int first_ge(const int* row_ptr, const int* col, int r, int c)
{
    int lo = row_ptr[r], hi = row_ptr[r + 1];
    while(lo < hi)
    {
        const int mid = (lo + hi) >> 1;
        if(col[mid] < c)
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo;
}

// the system whose range [off[s], off[s+1]) holds x (off increasing, n_sys >= 1)
__device__ __forceinline__ int system_of(const int* off, int n_sys, long long x)
{
    int lo = 0, hi = n_sys - 1;
    while(lo < hi)
    {
        const int mid = (lo + hi + 1) >> 1;
        if(off[mid] <= x)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

constexpr uint64_t kDpSentinel = ~(uint64_t)0;

// exclusive scan of v over a 256-thread workgroup (s: 256 ints of LDS);
// returns the exclusive prefix, *total the sum
__device__ int block_exclusive_scan(int v, int* s, int* total)
{
    const int t = threadIdx.x;
    s[t] = v;
    __syncthreads();
    for(int off = 1; off < kThreads; off <<= 1)
    {
        const int a = t >= off ? s[t - off] : 0;
        __syncthreads();
        s[t] += a;
        __syncthreads();
    }
    const int incl = s[t];
    *total = s[kThreads - 1];
    __syncthreads();
    return incl - v;
}

__global__ void k_dp_fill(int* p, int value, long long n)
{
    for(long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        p[i] = value;
}

__global__ void k_dp_csr_items(long long nb, const int* rows, const int* cols, DpSystems sys, const int* e2i,
                               int n_rows, int bits, uint64_t* keys, int* vals, int* diag_src, int* err)
{
    const uint64_t sentinel = (uint64_t)n_rows << bits;
    for(long long k = blockIdx.x * (long long)blockDim.x + threadIdx.x; k < nb; k += (long long)gridDim.x * blockDim.x)
    {
        const int s = system_of(sys.src_off, sys.n_sys, k);
        const int e0 = sys.ext_off[s], n_ext = sys.ext_off[s + 1] - e0;
        const int r = rows[k], c = cols[k];
        if((unsigned)r >= (unsigned)n_ext || (unsigned)c >= (unsigned)n_ext)
        {
            atomicOr(err, 1);
            keys[2 * k] = keys[2 * k + 1] = sentinel;
            vals[2 * k] = vals[2 * k + 1] = -1;
            continue;
        }
        const int iR = e2i[e0 + r];
        if(r == c)
        {
            keys[2 * k]     = (uint64_t)iR << bits | (uint64_t)iR;
            vals[2 * k]     = (int)k;
            keys[2 * k + 1] = sentinel;
            vals[2 * k + 1] = -1;
            atomicMax(&diag_src[iR], (int)k);  // the last diagonal block of the row
        }
        else
        {
            const int iC    = e2i[e0 + c];
            keys[2 * k]     = (uint64_t)iR << bits | (uint64_t)iC;
            vals[2 * k]     = (int)k;
            keys[2 * k + 1] = (uint64_t)iC << bits | (uint64_t)iR;
            vals[2 * k + 1] = (int)k | (int)0x80000000u;
        }
    }
}

// row_ptr from the sorted items: row r starts at the first item of a row >= r.
// The starts fall out of the sort; counting them as the items are made took an
// atomic an item (46 us for 590,000 blocks, 17 without) and a scan.
__global__ void k_dp_row_starts(long long n, const uint64_t* keys, int bits, int n_rows, int* row_ptr)
{
    for(long long x = blockIdx.x * (long long)blockDim.x + threadIdx.x; x <= n; x += (long long)gridDim.x * blockDim.x)
    {
        const int r = x < n ? (int)(keys[x] >> bits) : n_rows;
        for(int q = x > 0 ? (int)(keys[x - 1] >> bits) + 1 : 0; q <= r; ++q) row_ptr[q] = (int)x;
    }
}

__global__ void k_dp_csr_fill(long long nnz, const uint64_t* keys, const int* vals, int bits, int* col, int* entry_src)
{
    const uint64_t mask = ((uint64_t)1 << bits) - 1;
    for(long long x = blockIdx.x * (long long)blockDim.x + threadIdx.x; x < nnz; x += (long long)gridDim.x * blockDim.x)
    {
        col[x]       = (int)(keys[x] & mask);
        entry_src[x] = vals[x];
    }
}

__global__ void k_dp_gal_items(int lvl, long long n, const int* rows, const int* cols, const int* EI, const int* EJ,
                               const int* ES, int e_prev, DpSystems sys, const int* gn_all, const int* lvl_begin,
                               int bits, uint64_t* keys, int* vals, int* n_valid)
{
    // valid items are counted in LDS: a global add per thread made every wave
    // queue at one address (34 us a level from 0.6 million items, 9 now
    // with four items a thread)
    __shared__ int s_valid;
    if(threadIdx.x == 0) s_valid = 0;
    __syncthreads();
    int valid = 0;
    for(long long k = blockIdx.x * (long long)blockDim.x + threadIdx.x; k < n; k += (long long)gridDim.x * blockDim.x)
    {
        const int s = lvl == 1 ? system_of(sys.src_off, sys.n_sys, k) : ES[e_prev + k];
        if(sys.levels[s] <= lvl)
        {
            keys[k] = kDpSentinel;
            vals[k] = -1;
            continue;
        }
        const int* gn = gn_all + sys.gn_off[s];
        int a, b, src;
        bool diag;
        if(lvl == 1)
        {
            const int r = rows[k], c = cols[k];
            a    = gn[r];
            b    = gn[c];
            diag = r == c;
            src  = (int)k;
        }
        else
        {
            const int pi = EI[e_prev + k], pj = EJ[e_prev + k];
            a    = gn[pi];
            b    = gn[pj];
            diag = pi == pj;
            src  = e_prev + (int)k;
        }
        int I, J, mode;
        if(a < b) { I = a; J = b; mode = 0; }
        else if(a > b) { I = b; J = a; mode = 1; }
        else { I = a; J = a; mode = diag ? 0 : 2; }
        const int lb = lvl_begin[s];
        keys[k] = (uint64_t)s << (2 * bits) | (uint64_t)(I - lb) << bits | (uint64_t)(J - lb);
        vals[k] = src << 2 | mode;
        ++valid;
    }
    if(valid) atomicAdd(&s_valid, valid);
    __syncthreads();
    if(threadIdx.x == 0 && s_valid) atomicAdd(n_valid, s_valid);
}

__global__ void k_dp_run_ends(long long n, const uint64_t* keys, int* flag)
{
    for(long long x = blockIdx.x * (long long)blockDim.x + threadIdx.x; x <= n; x += (long long)gridDim.x * blockDim.x)
        flag[x] = x == n || keys[x] == kDpSentinel ? 0 : (x + 1 == n || keys[x + 1] != keys[x] ? 1 : 0);
}

__global__ void k_dp_gal_fill(long long n, const uint64_t* keys, const int* vals, const int* flag, const int* qpos,
                              int g_base, int e_base, const int* lvl_begin, int bits, int* gal_src, int* gal_ptr,
                              int* EI, int* EJ, int* ES)
{
    const uint64_t mask = ((uint64_t)1 << bits) - 1;
    for(long long x = blockIdx.x * (long long)blockDim.x + threadIdx.x; x < n; x += (long long)gridDim.x * blockDim.x)
    {
        const uint64_t key = keys[x];
        if(key == kDpSentinel) continue;  // sorted last: x is past the level's items
        gal_src[g_base + x] = vals[x];
        if(flag[x])
        {
            const int s  = (int)(key >> (2 * bits));
            const int lb = lvl_begin[s];
            const int q  = e_base + qpos[x];
            EI[q]          = lb + (int)((key >> bits) & mask);
            EJ[q]          = lb + (int)(key & mask);
            ES[q]          = s;
            gal_ptr[q + 1] = g_base + (int)x + 1;
        }
    }
}

__global__ void k_dp_ent_count_rows(int n_slots, int bank, const int* row_ptr, const int* col, const int* entry_src,
                                    int* row_cnt)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if(r > n_slots) return;
    int c = 0;
    if(r < n_slots)
    {
        const int r0 = r / bank * bank;
        for(int e = row_ptr[r]; e < row_ptr[r + 1]; ++e)
            c += entry_src[e] >= 0 && col[e] >= r0 && col[e] < r0 + bank;
    }
    row_cnt[r] = c;  // row_cnt[n_slots] = 0 closes the scan
}

__global__ void k_dp_ent_fill_rows(int n_slots, int bank, const int* row_ptr, const int* col, const int* entry_src,
                                   const int* row_off, int* pos, int* src)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if(r >= n_slots) return;
    const int r0 = r / bank * bank, lr = r - r0;
    int at = row_off[r];
    for(int e = row_ptr[r]; e < row_ptr[r + 1]; ++e)
    {
        const int lc = col[e] - r0;
        if(entry_src[e] < 0 || lc < 0 || lc >= bank) continue;  // transposed copy, or another bank
        pos[at] = (lr <= lc ? packed_index(bank, lr, lc) : packed_index(bank, lc, lr)) | (lr > lc ? 1 : 0) << 16;
        src[at] = entry_src[e];
        ++at;
    }
}

__device__ __forceinline__ int coarse_bank_of(const DpSystems& sys, int n_fine_banks, int bank, int s, int I)
{
    return n_fine_banks + (sys.coarse_base[s] + I - sys.n_slots[s]) / bank;
}

// Coarse entries are sorted by their row node within a level, so the lanes of
// a wave hold runs of entries whose rows lie in one bank: one atomic a run (one
// an entry queued at the bank's counter: 41 us each on a 40^3 grid's levels, 5 now).
// The lanes of this lane's run, all of them active.
__device__ __forceinline__ unsigned long long bank_run(int gb)
{
    const int lane = (int)threadIdx.x & 63;
    const int before = __shfl_up(gb, 1);
    const unsigned long long heads = __ballot(lane == 0 || before != gb);
    const unsigned long long upto = heads & (~0ull >> (63 - lane));       // heads at or before this lane
    const int first = 63 - __clzll((long long)upto);                      // lane 0 is a head
    const unsigned long long after = lane == 63 ? 0 : heads >> (lane + 1);
    const int last = after ? lane + __ffsll((long long)after) - 1 : 63;
    return (~0ull >> (63 - last)) & (~0ull << first);
}

__global__ void k_dp_ent_flag_coarse(int n_gal, int bank, int n_fine_banks, DpSystems sys, const int* EI, const int* EJ,
                                     const int* ES, int* flag, int* bank_cnt)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    int f = 0, gb = -1;
    if(e < n_gal)
    {
        const int I = EI[e], J = EJ[e];
        f  = I / bank == J / bank;
        gb = coarse_bank_of(sys, n_fine_banks, bank, ES[e], I);
    }
    const unsigned long long in_run = __ballot(f) & bank_run(gb);  // the run's entries inside the bank
    if(f && __ffsll((long long)in_run) - 1 == ((int)threadIdx.x & 63)) atomicAdd(&bank_cnt[gb], __popcll(in_run));
    if(e <= n_gal) flag[e] = f;
}

__global__ void k_dp_ent_first_coarse(int n_gal, int bank, int n_fine_banks, DpSystems sys, const int* EI,
                                      const int* ES, const int* flag, const int* fpos, int* bank_first)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    const bool in = e < n_gal;
    const int  f  = in ? flag[e] : 0;
    const int  gb = in ? coarse_bank_of(sys, n_fine_banks, bank, ES[e], EI[e]) : -1;
    const unsigned long long in_run = __ballot(f) & bank_run(gb);
    // fpos grows with e: the run's first entry holds its smallest
    if(f && __ffsll((long long)in_run) - 1 == ((int)threadIdx.x & 63)) atomicMin(&bank_first[gb], fpos[e]);
}

__global__ void k_dp_ent_fill_coarse(int n_gal, int bank, int n_fine_banks, DpSystems sys, const int* EI,
                                     const int* EJ, const int* ES, const int* flag, const int* fpos,
                                     const int* bank_first, const int* bank_ptr, int* pos, int* src)
{
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    if(e >= n_gal || !flag[e]) return;
    const int gb = coarse_bank_of(sys, n_fine_banks, bank, ES[e], EI[e]);
    const int at = bank_ptr[gb] + fpos[e] - bank_first[gb];
    pos[at] = packed_index(bank, EI[e] % bank, EJ[e] % bank);
    src[at] = e;
}

__global__ void k_dp_ent_bank_counts(int n_fine_banks, int bank, const int* row_off, int* bank_cnt)
{
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if(b < n_fine_banks) bank_cnt[b] = row_off[(b + 1) * bank] - row_off[b * bank];
}

// the greedy tile that starts at r0 (build_spmv_layout's cut, from any r0).
// Bound by the chain of row searches behind one start: a thread that adds its
// rows one by one makes ~100 dependent ones (165 us on 68,921 rows, 36 now).  Here a
// wave takes a start, its lanes 64 rows at a time: each lane finds what its row
// adds, a prefix sum finds the row that no longer fits.  A workgroup takes
// kSlStarts consecutive starts, whose tiles can only reach the next
// kSlStarts + kSpmvTileRows - 1 rows: their row pointers, the place of their
// diagonals and, when they fit kSlCols, their columns are staged in LDS.
constexpr int kSlStarts  = 128;
constexpr int kSlRows    = kSlStarts + kSpmvTileRows;
constexpr int kSlCols    = 12288;
constexpr int kSlThreads = 1024;

__global__ void __launch_bounds__(kSlThreads) k_dp_sl_next(int n, const int* row_ptr, const int* col,
                                                           const int* row_sys, const int* row_off, int cap, int* nxt,
                                                           int* kept)
{
    __shared__ int s_ptr[kSlRows + 1];
    __shared__ int s_diag[kSlRows];
    __shared__ int s_end[kSlStarts];
    __shared__ int s_col[kSlCols];
    const int R = blockIdx.x * kSlStarts;
    const int rw = min(n, R + kSlRows);  // rows [R, rw) are staged
    for(int i = threadIdx.x; i <= rw - R; i += kSlThreads) s_ptr[i] = row_ptr[R + i];
    // a tile ends at its system's end or at kSpmvTileRows
    for(int i = threadIdx.x; i < min(kSlStarts, n - R); i += kSlThreads)
        s_end[i] = min(row_off[row_sys[R + i] + 1], R + i + kSpmvTileRows);
    __syncthreads();
    const int e0 = s_ptr[0], ne = s_ptr[rw - R] - e0;
    const bool cached = ne <= kSlCols;  // uniform
    if(cached)
        for(int i = threadIdx.x; i < ne; i += kSlThreads) s_col[i] = col[e0 + i];
    __syncthreads();
    // first entry in [lo, hi) whose column is >= c
    auto first_ge_s = [&](int lo, int hi, int c) {
        while(lo < hi)
        {
            const int mid = (lo + hi) >> 1;
            if((cached ? s_col[mid - e0] : col[mid]) < c)
                lo = mid + 1;
            else
                hi = mid;
        }
        return lo;
    };
    for(int i = threadIdx.x; i < rw - R; i += kSlThreads) s_diag[i] = first_ge_s(s_ptr[i], s_ptr[i + 1], R + i);
    __syncthreads();
    const int lane = (int)threadIdx.x & 63;
    for(int r0 = R + (int)threadIdx.x / 64; r0 < min(n, R + kSlStarts); r0 += kSlThreads / 64)  // uniform in a wave
    {
        const int r_end = s_end[r0 - R];
        int k = s_ptr[r0 + 1 - R] - s_ptr[r0 - R];
        int r1 = r0 + 1;
        while(r1 < r_end)
        {
            // r < r_end <= min(n, R + kSlRows - 1): inside the staged rows
            const int r = r1 + lane;
            int q = 0;
            if(r < r_end)
                q = (s_ptr[r + 1 - R] - s_diag[r - R]) + (first_ge_s(s_ptr[r - R], s_diag[r - R], r0) - s_ptr[r - R]);
            const int sum = wave_prefix(q);
            const unsigned long long stop = __ballot(r >= r_end || k + sum > cap);
            if(stop)
            {
                const int f = __ffsll((long long)stop) - 1;  // the first row that is not added
                if(f > 0) k += __shfl(sum, f - 1);
                r1 += f;
                break;
            }
            k += __shfl(sum, 63);
            r1 += 64;
        }
        if(lane == 0)
        {
            nxt[r0]  = r1;
            kept[r0] = k;
        }
    }
}

// The chain of tiles from row 0, one workgroup, in windows of the tile ends
// staged in LDS (each step r -> nxt[r] advances by 1..256 rows).  One thread
// walking the window is a chain of ~300 LDS reads (63 us on 68,921 rows, 24 now), so
// the window is cut into segments: for each of the 256 rows where the chain
// can enter one, a thread walks it to its end; one thread then links the
// segments, and a thread per segment writes its tiles.
constexpr int kChainWindow   = 32768;
constexpr int kChainSegment  = 2048;  // longer than a step
constexpr int kChainSegments = kChainWindow / kChainSegment;
__global__ void __launch_bounds__(1024) k_dp_sl_chain(int n, const int* nxt, int* ts, int* n_tiles)
{
    __shared__ unsigned char step[kChainWindow];
    __shared__ int walk[kChainSegments * kSpmvTileRows];  // [segment][entry]: tiles << 8 | rows past the end
    __shared__ int s_entry[kChainSegments], s_first[kChainSegments];
    __shared__ int s_r, s_t;
    if(threadIdx.x == 0)
    {
        s_r = 0;
        s_t = 0;
    }
    for(;;)
    {
        __syncthreads();
        const int w0 = s_r;
        if(w0 >= n) break;  // uniform: every thread read the same s_r
        const int wn = min(kChainWindow, n - w0);
        const int ns = (wn + kChainSegment - 1) / kChainSegment;
#pragma unroll 8
        for(int i = threadIdx.x; i < wn; i += 1024) step[i] = (unsigned char)(nxt[w0 + i] - (w0 + i) - 1);
        __syncthreads();
        for(int i = threadIdx.x; i < ns * kSpmvTileRows; i += 1024)
        {
            const int g = i / kSpmvTileRows, end = min(wn, (g + 1) * kChainSegment);
            int r = g * kChainSegment + i % kSpmvTileRows, t = 0;
            while(r < end)
            {
                r += step[r] + 1;
                ++t;
            }
            walk[i] = t << 8 | ((r - end) & 255);  // r - end <= 255 wherever the chain enters
        }
        __syncthreads();
        if(threadIdx.x == 0)
        {
            int entry = 0, t = s_t;
            for(int g = 0; g < ns; ++g)
            {
                s_entry[g] = entry;
                s_first[g] = t;
                const int w = walk[g * kSpmvTileRows + entry];
                t += w >> 8;
                entry = w & 255;
            }
            s_r = w0 + wn + entry;
            s_t = t;
        }
        __syncthreads();
        if((int)threadIdx.x < ns)
        {
            const int g = (int)threadIdx.x, end = min(wn, (g + 1) * kChainSegment);
            int t = s_first[g];
            for(int r = g * kChainSegment + s_entry[g]; r < end; r += step[r] + 1) ts[t++] = w0 + r;
        }
    }
    if(threadIdx.x == 0) *n_tiles = s_t;
}

__global__ void __launch_bounds__(kThreads) k_dp_sl_tile_counts(int n_tiles, int n, const int* ts, const int* kept,
                                                                const int* row_ptr, const int* col, int* kept_al,
                                                                int* trans, int* err)
{
    __shared__ int s[kThreads];
    const int t = blockIdx.x;
    if(t > n_tiles) return;  // uniform per workgroup
    if(t == n_tiles)
    {
        if(threadIdx.x == 0) kept_al[t] = trans[t] = 0;  // closes both scans
        return;
    }
    const int r0 = ts[t], r1 = t + 1 < n_tiles ? ts[t + 1] : n, r = r0 + (int)threadIdx.x;
    int q = 0;
    if(r < r1) q = first_ge(row_ptr, col, r, r1) - first_ge(row_ptr, col, r, r + 1);
    int total;
    (void)block_exclusive_scan(q, s, &total);
    if(threadIdx.x == 0)
    {
        trans[t]   = total;
        kept_al[t] = (kept[r0] + kSpmvAlign - 1) / kSpmvAlign * kSpmvAlign;
        if(total > kSpmvMaxCap) atomicOr(err, 4);  // tpos has 14 bits
    }
}

// One tile's words.  Eight lanes take a row; a row's entries before the tile's
// first column (s_below) and from its diagonal on (s_diag) are kept, so an
// entry's place follows from its own index.  Columns are searched in LDS when
// the tile's fit kFillCols (a thread per row walking and searching in global
// memory: 75 us on 68,921 rows, 18 now).
constexpr int kFillCols = 6144;

__global__ void __launch_bounds__(kThreads) k_dp_sl_fill(int n_tiles, int n, const int* ts, const int* kept,
                                                         const int* e_base, const int* q_base, const int* row_ptr,
                                                         const int* col, const int* entry_src, const int* row_sys,
                                                         int* L_row_ptr, int* L_tptr, int* L_col, int* L_src, int4* wg,
                                                         int2* wg_ent, int* err)
{
    __shared__ int s_scan[kThreads];
    __shared__ int s_tstart[kThreads], s_ptr[kThreads + 1], s_below[kThreads], s_diag[kThreads], s_out[kThreads];
    __shared__ int s_col[kFillCols];
    const int t = blockIdx.x;
    const int r0 = ts[t], r1 = t + 1 < n_tiles ? ts[t + 1] : n, nr = r1 - r0;
    const int j = (int)threadIdx.x, r = r0 + j;
    const int x0 = row_ptr[r0], nx = row_ptr[r1] - x0;
    const bool cached = nx <= kFillCols;  // uniform
    for(int i = j; i <= nr; i += kThreads) s_ptr[i] = row_ptr[r0 + i];
    if(cached)
        for(int i = j; i < nx; i += kThreads) s_col[i] = col[x0 + i];
    __syncthreads();
    auto col_at = [&](int e) { return cached ? s_col[e - x0] : col[e]; };
    auto first_ge_s = [&](int lo, int hi, int c) {  // first entry in [lo, hi) whose column is >= c
        while(lo < hi)
        {
            const int mid = (lo + hi) >> 1;
            if(col_at(mid) < c)
                lo = mid + 1;
            else
                hi = mid;
        }
        return lo;
    };
    int cnt = 0, kr = 0;
    if(j < nr)
    {
        const int d = first_ge_s(s_ptr[j], s_ptr[j + 1], r), b = first_ge_s(s_ptr[j], d, r0);
        cnt = d - b;                                  // entries (r', r), r0 <= r' < r: by symmetry
        kr  = (s_ptr[j + 1] - d) + (b - s_ptr[j]);    // entries row r keeps
        s_diag[j]  = d;
        s_below[j] = b;
    }
    int n_trans, n_kept;
    const int tst  = block_exclusive_scan(cnt, s_scan, &n_trans);
    const int koff = block_exclusive_scan(kr, s_scan, &n_kept);
    s_tstart[j] = tst;
    s_out[j]    = e_base[t] + koff;
    __syncthreads();
    if(j == 0 && n_trans > kSpmvMaxCap) atomicOr(err, 4);
    if(n_trans <= kSpmvMaxCap)
    {
        if(j < nr)
        {
            L_row_ptr[r] = s_out[j];
            L_tptr[r]    = q_base[t] + tst;
        }
        for(int w = j / 8; w < nr; w += kThreads / 8)
        {
            const int rr = r0 + w, p = s_ptr[w], b = s_below[w], d = s_diag[w];
            for(int e = p + j % 8; e < s_ptr[w + 1]; e += 8)
            {
                if(e >= b && e < d) continue;  // the tile's lower copy: its upper twin covers it
                const int c = col_at(e), at = e < b ? e - p : e - d + (b - p);
                unsigned word = (unsigned)c;
                if(e >= d && c < r1)
                {
                    const int k = c - r0;
                    const int tpos = c == rr ? 0
                                             : s_tstart[k] + (first_ge_s(s_below[k], s_diag[k], rr) - s_below[k]) +
                                                   (e - first_ge_s(d, e, c));
                    word = kSpmvInTile | (unsigned)tpos << 16 | (unsigned)w << 8 | (unsigned)k;
                }
                if(at == 0) word |= kSpmvRowStart;
                L_col[s_out[w] + at] = (int)word;
                L_src[s_out[w] + at] = entry_src[e];
            }
        }
    }
    if(j == 0)
    {
        wg[t]     = make_int4(row_sys[r0], kWgPlain << 28, r0, r1);
        wg_ent[t] = make_int2(e_base[t], e_base[t] + kept[r0]);
        if(t == n_tiles - 1)
        {
            L_row_ptr[n] = e_base[t] + kept[r0];
            L_tptr[n]    = q_base[t] + n_trans;
        }
    }
}

__global__ void k_dp_sl_pad(long long total, int* L_col, int* L_src)
{
    for(long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < total; i += (long long)gridDim.x * blockDim.x)
    {
        L_col[i] = 0;
        L_src[i] = kSpmvPadSrc;
    }
}
}  // namespace

size_t dp_sort_bytes(long long n, int end_bit)
{
    size_t bytes = 0;
    (void)rocprim::radix_sort_pairs(nullptr, bytes, (const uint64_t*)nullptr, (uint64_t*)nullptr, (const int*)nullptr,
                                    (int*)nullptr, (size_t)n, 0u, (unsigned)end_bit);
    return bytes;
}

size_t dp_scan_bytes(long long n)
{
    size_t bytes = 0;
    (void)rocprim::exclusive_scan(nullptr, bytes, (const int*)nullptr, (int*)nullptr, 0, (size_t)n,
                                  rocprim::plus<int>());
    return bytes;
}

hipError_t dp_sort(void* tmp, size_t tmp_bytes, const uint64_t* keys_in, uint64_t* keys_out, const int* vals_in,
                   int* vals_out, long long n, int end_bit, hipStream_t st)
{
    if(n <= 0) return hipSuccess;
    return rocprim::radix_sort_pairs(tmp, tmp_bytes, keys_in, keys_out, vals_in, vals_out, (size_t)n, 0u,
                                     (unsigned)end_bit, st);
}

hipError_t dp_scan(void* tmp, size_t tmp_bytes, const int* in, int* out, long long n, hipStream_t st)
{
    if(n <= 0) return hipSuccess;
    return rocprim::exclusive_scan(tmp, tmp_bytes, in, out, 0, (size_t)n, rocprim::plus<int>(), st);
}

hipError_t dp_fill(int* p, int value, long long n, hipStream_t st)
{
    if(n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_dp_fill, dim3(grid_for(n)), dim3(kThreads), 0, st, p, value, n);
    return hipGetLastError();
}

hipError_t dp_csr_items(long long nb, const int* rows, const int* cols, DpSystems sys, const int* e2i, int n_rows,
                        int bits, uint64_t* keys, int* vals, int* diag_src, int* err, hipStream_t st)
{
    if(nb <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_dp_csr_items, dim3(grid_for(nb)), dim3(kThreads), 0, st, nb, rows, cols, sys, e2i, n_rows,
                       bits, keys, vals, diag_src, err);
    return hipGetLastError();
}

hipError_t dp_row_starts(long long n, const uint64_t* keys, int bits, int n_rows, int* row_ptr, hipStream_t st)
{
    hipLaunchKernelGGL(k_dp_row_starts, dim3(grid_for(n + 1)), dim3(kThreads), 0, st, n, keys, bits, n_rows, row_ptr);
    return hipGetLastError();
}

hipError_t dp_csr_fill(long long nnz, const uint64_t* keys, const int* vals, int bits, int* col, int* entry_src,
                       hipStream_t st)
{
    if(nnz <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_dp_csr_fill, dim3(grid_for(nnz)), dim3(kThreads), 0, st, nnz, keys, vals, bits, col, entry_src);
    return hipGetLastError();
}

hipError_t dp_gal_items(int lvl, long long n, const int* rows, const int* cols, const int* EI, const int* EJ,
                        const int* ES, int e_prev, DpSystems sys, const int* gn_all, const int* lvl_begin, int bits,
                        uint64_t* keys, int* vals, int* n_valid, hipStream_t st)
{
    if(n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_dp_gal_items, dim3(grid_for(n, 4 * kThreads)), dim3(kThreads), 0, st, lvl, n, rows, cols, EI, EJ, ES,
                       e_prev, sys, gn_all, lvl_begin, bits, keys, vals, n_valid);
    return hipGetLastError();
}

hipError_t dp_run_ends(long long n, const uint64_t* keys, int* flag, hipStream_t st)
{
    hipLaunchKernelGGL(k_dp_run_ends, dim3(grid_for(n + 1)), dim3(kThreads), 0, st, n, keys, flag);
    return hipGetLastError();
}

hipError_t dp_gal_fill(long long n, const uint64_t* keys, const int* vals, const int* flag, const int* qpos,
                       int g_base, int e_base, const int* lvl_begin, int bits, int* gal_src, int* gal_ptr, int* EI,
                       int* EJ, int* ES, hipStream_t st)
{
    if(n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_dp_gal_fill, dim3(grid_for(n)), dim3(kThreads), 0, st, n, keys, vals, flag, qpos, g_base,
                       e_base, lvl_begin, bits, gal_src, gal_ptr, EI, EJ, ES);
    return hipGetLastError();
}

hipError_t dp_ent_count_rows(int n_slots, int bank, const int* row_ptr, const int* col, const int* entry_src,
                             int* row_cnt, hipStream_t st)
{
    hipLaunchKernelGGL(k_dp_ent_count_rows, dim3((n_slots + kThreads) / kThreads), dim3(kThreads), 0, st, n_slots,
                       bank, row_ptr, col, entry_src, row_cnt);
    return hipGetLastError();
}

hipError_t dp_ent_fill_rows(int n_slots, int bank, const int* row_ptr, const int* col, const int* entry_src,
                            const int* row_off, int* pos, int* src, hipStream_t st)
{
    if(n_slots <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_dp_ent_fill_rows, dim3((n_slots + kThreads - 1) / kThreads), dim3(kThreads), 0, st, n_slots,
                       bank, row_ptr, col, entry_src, row_off, pos, src);
    return hipGetLastError();
}

hipError_t dp_ent_flag_coarse(int n_gal, int bank, int n_fine_banks, DpSystems sys, const int* EI, const int* EJ,
                              const int* ES, int* flag, int* bank_cnt, hipStream_t st)
{
    hipLaunchKernelGGL(k_dp_ent_flag_coarse, dim3((n_gal + kThreads) / kThreads), dim3(kThreads), 0, st, n_gal, bank,
                       n_fine_banks, sys, EI, EJ, ES, flag, bank_cnt);
    return hipGetLastError();
}

hipError_t dp_ent_first_coarse(int n_gal, int bank, int n_fine_banks, DpSystems sys, const int* EI, const int* ES,
                               const int* flag, const int* fpos, int* bank_first, hipStream_t st)
{
    if(n_gal <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_dp_ent_first_coarse, dim3((n_gal + kThreads - 1) / kThreads), dim3(kThreads), 0, st, n_gal,
                       bank, n_fine_banks, sys, EI, ES, flag, fpos, bank_first);
    return hipGetLastError();
}

hipError_t dp_ent_fill_coarse(int n_gal, int bank, int n_fine_banks, DpSystems sys, const int* EI, const int* EJ,
                              const int* ES, const int* flag, const int* fpos, const int* bank_first,
                              const int* bank_ptr, int* pos, int* src, hipStream_t st)
{
    if(n_gal <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_dp_ent_fill_coarse, dim3((n_gal + kThreads - 1) / kThreads), dim3(kThreads), 0, st, n_gal,
                       bank, n_fine_banks, sys, EI, EJ, ES, flag, fpos, bank_first, bank_ptr, pos, src);
    return hipGetLastError();
}

hipError_t dp_ent_bank_counts(int n_fine_banks, int bank, const int* row_off, int* bank_cnt, hipStream_t st)
{
    if(n_fine_banks <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_dp_ent_bank_counts, dim3((n_fine_banks + kThreads - 1) / kThreads), dim3(kThreads), 0, st,
                       n_fine_banks, bank, row_off, bank_cnt);
    return hipGetLastError();
}

hipError_t dp_sl_next(int n, const int* row_ptr, const int* col, const int* row_sys, const int* row_off, int cap,
                      int* nxt, int* kept, hipStream_t st)
{
    if(n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_dp_sl_next, dim3((n + kSlStarts - 1) / kSlStarts), dim3(kSlThreads), 0, st, n, row_ptr, col,
                       row_sys, row_off, cap, nxt, kept);
    return hipGetLastError();
}

hipError_t dp_sl_chain(int n, const int* nxt, int* ts, int* n_tiles, hipStream_t st)
{
    hipLaunchKernelGGL(k_dp_sl_chain, dim3(1), dim3(1024), 0, st, n, nxt, ts, n_tiles);
    return hipGetLastError();
}

hipError_t dp_sl_tile_counts(int n_tiles, int n, const int* ts, const int* kept, const int* row_ptr, const int* col,
                             int* kept_al, int* trans, int* err, hipStream_t st)
{
    hipLaunchKernelGGL(k_dp_sl_tile_counts, dim3(n_tiles + 1), dim3(kThreads), 0, st, n_tiles, n, ts, kept, row_ptr,
                       col, kept_al, trans, err);
    return hipGetLastError();
}

hipError_t dp_sl_fill(int n_tiles, int n, const int* ts, const int* kept, const int* e_base, const int* q_base,
                      const int* row_ptr, const int* col, const int* entry_src, const int* row_sys, int* L_row_ptr,
                      int* L_tptr, int* L_col, int* L_src, int4* wg, int2* wg_ent, int* err, hipStream_t st)
{
    if(n_tiles <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_dp_sl_fill, dim3(n_tiles), dim3(kThreads), 0, st, n_tiles, n, ts, kept, e_base, q_base,
                       row_ptr, col, entry_src, row_sys, L_row_ptr, L_tptr, L_col, L_src, wg, wg_ent, err);
    return hipGetLastError();
}

hipError_t dp_sl_pad(long long total, int* L_col, int* L_src, hipStream_t st)
{
    if(total <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_dp_sl_pad, dim3(grid_for(total)), dim3(kThreads), 0, st, total, L_col, L_src);
    return hipGetLastError();
}
}  // namespace masx
