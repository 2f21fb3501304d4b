// Triplets -> unique BCOO sorted by (row, col) with duplicates summed, on the
// GPU (the job of Converter::convert, linear_system/utils/converter.cu:137-284,
// and optionally Converter::ge2sym, :286-336, which keeps row <= col).
//
// Instead of a global radix sort of (row << 32 | col) keys, triplets are
// bucketed by block row (integer histogram, scan, scatter) and each row's
// bucket -- a few dozen entries for a mesh -- is ordered by (col, input
// index) with a rank sort in registers, one wavefront per row (longer rows in
// LDS).  The order inside a duplicate group is the input order, so every sum
// is formed in a fixed order and the output is bit-reproducible.
//
// Bound by the values (72 B per triplet and per unique block) and, before
// them, by the atomics of the histogram.  4.04 M triplets in element order,
// 591 k unique blocks, in this form (and with an atomic per triplet in the count and
// the scatter, a sort in LDS and a thread per unique block): count 36 (148),
// scatter 16 (230), row sort 65 (148), sums 107 us (319), 3.3 TB/s of their
// bytes.
#include "converter.hpp"

#include <algorithm>
#include <stdexcept>
#include <string>

namespace masx
{
namespace
{
constexpr int kScanBlock = 256;
constexpr int kScanItems = 8;               // elements per thread in the block scan
constexpr int kScanTile  = kScanBlock * kScanItems;
constexpr int kRowRegs   = 128;             // longest row sorted in registers (two keys per lane)
constexpr int kRowCap    = 1024;            // longest row sorted in LDS; longer rows sort in global scratch
// The rows longer than kRowRegs go to 64 lists (a workgroup's to the list of its
// index), their counts a line apart, and at most 40 one-wave workgroups walk a
// list: as many as the keys' LDS lets run at once.  20,000 rows of 200 triplets
// in random order: 228 us of queueing at one list's counter and 691 of sorting
// (1,024 workgroups, keys read by flat instructions), 8 and 160 now; a walk by
// 16 workgroups a list takes 7-15 % longer over 140 to 1,000 triplets a row.
constexpr int kLongLists = 64, kLongPerList = 40, kLongStride = 16;
constexpr uint32_t kHead = 0x80000000u;     // bucket entry: first of its column run (an input index has 31 bits)
constexpr uint32_t kNone = 0xffffffffu;     // rank of a triplet that is dropped

enum ConvFlag : int { kBadIndex = 1 };

// Counts the triplets of every row and gives each its place in its row's
// bucket (its arrival there: any order will do, the sort below fixes it), so
// the scatter needs no atomics of its own.  Lanes of a wave with the same row
// (element order repeats a tet's rows) share one atomic; after kMerge
// distinct rows the rest take one each, and all of a wave's atomics go out
// in one instruction.
// The rule holds out of order too, where nearly every lane keeps an atomic of
// its own: 2.3 M triplets of a 29^3 grid, shuffled, take 553 us with an atomic per
// triplet in the count and the scatter, 338 this way (in element order 730, 190).
constexpr int kMerge = 24;
__global__ void __launch_bounds__(256) k_conv_count(int n, int nr, const int* __restrict__ rows,
                                                    const int* __restrict__ cols, int drop_lower, int* row_count,
                                                    uint32_t* __restrict__ rank, int* flag)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = threadIdx.x & 63;
    int  r = -1;
    bool ok = false;
    if(t < n)
    {
        r = rows[t];
        const int c = cols[t];
        if(r < 0 || r >= nr || c < 0 || c >= nr)
            atomicOr(flag, (int)kBadIndex);
        else
            ok = !(drop_lower && r > c);
    }
    unsigned long long left = __ballot(ok);
    int leader = lane, before = 0, size = ok ? 1 : 0;
    for(int k = 0; k < kMerge && left; ++k)
    {
        const int first = __ffsll((long long)left) - 1;
        const int row = __builtin_amdgcn_readlane(r, first);
        const bool mine = ok && r == row;
        const unsigned long long same = __ballot(mine);
        if(mine)
        {
            leader = first;
            before = __popcll(same & ((1ull << lane) - 1ull));
            size   = __popcll(same);
        }
        left &= ~same;
    }
    int base = 0;
    if(ok && leader == lane) base = atomicAdd(&row_count[r], size);
    base = __shfl(base, leader, 64);
    if(t < n) rank[t] = ok ? (uint32_t)(base + before) : kNone;
}

__global__ void __launch_bounds__(256) k_conv_scatter(int n, const int* __restrict__ rows,
                                                      const uint32_t* __restrict__ rank,
                                                      const int* __restrict__ row_start, uint32_t* __restrict__ bucket)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if(t >= n) return;
    const uint32_t k = rank[t];
    if(k != kNone) bucket[row_start[rows[t]] + k] = (uint32_t)t;
}

// exclusive scan, level 1: each workgroup scans one tile and emits its total
__global__ void __launch_bounds__(kScanBlock) k_scan_tiles(const int* in, int* out, int m, int* tile_sums)
{
    __shared__ int s[kScanBlock];
    const int base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
    int v[kScanItems], sum = 0;
#pragma unroll
    for(int k = 0; k < kScanItems; ++k)
    {
        v[k] = base + k < m ? in[base + k] : 0;
        sum += v[k];
    }
    s[threadIdx.x] = sum;
    __syncthreads();
    for(int off = 1; off < kScanBlock; off <<= 1)
    {
        const int add = threadIdx.x >= off ? s[threadIdx.x - off] : 0;
        __syncthreads();
        s[threadIdx.x] += add;
        __syncthreads();
    }
    int run = s[threadIdx.x] - sum;  // exclusive prefix of this thread
#pragma unroll
    for(int k = 0; k < kScanItems; ++k)
    {
        if(base + k < m) out[base + k] = run;
        run += v[k];
    }
    if(threadIdx.x == kScanBlock - 1) tile_sums[blockIdx.x] = s[kScanBlock - 1];
}

// level 2: every workgroup sums the totals of the tiles before its own
__global__ void __launch_bounds__(kScanBlock) k_scan_add(int* out, int m, const int* tile_sums, int tiles)
{
    __shared__ int s[kScanBlock];
    const int mine = blockIdx.x;
    int before = 0;
    for(int i = threadIdx.x; i < mine; i += kScanBlock) before += tile_sums[i];
    s[threadIdx.x] = before;
    __syncthreads();
    for(int off = kScanBlock / 2; off > 0; off >>= 1)
    {
        if((int)threadIdx.x < off) s[threadIdx.x] += s[threadIdx.x + off];
        __syncthreads();
    }
    const int add = s[0];
    const int i = mine * kScanTile + threadIdx.x;
#pragma unroll
    for(int k = 0; k < kScanItems; ++k)
        if(i + k * kScanBlock < m) out[i + k * kScanBlock] += add;
    if(mine == tiles - 1 && threadIdx.x == 0) out[m] = add + tile_sums[mine];
}

// One wavefront per block row of at most kRowRegs triplets: ordered by (col,
// input index) in registers, each lane ranking its two keys against every
// other (readlane broadcasts), then the input indices in that order with the
// first of every column run marked.  Longer rows are listed for the kernel
// below.
__global__ void __launch_bounds__(256) k_conv_row_sort(int nr, const int* __restrict__ row_start,
                                                       uint32_t* __restrict__ bucket, const int* __restrict__ cols,
                                                       int* __restrict__ uniq, int* __restrict__ long_rows,
                                                       int list_cap, int* n_long)
{
    const int r = blockIdx.x * 4 + (int)(threadIdx.x >> 6);
    if(r >= nr) return;
    const int rs = row_start[r], L = row_start[r + 1] - rs, lane = threadIdx.x & 63;
    if(L > kRowRegs)
    {
        const int list = blockIdx.x % kLongLists;
        if(lane == 0) long_rows[(size_t)list * list_cap + atomicAdd(&n_long[list * kLongStride], 1)] = r;
        return;
    }
    uint32_t t[2], c[2];
    int      rank[2] = {0, 0};
#pragma unroll
    for(int h = 0; h < 2; ++h) t[h] = lane + 64 * h < L ? bucket[rs + lane + 64 * h] : 0u;
#pragma unroll
    for(int h = 0; h < 2; ++h) c[h] = lane + 64 * h < L ? (uint32_t)cols[t[h]] : 0xffffffffu;
    unsigned long long key[2];
#pragma unroll
    for(int h = 0; h < 2; ++h) key[h] = ((unsigned long long)c[h] << 32) | t[h];
    const int n0 = __builtin_amdgcn_readfirstlane(min(L, 64)), n1 = __builtin_amdgcn_readfirstlane(L - min(L, 64));
    for(int j = 0; j < n0; ++j)
    {
        const unsigned long long k = ((unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)c[0], j) << 32) |
                                     (uint32_t)__builtin_amdgcn_readlane((int)t[0], j);
        rank[0] += k < key[0];
        rank[1] += k < key[1];
    }
    for(int j = 0; j < n1; ++j)
    {
        const unsigned long long k = ((unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)c[1], j) << 32) |
                                     (uint32_t)__builtin_amdgcn_readlane((int)t[1], j);
        rank[0] += k < key[0];
        rank[1] += k < key[1];
    }
    // to sorted order through LDS (keys are distinct: rank = position)
    __shared__ uint32_t s_t[4][kRowRegs], s_c[4][kRowRegs];
    uint32_t* st = s_t[threadIdx.x >> 6];
    uint32_t* sc = s_c[threadIdx.x >> 6];
#pragma unroll
    for(int h = 0; h < 2; ++h)
        if(lane + 64 * h < L)
        {
            st[rank[h]] = t[h];
            sc[rank[h]] = c[h];
        }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    int count = 0;
#pragma unroll
    for(int h = 0; h < 2; ++h)
    {
        const int  i = lane + 64 * h;
        const bool head = i < L && (i == 0 || sc[i] != sc[i - 1]);
        if(i < L) bucket[rs + i] = st[i] | (head ? kHead : 0u);
        count += __popcll(__ballot(head));
    }
    if(lane == 0) uniq[r] = count;
}

// The rows longer than kRowRegs, one wavefront each, with the keys in LDS (or
// global scratch past kRowCap): a lane ranks four of its keys at a time against
// every key.  The two places are told apart outside the loops, so the LDS
// reads are LDS instructions.
__global__ void __launch_bounds__(64) k_conv_row_sort_long(const int* __restrict__ long_rows, int list_cap,
                                                           const int* n_long, const int* __restrict__ row_start,
                                                           uint32_t* bucket, const int* __restrict__ cols,
                                                           unsigned long long* gkeys, unsigned long long* gsorted,
                                                           int* uniq)
{
    __shared__ unsigned long long s_keys[kRowCap], s_sorted[kRowCap];
    const int lane = threadIdx.x, list = blockIdx.x % kLongLists;
    const int rows_left = n_long[list * kLongStride];
    auto sort_row = [&](int r, int rs, int L, unsigned long long* keys, unsigned long long* sorted) {
        for(int i = lane; i < L; i += 64)
        {
            const uint32_t t = bucket[rs + i];
            keys[i] = ((unsigned long long)(uint32_t)cols[t] << 32) | t;
        }
        __syncthreads();
        // keys are distinct (the input index is part of the key): rank = position
        for(int i = lane; i < L; i += 256)
        {
            unsigned long long k[4];
            int                rank[4];
#pragma unroll
            for(int h = 0; h < 4; ++h)
            {
                k[h]    = keys[min(i + 64 * h, L - 1)];
                rank[h] = 0;
            }
#pragma unroll 4
            for(int j = 0; j < L; ++j)
            {
                const unsigned long long o = keys[j];
#pragma unroll
                for(int h = 0; h < 4; ++h) rank[h] += o < k[h];
            }
#pragma unroll
            for(int h = 0; h < 4; ++h)
                if(i + 64 * h < L) sorted[rank[h]] = k[h];
        }
        __syncthreads();
        int count = 0;
        for(int base = 0; base < L; base += 64)
        {
            const int i = base + lane;
            const unsigned long long k = i < L ? sorted[i] : 0;
            const bool head = i < L && (i == 0 || (k >> 32) != (sorted[i - 1] >> 32));
            count += __popcll(__ballot(head));
            if(i < L) bucket[rs + i] = (uint32_t)(k & 0xffffffffu) | (head ? kHead : 0u);
        }
        if(lane == 0) uniq[r] = count;
        __syncthreads();  // the next row reuses the LDS
    };
    for(int q = blockIdx.x / kLongLists; q < rows_left; q += gridDim.x / kLongLists)
    {
        const int r = long_rows[(size_t)list * list_cap + q], rs = row_start[r], L = row_start[r + 1] - rs;
        if(L <= kRowCap)
            sort_row(r, rs, L, s_keys, s_sorted);
        else
            sort_row(r, rs, L, gkeys + rs, gsorted + rs);
    }
}

// One wavefront per block row: its triplets' values pass through LDS in
// chunks of 63 (nine lanes read a block's 72 contiguous bytes), and the lanes
// sum the runs there, in input order, into 9 contiguous values per unique
// block.  A run that a chunk cuts is carried over to the next.
constexpr int kWriteChunk = 63;
__global__ void __launch_bounds__(256) k_conv_write(int nr, const int* __restrict__ row_start,
                                                    const uint32_t* __restrict__ bucket,
                                                    const int* __restrict__ out_start, const int* __restrict__ cols,
                                                    const double* __restrict__ vals, int* __restrict__ out_rows,
                                                    int* __restrict__ out_cols, double* __restrict__ out_vals)
{
    __shared__ double s_v[4][kWriteChunk * 9];
    __shared__ double s_carry[4][2][9];  // read from one, written to the other
    __shared__ int    s_head[4][64];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = blockIdx.x * 4 + wave;
    if(r >= nr) return;
    const int rs = __builtin_amdgcn_readfirstlane(row_start[r]);
    const int re = __builtin_amdgcn_readfirstlane(row_start[r + 1]);
    long long o = out_start[r];  // unique blocks finished before the current chunk's first run
    double* V = s_v[wave];
    int     flip = 0;
    int*    H = s_head[wave];
    const int g = lane / 9, q = lane % 9;
    for(int c0 = rs; c0 < re; c0 += kWriteChunk)
    {
        const int n = min(kWriteChunk, re - c0);
        const uint32_t code = lane < n ? bucket[c0 + lane] : 0u;
        const int t = (int)(code & ~kHead);
        const unsigned long long heads = __ballot(lane < n && (code & kHead));
        const int cont = heads & 1ull ? 0 : 1;  // the chunk begins inside a run
        const int runs = __popcll(heads) + cont;
        const bool open = c0 + n < re && !(bucket[c0 + n] & kHead);  // its last run goes on
        if(lane < n && (code & kHead))
        {
            const int k = __popcll(heads & ((1ull << lane) - 1ull)) + cont;
            H[k] = lane;
            out_rows[o + k] = r;
            out_cols[o + k] = cols[t];
        }
        if(cont && lane == 0) H[0] = 0;
        double v[9];
#pragma unroll
        for(int k = 0; k < 9; ++k)
        {
            const int e = min(g + 7 * k, n - 1);
            v[k] = __builtin_nontemporal_load(vals + 9 * (long long)__shfl(t, e, 64) + q);
        }
#pragma unroll
        for(int k = 0; k < 9; ++k)
            if(g + 7 * k < n && lane < 63) V[9 * (g + 7 * k) + q] = v[k];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        for(int i = lane; i < 9 * runs; i += 64)
        {
            const int k = i / 9, c = i - 9 * k;
            const int b = H[k], e = k + 1 < runs ? H[k + 1] : n;
            double acc = k == 0 && cont ? s_carry[wave][flip][c] : 0.0;
            for(int j = b; j < e; ++j) acc += V[9 * j + c];
            if(k + 1 == runs && open)
                s_carry[wave][flip ^ 1][c] = acc;
            else
                out_vals[9 * o + i] = acc;
        }
        o += runs - (open ? 1 : 0);
        flip ^= 1;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

unsigned grid_for(long long n, int b) { return (unsigned)((n + b - 1) / b); }

#define CONV_HIP(x)                                                                                      \
    do {                                                                                                 \
        const hipError_t e_ = (x);                                                                       \
        if(e_ != hipSuccess) throw std::runtime_error(std::string("converter: ") + hipGetErrorString(e_)); \
    } while(0)

template <typename T>
void grow(T*& p, size_t& cap, size_t need)
{
    if(need <= cap) return;
    if(p) (void)hipFree(p);
    p = nullptr;
    cap = 0;
    CONV_HIP(hipMalloc((void**)&p, need * sizeof(T)));
    cap = need;
}
}  // namespace

Converter::~Converter()
{
    for(void* p : {(void*)row_count_, (void*)row_start_, (void*)rank_, (void*)bucket_, (void*)uniq_, (void*)out_start_,
                   (void*)tiles_, (void*)long_rows_, (void*)keys_, (void*)sorted_})
        if(p) (void)hipFree(p);
    if(h_pinned_) (void)hipHostFree(h_pinned_);
}

void Converter::scan(const int* in, int* out, int m, hipStream_t st)
{
    // out[0..m] = exclusive prefix sums of in[0..m-1]; out[m] = total
    const int tiles = std::max(1, (m + kScanTile - 1) / kScanTile);
    grow(tiles_, tiles_cap_, (size_t)tiles);
    hipLaunchKernelGGL(k_scan_tiles, dim3(tiles), dim3(kScanBlock), 0, st, in, out, m, tiles_);
    hipLaunchKernelGGL(k_scan_add, dim3(tiles), dim3(kScanBlock), 0, st, out, m, tiles_, tiles);
    CONV_HIP(hipGetLastError());
}

int Converter::convert(int n, int n_block_rows, const int* rows, const int* cols, const double* vals, int drop_lower,
                       int* out_rows, int* out_cols, double* out_vals, hipStream_t st)
{
    if(n < 0 || n_block_rows <= 0) throw std::invalid_argument("bad triplet or block-row count");
    if(n == 0) return 0;
    if(!rows || !cols || !vals || !out_rows || !out_cols || !out_vals) throw std::invalid_argument("null pointer");
    const int nr = n_block_rows;
    // row counts, then the bad-index flag and the counts of the long rows' lists (one clear)
    const size_t n_clear  = ((size_t)nr + 1 + kLongLists * kLongStride + 3) / 4 * 4;
    const int    list_cap = (int)((grid_for(nr, 4) + kLongLists - 1) / kLongLists) * 4;
    grow(row_count_, row_count_cap_, n_clear);
    grow(row_start_, row_start_cap_, (size_t)nr + 1);
    grow(uniq_, uniq_cap_, (size_t)nr);
    grow(out_start_, out_start_cap_, (size_t)nr + 1);
    grow(long_rows_, long_rows_cap_, (size_t)list_cap * kLongLists);
    grow(rank_, rank_cap_, (size_t)n);
    grow(bucket_, bucket_cap_, (size_t)n);
    grow(keys_, keys_cap_, (size_t)n);
    grow(sorted_, sorted_cap_, (size_t)n);
    if(!h_pinned_) CONV_HIP(hipHostMalloc((void**)&h_pinned_, 2 * sizeof(int), hipHostMallocDefault));
    int *flag = row_count_ + nr, *n_long = flag + 1;

    CONV_HIP(hipMemsetAsync(row_count_, 0, sizeof(int) * n_clear, st));
    hipLaunchKernelGGL(k_conv_count, dim3(grid_for(n, 256)), dim3(256), 0, st, n, nr, rows, cols, drop_lower,
                       row_count_, rank_, flag);
    CONV_HIP(hipGetLastError());
    scan(row_count_, row_start_, nr, st);
    hipLaunchKernelGGL(k_conv_scatter, dim3(grid_for(n, 256)), dim3(256), 0, st, n, rows, rank_, row_start_, bucket_);
    hipLaunchKernelGGL(k_conv_row_sort, dim3(grid_for(nr, 4)), dim3(256), 0, st, nr, row_start_, bucket_, cols, uniq_,
                       long_rows_, list_cap, n_long);
    const int per_list = std::min({list_cap, kLongPerList, n / kRowRegs + 1});  // no list holds more rows
    hipLaunchKernelGGL(k_conv_row_sort_long, dim3((unsigned)(kLongLists * per_list)), dim3(64), 0, st, long_rows_, list_cap, n_long, row_start_, bucket_, cols, keys_, sorted_, uniq_);
    CONV_HIP(hipGetLastError());
    scan(uniq_, out_start_, nr, st);
    hipLaunchKernelGGL(k_conv_write, dim3(grid_for(nr, 4)), dim3(256), 0, st, nr, row_start_, bucket_, out_start_, cols,
                       vals, out_rows, out_cols, out_vals);
    CONV_HIP(hipGetLastError());
    CONV_HIP(hipMemcpyAsync(h_pinned_, out_start_ + nr, sizeof(int), hipMemcpyDeviceToHost, st));
    CONV_HIP(hipMemcpyAsync(h_pinned_ + 1, flag, sizeof(int), hipMemcpyDeviceToHost, st));
    CONV_HIP(hipStreamSynchronize(st));
    if(h_pinned_[1] & kBadIndex) throw std::invalid_argument("triplet block index outside [0, n_block_rows)");
    return h_pinned_[0];
}

}  // namespace masx
