// Sort-by-tet and compaction of the particle arrays.
//
// Keys: owning tet for live particles, n_tets for live particles outside the
// mesh, n_tets + 1 for settled ones.  Ordering by key puts particles of a tet
// next to each other (coalesced tet/E/map loads, few distinct nodes per block
// for the charge reduction) and moves settled particles behind the live ones;
// the step kernels then only cover the live prefix (n_active).
//
// The keys are small integers, so a counting sort places every row with one
// count per key: rank (each row's place among those of its key), the key
// counts' prefix sums, one scatter of every array.  Four launches, bound by the
// scatter's memory traffic and, where rows are in no order, by the atomics of
// the ranks; a library radix sort of (key, row) pairs took some 20 passes of
// 6 us each.  With one sort each, 200 fused steps of 1M particles on 750k tets
// went from 1.17 to 1.09 ms, 100 steps of 150,001 particles on 179k tets from
// 274 to 233 us.
// Large populations whose ranks' atomics and scattered stores cost more are
// radix sorted instead (below).
// The order of the rows of one key is not fixed (nothing depends on it but
// the order in which charges are added).
#include "kernels.h"

namespace sg {

constexpr int kScan = 4096;  // keys per workgroup of the prefix sums: 256 threads x 4 int4

__host__ __device__ inline int64_t padded_keys(int64_t n_tets) { return (n_tets + 2 + kScan - 1) / kScan * kScan; }

__device__ inline int32_t key_of(int32_t tet, int32_t flags, int32_t n_tets)
{
    return (flags & kSettled) ? n_tets + 1 : (tet < 0 ? n_tets : tet);
}

// rank[j]: row j's place among the rows of its key; count (zero on entry): rows
// per key.  Atomics to one address queue at about 6 ns each, so there is one
// per run of equal keys in a wave (after the first sort rows are nearly in
// order), one per workgroup for each of the two keys of particles without a
// tet, which lie scattered among the others, and one for a workgroup whose
// rows are all in one tet (a point source).  Against one atomic per wave and
// key: 93 -> 13 us for 1M rows of which half come from a point, 33 -> 10 us for
// 262,144 rows of which a growing part has settled.
constexpr int kRankThreads = 1024;
__global__ void __launch_bounds__(kRankThreads) rank_kernel(const int32_t* __restrict__ tet,
                                                            const int32_t* __restrict__ flags, int64_t n,
                                                            int32_t n_tets, int32_t* __restrict__ count,
                                                            int32_t* __restrict__ rank)
{
    constexpr int kWaves = kRankThreads / 64;
    __shared__ int32_t s_key[kWaves], s_cnt[2][kWaves], s_base[3];
    const int64_t j = blockIdx.x * (int64_t)kRankThreads + threadIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const unsigned long long below = (1ull << lane) - 1, upto = below | 1ull << lane;
    const int32_t key = j < n ? key_of(tet[j], flags[j], n_tets) : -1;
    const int32_t before = __shfl_up(key, 1);
    const bool head = lane == 0 || before != key;
    const unsigned long long heads = __ballot(head);
    const unsigned long long m0 = __ballot(key == n_tets), m1 = __ballot(key == n_tets + 1);
    if (lane == 0) {
        s_key[wave] = heads == 1ull && key < n_tets ? key : -1;  // the wave's only key
        s_cnt[0][wave] = __popcll(m0);
        s_cnt[1][wave] = __popcll(m1);
    }
    __syncthreads();
    bool one = s_key[0] >= 0;
    int32_t total[2] = {0, 0}, mine[2] = {0, 0};  // rows of the two keys: the workgroup's, the earlier waves'
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        one = one && s_key[w] == s_key[0];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            mine[q] += w < wave ? s_cnt[q][w] : 0;
            total[q] += s_cnt[q][w];
        }
    }
    if (threadIdx.x < 2 && total[threadIdx.x] > 0)
        s_base[threadIdx.x] = atomicAdd(&count[n_tets + (int)threadIdx.x], total[threadIdx.x]);
    if (threadIdx.x == 2 && one) s_base[2] = atomicAdd(&count[s_key[0]], kRankThreads);
    int32_t r = 0;
    if (key >= 0 && key < n_tets && head && !one) {
        const unsigned long long rest = heads & ~upto;
        const int end = rest ? __ffsll((long long)rest) - 1 : 64;
        r = atomicAdd(&count[key], end - lane);
    }
    const int first = 63 - __clzll((long long)(heads & upto));
    r = __shfl(r, first) + (lane - first);
    __syncthreads();
    if (one) r = s_base[2] + (int32_t)threadIdx.x;
    else if (key == n_tets) r = s_base[0] + mine[0] + __popcll(m0 & below);
    else if (key == n_tets + 1) r = s_base[1] + mine[1] + __popcll(m1 & below);
    if (j < n) rank[j] = r;
}

__device__ inline int32_t wave_sum(int32_t v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// rows of each workgroup's kScan keys
__global__ void __launch_bounds__(256) key_sums_kernel(const int4* __restrict__ count, int32_t* __restrict__ sums)
{
    __shared__ int32_t part[4];
    int32_t v = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int4 c = count[blockIdx.x * (int64_t)(kScan / 4) + k * 256 + threadIdx.x];
        v += (c.x + c.y) + (c.z + c.w);
    }
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) sums[blockIdx.x] = (part[0] + part[1]) + (part[2] + part[3]);
}

// first row of every key: the sums of the workgroups before this one (a few
// hundred), then the keys before each in its own part.  count is left zero for
// the next sort; the settled rows start where the live ones end.
__global__ void __launch_bounds__(256) key_starts_kernel(int4* __restrict__ count, const int32_t* __restrict__ sums,
                                                         int4* __restrict__ start, int32_t n_tets,
                                                         int64_t* __restrict__ n_active)
{
    __shared__ int32_t part[4];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    int32_t v = 0;
    for (unsigned b = threadIdx.x; b < blockIdx.x; b += 256) v += sums[b];
    v = wave_sum(v);
    if (lane == 0) part[wave] = v;
    __syncthreads();
    int32_t carry = (part[0] + part[1]) + (part[2] + part[3]);
    for (int k = 0; k < 4; ++k) {
        const int64_t at = blockIdx.x * (int64_t)(kScan / 4) + k * 256 + threadIdx.x;
        const int4 c = count[at];
        count[at] = make_int4(0, 0, 0, 0);
        const int32_t own = (c.x + c.y) + (c.z + c.w);
        int32_t upto = own;  // of the wave's lanes up to this one
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int32_t w = __shfl_up(upto, off);
            if (lane >= off) upto += w;
        }
        __syncthreads();  // part is read by all before it is written again
        if (lane == 63) part[wave] = upto;
        __syncthreads();
        int32_t s = carry + upto - own;
#pragma unroll
        for (int w = 0; w < 4; ++w) s += w < wave ? part[w] : 0;
        carry += (part[0] + part[1]) + (part[2] + part[3]);
        const int4 st = make_int4(s, s + c.x, s + c.x + c.y, s + c.x + c.y + c.z);
        start[at] = st;
        const int64_t q = (int64_t)n_tets + 1 - 4 * at;
        if (q >= 0 && q < 4) *n_active = q == 0 ? st.x : (q == 1 ? st.y : (q == 2 ? st.z : st.w));
    }
}

template <typename R>
__global__ void place_kernel(DevParticles<R> src, R* __restrict__ x, R* __restrict__ y, R* __restrict__ z,
                             double* __restrict__ vx, double* __restrict__ vy, double* __restrict__ vz,
                             int32_t* __restrict__ tet, int32_t* __restrict__ flags, int32_t* __restrict__ hit,
                             uint32_t* __restrict__ pidx, const int32_t* __restrict__ rank,
                             const int32_t* __restrict__ start, int32_t n_tets, int64_t n)
{
    const int64_t s = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (s >= n) return;
    const int32_t t = src.tet[s], f = src.flags[s];
    const int64_t j = (int64_t)start[key_of(t, f, n_tets)] + rank[s];
    if (j >= n) return;  // (only if a launch of an earlier sort failed and left counts behind)
    x[j] = src.x[s];
    y[j] = src.y[s];
    z[j] = src.z[s];
    vx[j] = src.vx[s];
    vy[j] = src.vy[s];
    vz[j] = src.vz[s];
    tet[j] = t;
    flags[j] = f;
    hit[j] = src.hit[s];
    pidx[j] = src.pidx[s];
}

// ---------------------------------------------------------------------------
// Large populations: radix sort of (key, row) by 11 bits a pass, two passes for
// up to 4M tets, then a gather.  Four short launches a pass; the gather's random
// reads bound it.  A sort in us, FP64, by a library radix sort and gather, by the
// counting sort, by this one:
//   rows on tets          unordered              nearly ordered
//   1M on 374k        324    294    225      220    125    143
//   2M on 3M          461    578    432      271    300    250
//   2M on 750k        480    562    455      164     75    123
//   4M on 720k        860  1,199    845      466    575    440
//   4M on 750k        910    890    882      240    153    201
//   8M on 3M        1,737  2,119  1,690    1,010  1,230    960
//   8M on 750k      1,788  2,288  1,765      455    335    350
//   16M on 3M       3,500  5,030  3,400    2,090  2,350  1,940
//   24.6M on 750k   6,300  9,109  6,190    1,355  1,100  1,030
// (nearly ordered: on 3M, 720k and 374k tets particles cross some two tets
// between sorts, on 750k few do.)  Where the rows are new (in no order), 1M of
// them suffice; where fewer than two share a tet, every row is a run of its own
// to the counting sort, and 1.5M do; else it is the rows that moved, which the
// host does not know, and from 4M on this one is taken as the library's was.
// ---------------------------------------------------------------------------
constexpr int64_t kRadixRows = 1'000'000;
static bool use_radix(int64_t n, int64_t n_tets, bool unordered)
{
    return n >= 4 * kRadixRows || (unordered && n >= kRadixRows) || (2 * n >= 3 * kRadixRows && n < 2 * n_tets);
}
constexpr int kDigitBits = 11, kDigits = 1 << kDigitBits;
constexpr int kTileThreads = 1024, kTileWaves = kTileThreads / 64, kTileSteps = 8;
constexpr int kTileRows = kTileThreads * kTileSteps;
constexpr int kChunks = 32;  // of the tiles, for the prefix sums

// The (key, row) pairs of a workgroup's tile: the rows as they are in the first
// pass.  Wave w holds rows w * 512.. of it, 64 at a time: rows ascend with
// (wave, step, lane).  Rows past the end repeat the last one.
struct RadixIn {
    const int32_t *tet, *flags;
    const int2* pairs;
    int64_t n;
    int32_t n_tets, shift;
    __device__ inline int32_t digit(int32_t key) const { return key >> shift & (kDigits - 1); }
};
template <bool kFirst>
struct RadixTile {
    int64_t first;
    int rows;  // of the tile
    int2 pair[kTileSteps];
    __device__ inline int row(int step) const
    {
        return (threadIdx.x >> 6) * (64 * kTileSteps) + step * 64 + (threadIdx.x & 63);
    }
    __device__ inline void load(const RadixIn& in)
    {
        first = blockIdx.x * (int64_t)kTileRows;
        rows = (int)min((int64_t)kTileRows, in.n - first);
#pragma unroll
        for (int i = 0; i < kTileSteps; ++i) {
            const unsigned r = (unsigned)min(row(i), rows - 1);
            pair[i] = kFirst ? make_int2(key_of((in.tet + first)[r], (in.flags + first)[r], in.n_tets), (int)(first + r))
                             : (in.pairs + first)[r];
        }
    }
};

// rows per (tile, digit), and the settled rows per tile
template <bool kFirst>
__global__ void __launch_bounds__(kTileThreads, 8) radix_count_kernel(RadixIn in, int32_t* __restrict__ hist,
                                                                      int32_t* __restrict__ settled)
{
    __shared__ int32_t count[kDigits];
    RadixTile<kFirst> tile;
    tile.load(in);
    for (int d = threadIdx.x; d < kDigits; d += kTileThreads) count[d] = 0;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kTileSteps; ++i)
        if (tile.row(i) < tile.rows) atomicAdd(&count[in.digit(tile.pair[i].x)], 1);
    __syncthreads();
    for (int d = threadIdx.x; d < kDigits; d += kTileThreads) hist[blockIdx.x * (int64_t)kDigits + d] = count[d];
    if (kFirst) {
        int s = 0;
#pragma unroll
        for (int i = 0; i < kTileSteps; ++i) s += __syncthreads_count(tile.row(i) < tile.rows && tile.pair[i].x == in.n_tets + 1);
        if (threadIdx.x == 0) settled[blockIdx.x] = s;
    }
}

// A workgroup takes 64 digits of a chunk of tiles.  sums: rows per (chunk, digit).
constexpr int kChunkWaves = 4;
__device__ inline int64_t chunk_first(int64_t tiles, int chunk) { return tiles * chunk / kChunks; }
__global__ void __launch_bounds__(64 * kChunkWaves) digit_sums_kernel(const int32_t* __restrict__ hist, int64_t tiles,
                                                                      int32_t* __restrict__ sums)
{
    __shared__ int32_t part[kChunkWaves][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, d = blockIdx.x * 64 + lane;
    const int64_t a = chunk_first(tiles, blockIdx.y), b = chunk_first(tiles, blockIdx.y + 1);
    int32_t v = 0;
    for (int64_t t = a + wave; t < b; t += kChunkWaves) v += hist[t * kDigits + d];
    part[wave][lane] = v;
    __syncthreads();
    if (wave == 0) sums[blockIdx.y * kDigits + d] = (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
}
// hist -> place of a tile's rows among those of the digit, in place (a thread
// per chunk and digit); totals: rows of the digit
__global__ void __launch_bounds__(64) digit_starts_kernel(int32_t* __restrict__ hist, int64_t tiles,
                                                          const int32_t* __restrict__ sums,
                                                          int32_t* __restrict__ totals)
{
    const int d = blockIdx.x * 64 + threadIdx.x;
    const int64_t a = chunk_first(tiles, blockIdx.y), b = chunk_first(tiles, blockIdx.y + 1);
    int32_t before[kChunks], r = 0;
#pragma unroll
    for (int k = 0; k < kChunks; ++k) before[k] = sums[k * kDigits + d];
#pragma unroll
    for (int k = 0; k < kChunks; ++k) r += k < (int)blockIdx.y ? before[k] : 0;
    int64_t t = a;
    for (; t + 8 <= b; t += 8) {
        int32_t c[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) c[q] = hist[(t + q) * kDigits + d];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            hist[(t + q) * kDigits + d] = r;
            r += c[q];
        }
    }
    for (; t < b; ++t) {
        const int32_t c = hist[t * kDigits + d];
        hist[t * kDigits + d] = r;
        r += c;
    }
    if (blockIdx.y == kChunks - 1) totals[d] = r;
}

// Every row to its place by the pass's digit, rows of one digit in the order
// they had (start: places of the tiles' rows within the digit).  Lanes of equal
// digit find each other by one ballot per bit; the counters are a wave's own, so
// nothing is added atomically.  The last pass leaves the rows alone.
template <bool kFirst>
__global__ void __launch_bounds__(kTileThreads, 8) radix_place_kernel(RadixIn in, const int32_t* __restrict__ start,
                                                                      const int32_t* __restrict__ totals,
                                                                      int2* __restrict__ pairs_out,
                                                                      int32_t* __restrict__ rows_out)
{
    __shared__ uint16_t count[kTileWaves][kDigits];  // at most kTileRows
    __shared__ int32_t base[kDigits], s_wave[kTileWaves];
    static_assert(kDigits == 2 * kTileThreads, "two digits a thread");
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    RadixTile<kFirst> tile;
    tile.load(in);
    {
        // first row of each digit
        const int2 c = ((const int2*)totals)[threadIdx.x];
        int32_t upto = c.x + c.y;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int32_t w = __shfl_up(upto, off);
            if (lane >= off) upto += w;
        }
        if (lane == 63) s_wave[wave] = upto;
        __syncthreads();
        int32_t r = upto - c.x - c.y;
#pragma unroll
        for (int w = 0; w < kTileWaves; ++w) r += w < wave ? s_wave[w] : 0;
        base[2 * threadIdx.x] = r;
        base[2 * threadIdx.x + 1] = r + c.x;
    }
    int32_t at[kTileSteps];
    for (int d = threadIdx.x; d < kTileWaves * kDigits / 2; d += kTileThreads) ((uint32_t*)count)[d] = 0u;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kTileSteps; ++i) {
        const int32_t d = in.digit(tile.pair[i].x);
        const bool valid = tile.row(i) < tile.rows;
        const unsigned long long live = __ballot(valid);
        uint32_t lo = (uint32_t)live, hi = (uint32_t)(live >> 32);  // lanes of this digit
#pragma unroll
        for (int b = 0; b < kDigitBits; ++b) {
            const uint32_t bit = (uint32_t)((int32_t)((uint32_t)d << (31 - b)) >> 31);  // in every place
            const unsigned long long m = __ballot(bit);
            lo &= ~((uint32_t)m ^ bit);
            hi &= ~((uint32_t)(m >> 32) ^ bit);
        }
        const int before = (int)__builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0u));
        // (a wave's LDS accesses keep their order)
        const int32_t c = count[wave][d];
        at[i] = c + before;
        if (valid && before == 0) count[wave][d] = (uint16_t)(c + __popc(lo) + __popc(hi));
        asm volatile("" ::: "memory");
    }
    __syncthreads();
    for (int d = threadIdx.x; d < kDigits; d += kTileThreads) {
        uint16_t c[kTileWaves], sum = 0;  // of the earlier waves
#pragma unroll
        for (int w = 0; w < kTileWaves; ++w) c[w] = count[w][d];
#pragma unroll
        for (int w = 0; w < kTileWaves; ++w) {
            count[w][d] = sum;
            sum += c[w];
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kTileSteps; ++i) {
        const unsigned d = (unsigned)in.digit(tile.pair[i].x);
        at[i] += (start + blockIdx.x * (int64_t)kDigits)[d] + base[d] + count[wave][d];
    }
#pragma unroll
    for (int i = 0; i < kTileSteps; ++i) {
        // (a place past the end: only if an earlier launch failed)
        if (tile.row(i) >= tile.rows || (unsigned)at[i] >= (uint64_t)in.n) continue;
        if (pairs_out) pairs_out[(unsigned)at[i]] = tile.pair[i];
        else rows_out[(unsigned)at[i]] = tile.pair[i].y;
    }
}

// Row perm[j] to j, two arrays at a time (with all ten loads in flight the
// lines of a wave drive each other out of the caches: 1,745 against 1,574 us
// for 16M nearly ordered rows).  The live rows lead: all but the settled ones
// of the tiles.
template <typename R>
__global__ void __launch_bounds__(256) gather_rows_kernel(DevParticles<R> src, R* __restrict__ x, R* __restrict__ y,
                                                          R* __restrict__ z, double* __restrict__ vx,
                                                          double* __restrict__ vy, double* __restrict__ vz,
                                                          int32_t* __restrict__ tet, int32_t* __restrict__ flags,
                                                          int32_t* __restrict__ hit, uint32_t* __restrict__ pidx,
                                                          const int32_t* __restrict__ perm, int64_t n,
                                                          const int32_t* __restrict__ settled, int64_t tiles,
                                                          int64_t* __restrict__ n_active)
{
    const int64_t j = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (j < n) {
        const int64_t s = min((int64_t)(uint32_t)perm[j], n - 1);
        x[j] = src.x[s];
        y[j] = src.y[s];
        asm volatile("" ::: "memory");
        z[j] = src.z[s];
        vx[j] = src.vx[s];
        asm volatile("" ::: "memory");
        vy[j] = src.vy[s];
        vz[j] = src.vz[s];
        asm volatile("" ::: "memory");
        tet[j] = src.tet[s];
        flags[j] = src.flags[s];
        asm volatile("" ::: "memory");
        hit[j] = src.hit[s];
        pidx[j] = src.pidx[s];
    }
    if (blockIdx.x == 0) {
        __shared__ int32_t part[4];
        int32_t v = 0;
        for (int64_t t = threadIdx.x; t < tiles; t += 256) v += settled[t];
        v = wave_sum(v);
        if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
        __syncthreads();
        if (threadIdx.x == 0) *n_active = n - ((part[0] + part[1]) + (part[2] + part[3]));
    }
}

// Scratch of the sort besides the ranks, in int32: the key counts (zero
// before the first sort), the key starts, the workgroup sums.
size_t sort_scratch_len(int64_t n_tets)
{
    const size_t k = (size_t)padded_keys(n_tets);
    return 2 * k + (k / kScan + 3) / 4 * 4;
}
size_t sort_zeroed_len(int64_t n_tets) { return (size_t)padded_keys(n_tets); }

template <typename R>
hipError_t sort_particles(hipStream_t s, const DevParticles<R>& P, R* x, R* y, R* z, double* vx, double* vy, double* vz,
                          int32_t* tet, int32_t* flags, int32_t* hit, uint32_t* pidx, int32_t* rank, int32_t* scratch,
                          WorkItem* work, int32_t n_tets, bool unordered, int64_t* n_active)
{
    const int64_t n = P.n;
    if (n == 0) return hipSuccess;
    if (use_radix(n, n_tets, unordered)) {
        const int64_t tiles = (n + kTileRows - 1) / kTileRows;
        // pairs (two sets), counts and their sums in the work list's rows
        static_assert(kRadixRows * sizeof(WorkItem) >=
                          kRadixRows * 2 * sizeof(int2) +
                              (kRadixRows / kTileRows + 1) * (kDigits + 1) * sizeof(int32_t) +
                              kDigits * (kChunks + 1) * sizeof(int32_t) && sizeof(WorkItem) >= 2 * sizeof(int2) + 2,
                      "scratch of the radix sort");
        int2* pairs[2] = {(int2*)work, (int2*)work + n};
        int32_t *hist = (int32_t*)(pairs[1] + n), *sums = hist + kDigits * tiles, *totals = sums + kDigits * kChunks,
                *settled = totals + kDigits;
        int32_t* const perm = rank;
        const unsigned tb = (unsigned)tiles;
        const dim3 parts(kDigits / 64, kChunks);
        RadixIn in{P.tet, P.flags, nullptr, n, n_tets, 0};
        for (int set = 0;; set ^= 1) {
            const bool first = in.shift == 0, last = ((int64_t)n_tets + 1) >> in.shift < kDigits;
            int2* const out = last ? nullptr : pairs[set];
            if (first) radix_count_kernel<true><<<tb, kTileThreads, 0, s>>>(in, hist, settled);
            else radix_count_kernel<false><<<tb, kTileThreads, 0, s>>>(in, hist, settled);
            digit_sums_kernel<<<parts, 64 * kChunkWaves, 0, s>>>(hist, tiles, sums);
            digit_starts_kernel<<<parts, 64, 0, s>>>(hist, tiles, sums, totals);
            if (first) radix_place_kernel<true><<<tb, kTileThreads, 0, s>>>(in, hist, totals, out, perm);
            else radix_place_kernel<false><<<tb, kTileThreads, 0, s>>>(in, hist, totals, out, perm);
            if (last) break;
            in.pairs = out;
            in.shift += kDigitBits;
        }
        gather_rows_kernel<R><<<(unsigned)((n + 255) / 256), 256, 0, s>>>(P, x, y, z, vx, vy, vz, tet, flags, hit, pidx,
                                                                           perm, n, settled, tiles, n_active);
        return hipGetLastError();
    }
    const int64_t keys = padded_keys(n_tets);
    int32_t *count = scratch, *start = scratch + keys, *sums = scratch + 2 * keys;
    const unsigned nb = (unsigned)((n + 255) / 256), kb = (unsigned)(keys / kScan);
    rank_kernel<<<(unsigned)((n + kRankThreads - 1) / kRankThreads), kRankThreads, 0, s>>>(P.tet, P.flags, n, n_tets, count, rank);
    key_sums_kernel<<<kb, 256, 0, s>>>((const int4*)count, sums);
    key_starts_kernel<<<kb, 256, 0, s>>>((int4*)count, sums, (int4*)start, n_tets, n_active);
    place_kernel<R><<<nb, 256, 0, s>>>(P, x, y, z, vx, vy, vz, tet, flags, hit, pidx, rank, start, n_tets, n);
    return hipGetLastError();
}

template hipError_t sort_particles<double>(hipStream_t, const DevParticles<double>&, double*, double*, double*,
                                           double*, double*, double*, int32_t*, int32_t*, int32_t*, uint32_t*,
                                           int32_t*, int32_t*, WorkItem*, int32_t, bool,
                                           int64_t*);
template hipError_t sort_particles<float>(hipStream_t, const DevParticles<float>&, float*, float*, float*, double*,
                                          double*, double*, int32_t*, int32_t*, int32_t*, uint32_t*, int32_t*,
                                          int32_t*, WorkItem*, int32_t, bool,
                                           int64_t*);

}  // namespace sg
