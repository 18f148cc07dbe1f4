// Sort-by-tet and compaction of the particle arrays.
//
// Keys: owning tet for live particles, n_tets for live particles outside the
// mesh, n_tets + 1 for settled ones.  Ordering by key puts particles of a tet
// next to each other (coalesced tet/E/map loads, few distinct nodes per block
// for the charge reduction) and moves settled particles behind the live ones;
// the step kernels then only cover the live prefix (n_active).
//
// The keys are small integers, so a counting sort places every row with one
// count per key instead of sorting (key, index) pairs: rank (each row's place
// among those of its key), the key counts' prefix sums, one scatter of every
// array.  Four launches, bound by the scatter's memory traffic; a radix sort
// of the pairs took some 20 passes of 6 us each.  With one sort each, 200
// fused steps of 1M particles on 750k tets went from 1.17 to 1.09 ms, 100 steps
// of 150,001 particles on 179k tets from 274 to 233 us.
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
                          int32_t n_tets, int64_t* n_active)
{
    const int64_t n = P.n;
    if (n == 0) return hipSuccess;
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
                                           int32_t*, int32_t*, int32_t, int64_t*);
template hipError_t sort_particles<float>(hipStream_t, const DevParticles<float>&, float*, float*, float*, double*,
                                          double*, double*, int32_t*, int32_t*, int32_t*, uint32_t*, int32_t*,
                                          int32_t*, int32_t, int64_t*);

}  // namespace sg
