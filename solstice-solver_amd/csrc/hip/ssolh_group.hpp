// Grouping of items by key (included by ssolh.hip inside its anonymous
// namespace): the realisations of a wavefront by start key, the records of
// the per-primitive log by primitive.
//
// A counting sort in three launches that read their item count from device
// memory. k_group_rank counts a block's items by key in LDS and reserves the
// block's places of each key with one global atomic; k_group_scan turns the
// keys' counts into offsets; k_group_place writes each item's index at its
// place. Items of one key keep the order of their blocks' reservations, not
// of their indices: the groups are summed, or run side by side, in any order.
//
// Up to GROUP_KEYS keys, whose counters fill 64 KB of LDS, and while the
// reservations (at most one per key and block) are few: group_pays. Beyond,
// a radix sort of (key, index) pairs makes fewer passes over memory, but
// needs the item count on the host and, below a few million items, 7 to 20
// launches of 5 us each. 1e6 realisations over 10,003 keys: 103 us by radix
// sort, 53 us grouped; 5e4 records over 4,096 keys: 75 and 15 us.
constexpr uint32_t GROUP_KEYS = 16384;
constexpr int GROUP_THREADS = 1024, GROUP_PER = 4;
constexpr uint32_t GROUP_BLOCK = GROUP_THREADS * GROUP_PER;  // items of a block

bool group_pays(uint64_t items, uint64_t keys) {
  const uint64_t reservations = (items / GROUP_BLOCK + 1) * std::min<uint64_t>(keys, GROUP_BLOCK);
  return keys <= GROUP_KEYS && reservations <= std::max<uint64_t>(1u << 21, items / 16);
}

// Keys of the items: counts[key] per key (zero before, GROUP_KEYS of them),
// then offsets[key] in the grouped order, offsets[keys] = items (GROUP_KEYS +
// 4 of them)
struct GroupKeys {
  uint32_t *counts, *offsets;
  uint32_t keys;
};
// device memory of two groupings
constexpr size_t GROUP_BYTES = 2 * (2 * GROUP_KEYS + 4) * sizeof(uint32_t);

// The key of a logged record
struct LogKeyOf {
  const uint32_t* key;
  __device__ uint32_t operator()(uint32_t i) const { return key[i]; }
};

// The items of a log lie in segments of cap places (blockIdx.y), of which
// those below the segment's count n_ptr[s * LOG_LINE] are in use; without
// n_ptr they are 0 .. cap - 1. key[i] (if not null) and rank[i], its place
// among the items of its key
template <class KeyOf>
__global__ void __launch_bounds__(GROUP_THREADS)
k_group_rank(KeyOf key_of, const unsigned long long* n_ptr, uint32_t cap, GroupKeys g,
             uint32_t* __restrict__ key, uint32_t* __restrict__ rank) {
  __shared__ uint32_t hist[GROUP_KEYS];
  const uint32_t base = blockIdx.y * cap;
  const uint32_t used =
      n_ptr ? (uint32_t)min(n_ptr[blockIdx.y * LOG_LINE], (unsigned long long)cap) : cap;
  const uint32_t first = base + blockIdx.x * GROUP_BLOCK, n = base + used;
  if (first >= n) return;
  for (uint32_t k = threadIdx.x; k < g.keys; k += GROUP_THREADS) hist[k] = 0;
  __syncthreads();
  uint32_t ks[GROUP_PER], r[GROUP_PER];
#pragma unroll
  for (int j = 0; j < GROUP_PER; ++j) {
    const uint32_t i = first + j * GROUP_THREADS + threadIdx.x;
    ks[j] = r[j] = 0;
    if (i < n) {
      ks[j] = key_of(i);
      if (key) key[i] = ks[j];
      r[j] = atomicAdd(&hist[ks[j]], 1u);
    }
  }
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < g.keys; k += GROUP_THREADS) {
    const uint32_t c = hist[k];
    if (c) hist[k] = atomicAdd(g.counts + k, c);
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < GROUP_PER; ++j) {
    const uint32_t i = first + j * GROUP_THREADS + threadIdx.x;
    if (i < n) rank[i] = hist[ks[j]] + r[j];
  }
}

// One block. Also empties the counts for the next grouping and, of a log,
// the record counts of its segments (of which cap each were kept): kept takes
// the records grouped, C the reduction and the records that found their
// segment full.
__global__ void __launch_bounds__(GROUP_THREADS)
k_group_scan(GroupKeys g, unsigned long long* n_ptr, uint32_t segs, uint32_t cap, uint32_t* kept,
             Counters* C) {
  __shared__ uint32_t part[GROUP_THREADS];
  constexpr uint32_t per = GROUP_KEYS / GROUP_THREADS;
  const uint32_t tid = threadIdx.x;
  // counts past the last key are zero, so their offsets are the item count
  const bool mine = tid * per <= g.keys;
  uint4 c[per / 4];
  uint32_t sum = 0;
#pragma unroll
  for (uint32_t j = 0; j < per / 4; ++j) {
    c[j] = mine ? ((const uint4*)g.counts)[tid * (per / 4) + j] : make_uint4(0, 0, 0, 0);
    sum += c[j].x + c[j].y + c[j].z + c[j].w;
  }
  part[tid] = sum;
  __syncthreads();
  for (uint32_t off = 1; off < GROUP_THREADS; off <<= 1) {
    const uint32_t v = tid >= off ? part[tid - off] : 0u;
    __syncthreads();
    part[tid] += v;
    __syncthreads();
  }
  uint32_t run = part[tid] - sum;
  if (mine) {
#pragma unroll
    for (uint32_t j = 0; j < per / 4; ++j) {
      const uint4 v = c[j];
      ((uint4*)g.offsets)[tid * (per / 4) + j] =
          make_uint4(run, run + v.x, run + v.x + v.y, run + v.x + v.y + v.z);
      ((uint4*)g.counts)[tid * (per / 4) + j] = make_uint4(0, 0, 0, 0);
      run += v.x + v.y + v.z + v.w;
    }
  }
  if (tid == GROUP_THREADS - 1) g.offsets[GROUP_KEYS] = part[tid];
  if (tid < segs && n_ptr) {
    const unsigned long long n = n_ptr[tid * LOG_LINE];
    const uint32_t m = (uint32_t)min(n, (unsigned long long)cap);
    kept[tid] = m;
    n_ptr[tid * LOG_LINE] = 0;
    if (n > m) atomicAdd(&C->log_over, n - m);
  }
  if (tid == 0 && n_ptr && part[GROUP_THREADS - 1]) ++C->log_flushes;
}

__global__ void __launch_bounds__(256)
k_group_place(const uint32_t* __restrict__ key, const uint32_t* __restrict__ rank,
              const uint32_t* kept, uint32_t n, GroupKeys g, uint32_t* __restrict__ order) {
  const uint32_t j = blockIdx.x * 256u + threadIdx.x, i = blockIdx.y * n + j;
  if (j < (kept ? kept[blockIdx.y] : n)) order[g.offsets[key[i]] + rank[i]] = i;
}

// The keys and indices of a log's records side by side, for the radix sort:
// segment s (cap places, first[s + 1] - first[s] of them in use) from first[s]
struct LogSegments {
  uint32_t first[LOG_SEGS + 1];
};
__global__ void __launch_bounds__(256)
k_log_list(const uint32_t* __restrict__ log_key, uint32_t cap, LogSegments s,
           uint32_t* __restrict__ key, uint32_t* __restrict__ idx) {
  const uint32_t j = blockIdx.x * 256u + threadIdx.x, to = s.first[blockIdx.y] + j;
  if (to >= s.first[blockIdx.y + 1]) return;
  key[to] = log_key[blockIdx.y * cap + j];
  idx[to] = blockIdx.y * cap + j;
}

// First of the sorted keys skey[0 .. m) that is not below k: the wave probes
// 64 places at a time
__device__ __forceinline__ uint32_t wave_lower_bound(const uint32_t* __restrict__ skey, uint32_t m,
                                                     uint32_t k) {
  uint32_t lo = 0, hi = m;  // the answer is in [lo, hi]
  while (lo < hi) {
    const uint32_t step = (hi - lo + 63u) / 64u;
    const uint32_t i = lo + lane_id() * step;
    const uint32_t below = (uint32_t)__popcll(__ballot(i < hi && skey[i] < k));
    if (!below) return lo;
    const uint32_t last = lo + (below - 1u) * step;  // the last probe below k
    hi = min(last + step, hi);
    lo = last + 1u;
  }
  return lo;
}

// The per-primitive tally's sums over the grouped records: `shares` waves per
// key, each every shares-th 64 records of the key's (found in g.offsets, or
// in the m sorted keys skey). Every lane adds up x and x^2 of the 10 fields of
// its records; the wave's totals leave with one atomic per value. Bound by
// the gather of the records, which lie in the order the paths ended in.
__global__ void __launch_bounds__(256)
k_prim_reduce(GroupKeys g, const uint32_t* __restrict__ skey, const uint32_t* __restrict__ sidx,
              uint32_t m, const double* __restrict__ val, uint32_t shares, double* prim) {
  const uint32_t w = (blockIdx.x * 256u + threadIdx.x) / 64u;
  const uint32_t key = w / shares;
  if (key >= g.keys) return;
  const uint32_t lo = skey ? wave_lower_bound(skey, m, key) : g.offsets[key];
  const uint32_t hi = skey ? wave_lower_bound(skey, m, key + 1u) : g.offsets[key + 1u];
  const uint32_t first = lo + (w % shares) * 64u;
  if (first >= hi) return;
  double acc[20];
#pragma unroll
  for (int f = 0; f < 20; ++f) acc[f] = 0.0;
  for (uint32_t i = first + lane_id(); i < hi; i += shares * 64u) {
    double x[10];
    const double2* v = (const double2*)(val + (size_t)sidx[i] * 10u);
#pragma unroll
    for (int f = 0; f < 5; ++f) {
      const double2 t = v[f];
      x[2 * f] = t.x;
      x[2 * f + 1] = t.y;
    }
#pragma unroll
    for (int f = 0; f < 10; ++f) {
      acc[2 * f] += x[f];
      acc[2 * f + 1] += x[f] * x[f];
    }
  }
  add_totals<20>(acc, prim + (size_t)key * 20u);
}
