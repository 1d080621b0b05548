// CSR of a segment index: the stable order of the rows by segment (perm) and the run of every
// segment (off), for the operators that are called with a plain index array (the VJPs of the
// gather-cat and of the Fourier basis, the segment sums without a prepared CSR).
//
// An LSD radix sort of the row numbers by their clamped key min(index, num_segment), at most 8 bits
// per pass and ceil(log2(num_segment + 1) / 8) passes (one up to 255 segments, two up to 65 535).
// Nothing here depends on the order in which waves run: the counters hold integer counts, and a
// row's place is its digit's base plus its rank among the rows before it.
//   * up to kSmallRows rows: one workgroup per index sorts (key, row) pairs in LDS and searches
//     every segment's offset there: one launch (two above kSmallSegments segments: the search then has the chip);
//   * above: per pass a histogram launch and a scatter launch over at most 256 contiguous chunks (1 024 from 2^24 rows)
//     (each scatter workgroup sums the chunk histograms itself, so there is no scan launch), then
//     one search per segment over the sorted keys. Up to two indices share the launches.
// The same passes order the atoms along a Morton curve for the builders (fmd_nl_atom_order: 30-bit
// keys formed from the fractional coordinates in the first pass; four passes).
// Bound by launches and dependent loads, not by bytes (160 000 rows: 8 MB in all): the two CSRs of a
// gather-cat VJP at 160 000 rows, 10 000 segments are 5 launches (45 us) where torch's sort, bincount
// and cumsum were 44 (275 us). The flag of negative indices goes to host memory from the first kernel, behind an
// event of its own, so that the GPU does not idle between calls. What is left of such calls is host time, which
// differs by box and by where the autograd thread runs: that forward and VJP at F = 128 453-497 -> 130-190 us,
// the Fourier basis and its VJP at 107 520 triplets 440-511 -> 94-170, one edge block at 135 atoms (three CSRs)
// 679-751 -> 260-320.
#include "common.h"
#include "search.h"

namespace {

constexpr int kThreads = 256;               // multi-workgroup kernels: 4 waves
constexpr int kWaves = kThreads / FMD_WAVE;
constexpr int kDigits = 256;                // counters per pass (8 bits)
// Workgroups of a histogram / scatter launch: one per CU up to 2^24 rows, then four, whose latencies overlap (64
// million rows 7 510 -> 6 060 us, 256 million 35.3 -> 29.7 ms; every scatter workgroup reads all chunk histograms).
constexpr int64_t max_chunks(int64_t rows) { return rows < (int64_t(1) << 24) ? 256 : 1024; }
constexpr int kChunkRows = 1024;            // rows from which another chunk is added
constexpr int kGroups = 4;                  // rows per thread whose loads are issued together
constexpr int kSmallRows = 8192;
// The one workgroup searches 1 024 offsets in 0.7 us, another launch costs about 5: 1 000 rows in 3 000 000 segments
// 2 240 us in it.
constexpr int64_t kSmallSegments = 8192;
constexpr int kSmallThreads = 1024;
constexpr int kSmallWaves = kSmallThreads / FMD_WAVE;

struct Job {
  const void* index;
  int is64;
  int64_t stride;
  int32_t rows;
  int32_t nseg;
  int32_t* perm;
  int64_t* off;
  const float* frac;   // Morton keys of [rows, 3] fractional coordinates instead of an index (null: none)
  int32_t* negative;   // set to 1 if some index is negative (host memory the device can write)
  uint32_t* key[2];    // [rows] each
  int32_t* row[2];     // [rows] each
  uint32_t* hist;      // [chunks][kDigits]
  int chunks;
  int32_t chunk_rows;  // a multiple of kThreads
  int passes;
  int bits;            // of one pass
};

struct Jobs {
  Job j[2];
};

// 10 bits of v at every third position
__device__ __forceinline__ uint32_t spread3(uint32_t v) {
  v = (v | (v << 16)) & 0x030000FFu;
  v = (v | (v << 8)) & 0x0300F00Fu;
  v = (v | (v << 4)) & 0x030C30C3u;
  return (v | (v << 2)) & 0x09249249u;
}

__device__ __forceinline__ uint32_t morton_key(const float* f) {
  uint32_t code = 0;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float x = fminf(fmaxf(f[a], 0.f), 0.99999988f) * 1024.f;  // the largest float below 1
    code |= spread3((uint32_t)x & 1023u) << a;
  }
  return code;
}

// key of a row: its segment, or num_segment for an index outside [0, num_segment) (such rows follow
// every run and belong to none)
__device__ __forceinline__ uint32_t row_key(const Job& j, int64_t r, bool& neg) {
  if (j.frac) return morton_key(j.frac + 3 * r);
  const int64_t v = j.is64 ? static_cast<const int64_t*>(j.index)[r * j.stride]
                           : (int64_t)static_cast<const int32_t*>(j.index)[r * j.stride];
  neg = neg || v < 0;
  return v < 0 || v > j.nseg ? (uint32_t)j.nseg : (uint32_t)v;
}

// The flag is the caller's to read once the first launch has run: a store past the caches, to host
// memory, only from workgroups that saw a negative index.
__device__ __forceinline__ void flag_negative(const Job& j) {
  __hip_atomic_store(j.negative, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// the lanes of the wave (among `active`) whose digit is this lane's
__device__ __forceinline__ uint64_t same_digit(uint32_t digit, int bits, uint64_t active) {
  uint64_t m = active;
  for (int b = 0; b < bits; ++b) {
    const bool one = (digit >> b) & 1;
    const uint64_t v = __ballot(one);
    m &= one ? v : ~v;
  }
  return m;
}

__global__ void __launch_bounds__(kThreads) csr_hist_kernel(const Jobs jobs, int pass) {
  const Job& j = jobs.j[blockIdx.y];
  if (pass >= j.passes || (int)blockIdx.x >= j.chunks) return;
  __shared__ uint32_t s_hist[kDigits];
  const int t = threadIdx.x;
  s_hist[t] = 0;
  __syncthreads();
  const int shift = pass * j.bits;
  const uint32_t mask = (1u << j.bits) - 1;
  const int64_t lo = (int64_t)blockIdx.x * j.chunk_rows;
  const int64_t hi = lo + j.chunk_rows < j.rows ? lo + j.chunk_rows : j.rows;
  bool neg = false;
  for (int64_t r0 = lo + t; r0 < hi; r0 += (int64_t)kThreads * kGroups) {
    uint32_t key[kGroups];
#pragma unroll
    for (int g = 0; g < kGroups; ++g) {
      const int64_t r = r0 + g * kThreads;
      key[g] = r >= hi ? 0 : pass == 0 ? row_key(j, r, neg) : j.key[(pass - 1) & 1][r];
    }
#pragma unroll
    for (int g = 0; g < kGroups; ++g)
      if (r0 + g * kThreads < hi) atomicAdd(&s_hist[(key[g] >> shift) & mask], 1u);
  }
  if (neg) flag_negative(j);
  __syncthreads();
  j.hist[(int64_t)blockIdx.x * kDigits + t] = s_hist[t];
}

// Scatter of one chunk: the digit bases from the chunk histograms (thread d: digit d), the waves'
// own bases (a wave owns a contiguous quarter of the chunk), then 64 rows at a time in row order.
__global__ void __launch_bounds__(kThreads) csr_scatter_kernel(const Jobs jobs, int pass) {
  const Job& j = jobs.j[blockIdx.y];
  if (pass >= j.passes || (int)blockIdx.x >= j.chunks) return;
  __shared__ uint32_t s_base[kWaves][kDigits];
  __shared__ uint32_t s_scan[17];
  const int t = threadIdx.x, lane = t & (FMD_WAVE - 1), wave = t / FMD_WAVE;
  const int shift = pass * j.bits;
  const uint32_t mask = (1u << j.bits) - 1;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) s_base[w][t] = 0;
  __syncthreads();
  const int32_t wave_rows = j.chunk_rows / kWaves;  // a multiple of 64
  const int64_t lo = (int64_t)blockIdx.x * j.chunk_rows + (int64_t)wave * wave_rows;
  const int64_t end = lo + wave_rows < j.rows ? lo + wave_rows : j.rows;
  bool neg = false;
  auto key_of = [&](int64_t r) { return pass == 0 ? row_key(j, r, neg) : j.key[(pass - 1) & 1][r]; };
  for (int64_t r0 = lo + lane; r0 < end; r0 += FMD_WAVE * kGroups) {
    uint32_t key[kGroups];
#pragma unroll
    for (int g = 0; g < kGroups; ++g) key[g] = r0 + g * FMD_WAVE < end ? key_of(r0 + g * FMD_WAVE) : 0;
#pragma unroll
    for (int g = 0; g < kGroups; ++g)
      if (r0 + g * FMD_WAVE < end) atomicAdd(&s_base[wave][(key[g] >> shift) & mask], 1u);
  }
  uint32_t before = 0, total = 0;
  // histogram rows in flight per thread (8 left 20 dependent round trips at 160 000 rows)
  constexpr int kLoads = 32;
  for (int c0 = 0; c0 < j.chunks; c0 += kLoads) {
    uint32_t v[kLoads];
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {  // clamped, not predicated: no branch between the loads
      const int c = c0 + u < j.chunks ? c0 + u : j.chunks - 1;
      v[u] = j.hist[c * kDigits + t];
    }
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      total += c0 + u < j.chunks ? v[u] : 0;
      before += c0 + u < (int)blockIdx.x ? v[u] : 0;
    }
  }
  uint32_t all;
  uint32_t run = block_exclusive_scan<uint32_t>(total, s_scan, &all) + before;  // its barriers order s_base
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    const uint32_t c = s_base[w][t];
    s_base[w][t] = run;
    run += c;
  }
  __syncthreads();
  volatile uint32_t* base = s_base[wave];  // read and written by this wave alone from here on
  const bool last = pass == j.passes - 1;
  uint32_t* key_out = j.key[pass & 1];
  int32_t* row_out = last ? j.perm : j.row[pass & 1];
  for (int64_t r0 = lo + lane; r0 - lane < end; r0 += FMD_WAVE * kGroups) {
    uint32_t key[kGroups];
    int32_t row[kGroups];
#pragma unroll
    for (int g = 0; g < kGroups; ++g) {
      const int64_t r = r0 + g * FMD_WAVE;
      key[g] = r < end ? key_of(r) : 0;
      row[g] = r >= end || pass == 0 ? (int32_t)r : j.row[(pass - 1) & 1][r];
    }
#pragma unroll
    for (int g = 0; g < kGroups; ++g) {
      const bool in = r0 + g * FMD_WAVE < end;
      const uint32_t digit = (key[g] >> shift) & mask;
      const uint64_t same = same_digit(digit, j.bits, __ballot(in));
      const int rank = lane_prefix(same);
      const uint32_t first = base[digit];
      if (in) {
        key_out[first + rank] = key[g];
        row_out[first + rank] = row[g];
        if (rank == 0) base[digit] = first + (uint32_t)__popcll(same);
      }
    }
  }
}

// off[s] = rows with a key below s
__global__ void __launch_bounds__(kThreads) csr_offsets_kernel(const Jobs jobs) {
  const Job& j = jobs.j[blockIdx.y];
  const int64_t s = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (s <= j.nseg) j.off[s] = lower_bound(j.key[(j.passes - 1) & 1], j.rows, (uint32_t)s);
}

// One workgroup per index: the same passes on (key, row) pairs in LDS.
__global__ void __launch_bounds__(kSmallThreads) csr_small_kernel(const Jobs jobs) {
  const Job& j = jobs.j[blockIdx.y];
  __shared__ uint32_t s_key[2][kSmallRows];
  __shared__ uint16_t s_row[2][kSmallRows];
  __shared__ uint32_t s_base[kSmallWaves][kDigits];
  __shared__ uint32_t s_scan[17];
  const int t = threadIdx.x, lane = t & (FMD_WAVE - 1), wave = t / FMD_WAVE;
  const int rows = j.rows;
  bool neg = false;
  for (int r = t; r < rows; r += kSmallThreads) {
    s_key[0][r] = row_key(j, r, neg);
    s_row[0][r] = (uint16_t)r;
  }
  if (neg) flag_negative(j);
  // a wave's contiguous share, in groups of 64 rows
  const int wave_rows = (int)fmd_cdiv(rows, kSmallThreads) * FMD_WAVE;
  const int lo = wave * wave_rows, end = lo + wave_rows < rows ? lo + wave_rows : rows;
  const uint32_t mask = (1u << j.bits) - 1;
  for (int pass = 0; pass < j.passes; ++pass) {
    const int shift = pass * j.bits, src = pass & 1, dst = src ^ 1;
    for (int q = t; q < kSmallWaves * kDigits; q += kSmallThreads) (&s_base[0][0])[q] = 0;
    __syncthreads();  // also: the pairs of the previous pass are written
    for (int r = lo + lane; r < end; r += FMD_WAVE) atomicAdd(&s_base[wave][(s_key[src][r] >> shift) & mask], 1u);
    __syncthreads();
    uint32_t total = 0, all;
    if (t < kDigits)
      for (int w = 0; w < kSmallWaves; ++w) total += s_base[w][t];
    uint32_t run = block_exclusive_scan<uint32_t>(total, s_scan, &all);
    if (t < kDigits)
      for (int w = 0; w < kSmallWaves; ++w) {
        const uint32_t c = s_base[w][t];
        s_base[w][t] = run;
        run += c;
      }
    __syncthreads();
    volatile uint32_t* base = s_base[wave];
    for (int r0 = lo; r0 < end; r0 += FMD_WAVE) {
      const int r = r0 + lane;
      const bool in = r < end;
      const uint32_t key = in ? s_key[src][r] : 0;
      const uint32_t digit = (key >> shift) & mask;
      const uint64_t same = same_digit(digit, j.bits, __ballot(in));
      const int rank = lane_prefix(same);
      const uint32_t first = base[digit];
      if (in) {
        s_key[dst][first + rank] = key;
        s_row[dst][first + rank] = s_row[src][r];
        if (rank == 0) base[digit] = first + (uint32_t)__popcll(same);
      }
    }
    __syncthreads();
  }
  const int fin = j.passes & 1;
  for (int r = t; r < rows; r += kSmallThreads) {
    j.perm[r] = s_row[fin][r];
    if (j.key[0]) j.key[0][r] = s_key[fin][r];  // csr_offsets_kernel follows
  }
  if (j.off && !j.key[0])
    for (int64_t s = t; s <= j.nseg; s += kSmallThreads) j.off[s] = lower_bound(s_key[fin], rows, (uint32_t)s);
}

// The chunks of a job above kSmallRows and its buffers in `work`.
void job_chunks(Job& j, uint32_t* work) {
  const int64_t n = j.rows;
  int64_t c = fmd_cdiv(n, kChunkRows);
  c = c < 1 ? 1 : (c > max_chunks(n) ? max_chunks(n) : c);
  const int64_t per = fmd_cdiv(fmd_cdiv(n, c), kThreads) * kThreads;
  j.chunk_rows = (int32_t)(per < kThreads ? kThreads : per);
  j.chunks = (int)fmd_cdiv(n, j.chunk_rows);
  j.chunks = j.chunks < 1 ? 1 : j.chunks;
  j.key[0] = work;
  j.key[1] = work + n;
  j.row[0] = reinterpret_cast<int32_t*>(work + 2 * n);
  j.row[1] = reinterpret_cast<int32_t*>(work + 3 * n);
  j.hist = work + 4 * n;
}

}  // namespace

extern "C" {

int64_t fmd_csr_work_size(int64_t rows) {
  return 4 * (rows > 0 ? rows : 0) + max_chunks(rows) * kDigits;
}

int fmd_csr_from_index(int32_t count, const void* const* index, const int32_t* is64, const int64_t* stride,
                       const int64_t* rows, const int64_t* num_segment, int32_t* const* perm, int64_t* const* off,
                       uint32_t* const* work, int32_t* negative, hipEvent_t checked, hipStream_t stream) {
  FMD_REQUIRE(count >= 1 && count <= 2 && index && is64 && stride && rows && num_segment && perm && off && work);
  FMD_REQUIRE(negative);
  Jobs jobs{};
  bool small = true;
  int chunks = 1, passes = 1;
  int64_t nseg = 0;
  for (int q = 0; q < count; ++q) {
    FMD_REQUIRE(rows[q] >= 0 && rows[q] < (int64_t(1) << 31) - 1 && num_segment[q] >= 0);
    FMD_REQUIRE(num_segment[q] < (int64_t(1) << 31) - 1 && off[q] && (rows[q] == 0 || (index[q] && perm[q])));
    Job& j = jobs.j[q];
    j.index = index[q];
    j.is64 = is64[q];
    j.stride = stride[q];
    j.rows = (int32_t)rows[q];
    j.nseg = (int32_t)num_segment[q];
    j.perm = perm[q];
    j.off = off[q];
    j.negative = negative + q;
    int width = 1;  // of the largest key, num_segment
    while (width < 32 && (num_segment[q] >> width) != 0) ++width;
    j.passes = (width + 7) / 8;
    j.bits = (width + j.passes - 1) / j.passes;
    small = small && rows[q] <= kSmallRows;
    passes = j.passes > passes ? j.passes : passes;
    nseg = num_segment[q] > nseg ? num_segment[q] : nseg;
  }
  if (small) {
    const bool search = nseg > kSmallSegments && work[0] && work[count - 1];
    for (int q = 0; search && q < count; ++q) jobs.j[q].key[0] = jobs.j[q].key[1] = work[q];
    hipLaunchKernelGGL(csr_small_kernel, dim3(1, (unsigned)count), dim3(kSmallThreads), 0, stream, jobs);
    FMD_CHECK_LAUNCH();
    if (checked) {
      const hipError_t err = hipEventRecord(checked, stream);
      if (err != hipSuccess) return (int)err;
    }
    if (search) {
      hipLaunchKernelGGL(csr_offsets_kernel, dim3((unsigned)fmd_cdiv(nseg + 1, kThreads), (unsigned)count),
                         dim3(kThreads), 0, stream, jobs);
      FMD_CHECK_LAUNCH();
    }
    return FMD_OK;
  }
  for (int q = 0; q < count; ++q) {
    FMD_REQUIRE(work[q]);
    job_chunks(jobs.j[q], work[q]);
    chunks = jobs.j[q].chunks > chunks ? jobs.j[q].chunks : chunks;
  }
  for (int p = 0; p < passes; ++p) {
    hipLaunchKernelGGL(csr_hist_kernel, dim3((unsigned)chunks, (unsigned)count), dim3(kThreads), 0, stream, jobs, p);
    FMD_CHECK_LAUNCH();
    if (p == 0 && checked) {  // every index has been read
      const hipError_t err = hipEventRecord(checked, stream);
      if (err != hipSuccess) return (int)err;
    }
    hipLaunchKernelGGL(csr_scatter_kernel, dim3((unsigned)chunks, (unsigned)count), dim3(kThreads), 0, stream, jobs, p);
    FMD_CHECK_LAUNCH();
  }
  hipLaunchKernelGGL(csr_offsets_kernel, dim3((unsigned)fmd_cdiv(nseg + 1, kThreads), (unsigned)count), dim3(kThreads),
                     0, stream, jobs);
  FMD_CHECK_LAUNCH();
  return FMD_OK;
}

int fmd_nl_atom_order(const float* frac, int64_t n_atoms, uint32_t* work, int32_t* order, hipStream_t stream) {
  FMD_REQUIRE(n_atoms > 0 && n_atoms < (int64_t(1) << 31) - 1 && frac && work && order);
  Jobs jobs{};
  Job& j = jobs.j[0];
  j.frac = frac;
  j.rows = (int32_t)n_atoms;
  j.perm = order;
  j.passes = 4;
  j.bits = 8;
  if (n_atoms <= kSmallRows) {
    hipLaunchKernelGGL(csr_small_kernel, dim3(1, 1), dim3(kSmallThreads), 0, stream, jobs);
    FMD_CHECK_LAUNCH();
    return FMD_OK;
  }
  job_chunks(j, work);
  for (int p = 0; p < j.passes; ++p) {
    hipLaunchKernelGGL(csr_hist_kernel, dim3((unsigned)j.chunks, 1), dim3(kThreads), 0, stream, jobs, p);
    FMD_CHECK_LAUNCH();
    hipLaunchKernelGGL(csr_scatter_kernel, dim3((unsigned)j.chunks, 1), dim3(kThreads), 0, stream, jobs, p);
    FMD_CHECK_LAUNCH();
  }
  return FMD_OK;
}

}  // extern "C"
