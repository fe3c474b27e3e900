// Scatter-assembly on the device: element matrices -> global CSR.
//
// Reference behaviour (luiswirth/formoniq, crates/):
//   assemble_matrix       formoniq/src/galerkin.rs:138-188 (push v if v != 0.0,
//                         triplets in cell order, COO -> CSR sums duplicates)
//   relative assembly     formoniq/src/whitney_complex.rs:620-624 (E^T A E)
//   hdif_gram             formoniq/src/whitney_complex.rs:180-183 (CSR add)
//   HodgeDirac op         formoniq/src/problems/dirac.rs:242-250 (CSR x CSR)
//
// Every sparse build here is one primitive, the CooPlan: (row, col) keys of
// all contributions are radix-sorted once (stable, so contributions to one
// entry stay in input order, which is cell order for assembly), run heads give
// the CSR entries, and `src` keeps, per entry, the indices of its
// contributors. A value pass is then a deterministic segmented sum over `src`
// with no atomics, so the bits do not depend on scheduling, and re-assembling
// new geometry on a fixed mesh is that pass alone. Bit 31 of a src index
// negates the contribution (the sign flip of the sigma rows of the KKT system).
#include <cstring>
#include <rocprim/rocprim.hpp>

#include <algorithm>
#include <vector>

#include "feec_internal.hpp"

namespace feec {

namespace {

constexpr int TPB = 256;
constexpr uint32_t NEG = kCooNegate;

inline unsigned grid_for(int64_t n) { return (unsigned)std::max<int64_t>(1, (n + TPB - 1) / TPB); }

// Sort keys row * ncols + col (sentinel for dropped contributions) and the
// number of valid ones. Grid-stride with a bounded grid and one atomic per
// block: an atomic per wavefront on the one counter serialized (22 ms for the
// 201 M contributions of a 64^3 KKT system).
constexpr unsigned KEYS_MAX_BLOCKS = 2048;
__global__ void __launch_bounds__(TPB) k_keys(const int32_t* rows, const int32_t* cols, int64_t n,
                                              int64_t ncols, uint64_t sentinel, uint64_t* keys,
                                              unsigned long long* nvalid) {
  __shared__ unsigned long long sh[TPB / 64];
  unsigned long long cnt = 0;  // valid keys of the wavefront, on lane 0
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int32_t r = rows[i], c = cols[i];
    const bool ok = r >= 0 && c >= 0;
    keys[i] = ok ? (uint64_t)r * (uint64_t)ncols + (uint64_t)c : sentinel;
    // lane 0 is active whenever any lane of its wavefront is
    cnt += (unsigned long long)__popcll(__ballot(ok));
  }
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = cnt;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long t = 0;
    for (unsigned w = 0; w < blockDim.x / 64; ++w) t += sh[w];
    if (t) atomicAdd(nvalid, t);
  }
}

__global__ void k_heads(const uint64_t* keys, int64_t n, int32_t* head) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) head[i] = (i == 0 || keys[i] != keys[i - 1]) ? 1 : 0;
}

__global__ void k_entries(const uint64_t* keys, const int32_t* head, const int32_t* scan, int64_t n,
                          int64_t ncols, int64_t* seg, int32_t* col) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= n || !head[i]) return;
  int64_t e = scan[i] - 1;
  seg[e] = i;
  col[e] = (int32_t)(keys[i] % (uint64_t)ncols);
}

// row_ptr from the sorted entries: entry e (or the end, e = nnz) starts every
// row after the previous entry's row up to its own, so each of the nrows + 1
// pointers is written once (empty rows included), without counting atomics.
__global__ void k_row_starts(const uint64_t* keys, const int64_t* seg, int64_t nnz, int64_t ncols,
                             int64_t nrows, int64_t* row_ptr) {
  const int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (e > nnz) return;
  const int64_t prev = e == 0 ? -1 : (int64_t)(keys[seg[e - 1]] / (uint64_t)ncols);
  const int64_t cur = e == nnz ? nrows : (int64_t)(keys[seg[e]] / (uint64_t)ncols);
  for (int64_t r = prev + 1; r <= cur; ++r) row_ptr[r] = e;
}

template <class T>
void exclusive_scan_u64_to_i64(Ctx* ctx, const unsigned long long* in, int64_t* out, int64_t n) {
  size_t bytes = 0;
  FEEC_HIP(rocprim::exclusive_scan(nullptr, bytes, in, out, (int64_t)0, (size_t)n,
                                   rocprim::plus<int64_t>(), ctx->stream));
  void* tmp = ctx->ensure_temp(bytes);
  FEEC_HIP(rocprim::exclusive_scan(tmp, bytes, in, out, (int64_t)0, (size_t)n,
                                   rocprim::plus<int64_t>(), ctx->stream));
}

void inclusive_scan_i32(Ctx* ctx, const int32_t* in, int32_t* out, int64_t n) {
  size_t bytes = 0;
  FEEC_HIP(rocprim::inclusive_scan(nullptr, bytes, in, out, (size_t)n, rocprim::plus<int32_t>(),
                                   ctx->stream));
  void* tmp = ctx->ensure_temp(bytes);
  FEEC_HIP(rocprim::inclusive_scan(tmp, bytes, in, out, (size_t)n, rocprim::plus<int32_t>(),
                                   ctx->stream));
}

// One thread per CSR entry: sum contributors in order; keep = some contributor != 0.
__global__ void k_segsum(const int64_t* seg, const uint32_t* src, int64_t nnz, const double* vals,
                         double* out, uint8_t* keep, unsigned long long* ndropped) {
  int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (e >= nnz) return;
  int64_t b = seg[e], en = seg[e + 1];
  double acc = 0.0;
  bool nz = false;
  for (int64_t s = b; s < en; ++s) {
    uint32_t j = src[s];
    double v = vals[j & ~NEG];
    if (j & NEG) v = -v;
    nz |= (v != 0.0);
    acc = (s == b) ? v : acc + v;
  }
  out[e] = acc;
  if (keep) {
    keep[e] = nz ? 1 : 0;
    if (!nz) atomicAdd(ndropped, 1ull);
  }
}

// The same sums with the gathers shared by the wavefront: each wavefront
// takes 64 consecutive entries, whose contributions are contiguous in src;
// its lanes fetch all of them together (every lane busy, 64 gathers in
// flight) into LDS, then each lane adds its own entry's values in order, so
// every sum is the one k_segsum forms. A run longer than the LDS stage falls
// back to the per-lane gathers.
// XCD_CHUNK > 0: blocks are dealt to the 8 XCDs round-robin; the grid (a
// multiple of 8 * XCD_CHUNK) is renumbered so that each XCD takes runs of
// XCD_CHUNK consecutive blocks spread over the whole range, so that an
// element value's nearby readers share that XCD's L2.
// STAGE: contributions staged per wavefront (a smaller stage leaves room for
// more resident wavefronts; runs longer than it take the per-lane gathers).
template <int XCD_CHUNK, int STAGE>
__global__ void __launch_bounds__(TPB) k_segsum_wave(const int64_t* seg, const uint32_t* src, int64_t nnz,
                                                     const double* vals, double* out, uint8_t* keep,
                                                     unsigned long long* ndropped) {
  __shared__ double sv[TPB / 64][STAGE];
  const int w = threadIdx.x / 64, lane = threadIdx.x % 64;
  int64_t blk = blockIdx.x;
  if (XCD_CHUNK > 0) {
    const int64_t x = blockIdx.x % 8, k = blockIdx.x / 8;
    blk = ((k / XCD_CHUNK) * 8 + x) * XCD_CHUNK + k % XCD_CHUNK;
  }
  const int64_t e0 = (blk * (TPB / 64) + w) * 64;
  const bool active = e0 < nnz;
  const int64_t e1 = active ? (e0 + 64 < nnz ? e0 + 64 : nnz) : e0;
  const int64_t s0 = active ? seg[e0] : 0, s1 = active ? seg[e1] : 0;
  const bool staged = active && s1 - s0 <= STAGE;
  if (staged)
    for (int64_t q = s0 + lane; q < s1; q += 64) {
      const uint32_t j = src[q];
      const double v = vals[j & ~NEG];
      sv[w][q - s0] = (j & NEG) ? -v : v;
    }
  __syncthreads();
  const int64_t e = e0 + lane;
  if (!active || e >= e1) return;
  const int64_t b = seg[e], en = seg[e + 1];
  double acc = 0.0;
  bool nz = false;
  for (int64_t q = b; q < en; ++q) {
    double v;
    if (staged) {
      v = sv[w][q - s0];
    } else {
      const uint32_t j = src[q];
      v = vals[j & ~NEG];
      if (j & NEG) v = -v;
    }
    nz |= (v != 0.0);
    acc = (q == b) ? v : acc + v;
  }
  out[e] = acc;
  if (keep) {
    keep[e] = nz ? 1 : 0;
    if (!nz) atomicAdd(ndropped, 1ull);
  }
}

__global__ void k_rows_of(const int64_t* row_ptr, int64_t nrows, int32_t* rows) {
  int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (r >= nrows) return;
  for (int64_t p = row_ptr[r]; p < row_ptr[r + 1]; ++p) rows[p] = (int32_t)r;
}

// Compaction of a pattern to its kept entries. Entry p moves to newpos[p]
// (the exclusive scan of keep), one lane per entry so loads and stores run in
// entry order; a row starts at the new position of its first old entry, or at
// the end when it has none left in the old array.
__global__ void k_compact_entries(const int32_t* col, const double* val, const uint8_t* keep,
                                  const int64_t* newpos, int64_t n, int32_t* ocol, double* oval) {
  int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (p < n && keep[p]) {
    ocol[newpos[p]] = col[p];
    oval[newpos[p]] = val[p];
  }
}
__global__ void k_compact_rows(const int64_t* row_ptr, int64_t nrows, const int64_t* newpos,
                               int64_t n, int64_t nnz_kept, int64_t* orow) {
  int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (r > nrows) return;
  const int64_t p = row_ptr[r];
  orow[r] = p < n ? newpos[p] : nnz_kept;
}

__global__ void k_u8_to_u64(const uint8_t* a, int64_t n, unsigned long long* b) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) b[i] = a[i];
}

__global__ void k_set_last(int64_t* a, int64_t idx, int64_t v) { a[idx] = v; }

template <class T>
__global__ void k_copy_scale(const T* a, int64_t n, double s, T* b) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) b[i] = a[i];
}

__global__ void k_diag(const int64_t* row_ptr, const int32_t* col, const double* val, int64_t n,
                       double* diag) {
  int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (r >= n) return;
  double d = 0.0;
  for (int64_t p = row_ptr[r]; p < row_ptr[r + 1]; ++p)
    if (col[p] == r) d = val[p];
  diag[r] = d;
}

}  // namespace

void require_entries(int64_t total) {
  FEEC_REQUIRE(total < (int64_t(1) << 31), FEEC_E_ARG, "too many contributions for one matrix");
}

void coo_plan_build(Ctx* ctx, CooPlan& plan, int64_t nrows, int64_t ncols, int64_t n,
                    const int32_t* rows, const int32_t* cols, const uint32_t* srcs) {
  plan.nrows = nrows;
  plan.ncols = ncols;
  FEEC_REQUIRE(nrows >= 0 && ncols >= 0, FEEC_E_ARG, "negative matrix shape");
  const uint64_t sentinel = (uint64_t)nrows * (uint64_t)std::max<int64_t>(ncols, 1);
  int end_bit = 1;
  while (end_bit < 64 && (uint64_t(1) << end_bit) <= sentinel) ++end_bit;
  plan.row_ptr.alloc(ctx, nrows + 1);
  if (n == 0 || nrows == 0 || ncols == 0) {
    FEEC_HIP(hipMemsetAsync(plan.row_ptr.p, 0, (nrows + 1) * sizeof(int64_t), ctx->stream));
    plan.nnz = 0;
    plan.col.alloc(ctx, 0);
    plan.seg.alloc(ctx, 1);
    FEEC_HIP(hipMemsetAsync(plan.seg.p, 0, sizeof(int64_t), ctx->stream));
    plan.src.alloc(ctx, 0);
    ctx->sync();
    return;
  }
  DBuf<uint64_t> k0(ctx, n), k1(ctx, n);
  DBuf<unsigned long long> nvalid(ctx, 1);
  FEEC_HIP(hipMemsetAsync(nvalid.p, 0, sizeof(unsigned long long), ctx->stream));
  k_keys<<<std::min(grid_for(n), KEYS_MAX_BLOCKS), TPB, 0, ctx->stream>>>(
      rows, cols, n, std::max<int64_t>(ncols, 1), sentinel, k0.p, nvalid.p);
  DBuf<uint32_t> s0(ctx, n);
  FEEC_HIP(hipMemcpyAsync(s0.p, srcs, n * sizeof(uint32_t), hipMemcpyDeviceToDevice, ctx->stream));
  plan.src.alloc(ctx, n);
  {
    size_t bytes = 0;
    FEEC_HIP(rocprim::radix_sort_pairs(nullptr, bytes, k0.p, k1.p, s0.p, plan.src.p, (size_t)n, 0,
                                       (unsigned)end_bit, ctx->stream));
    void* tmp = ctx->ensure_temp(bytes);
    FEEC_HIP(rocprim::radix_sort_pairs(tmp, bytes, k0.p, k1.p, s0.p, plan.src.p, (size_t)n, 0,
                                       (unsigned)end_bit, ctx->stream));
  }
  k0.reset();
  s0.reset();
  unsigned long long hv = 0;
  FEEC_HIP(hipMemcpyAsync(&hv, nvalid.p, sizeof(hv), hipMemcpyDeviceToHost, ctx->stream));
  ctx->sync();
  int64_t nv = (int64_t)hv;
  require_entries(nv);
  DBuf<int32_t> head(ctx, std::max<int64_t>(nv, 1)), scan(ctx, std::max<int64_t>(nv, 1));
  int64_t nnz = 0;
  if (nv > 0) {
    k_heads<<<grid_for(nv), TPB, 0, ctx->stream>>>(k1.p, nv, head.p);
    inclusive_scan_i32(ctx, head.p, scan.p, nv);
    int32_t last = 0;
    FEEC_HIP(hipMemcpyAsync(&last, scan.p + nv - 1, sizeof(int32_t), hipMemcpyDeviceToHost,
                            ctx->stream));
    ctx->sync();
    nnz = last;
  }
  plan.nnz = nnz;
  plan.seg.alloc(ctx, nnz + 1);
  plan.col.alloc(ctx, nnz);
  if (nv > 0)
    k_entries<<<grid_for(nv), TPB, 0, ctx->stream>>>(k1.p, head.p, scan.p, nv,
                                                     std::max<int64_t>(ncols, 1), plan.seg.p,
                                                     plan.col.p);
  k_set_last<<<1, 1, 0, ctx->stream>>>(plan.seg.p, nnz, nv);
  k_row_starts<<<grid_for(nnz + 1), TPB, 0, ctx->stream>>>(k1.p, plan.seg.p, nnz, std::max<int64_t>(ncols, 1),
                                                           nrows, plan.row_ptr.p);
  FEEC_HIP(hipGetLastError());
  ctx->sync();
}

int64_t coo_plan_values(Ctx* ctx, const CooPlan& plan, const double* vals, double* out,
                        uint8_t* keep) {
  if (plan.nnz == 0) return 0;
  unsigned long long* nd = ctx->dcount;
  // per-lane gathers, or the wavefront's shared ones in XCD runs with a stage
  // of 512 or 1,024 contributions: the same sums, bit for bit. Below 2^22 entries the per-lane gathers were the fastest at every
  // size measured, so only larger plans are timed.
  const bool timed = plan.nnz >= (int64_t(1) << 22);
  tune_run(ctx, "segsum", 0, 0, plan.nnz, 3, [&](int c) {
    if (keep) FEEC_HIP(hipMemsetAsync(nd, 0, sizeof(unsigned long long), ctx->stream));
    const unsigned g = grid_for(plan.nnz);
    constexpr int C = 128;
    const unsigned gx = (g + 8 * C - 1) / (8 * C) * (8 * C);
    if (c == 0)
      k_segsum<<<g, TPB, 0, ctx->stream>>>(plan.seg.p, plan.src.p, plan.nnz, vals, out, keep, nd);
    else if (c == 1)  // about 2-3 contributions per entry (the KKT)
      k_segsum_wave<C, 512><<<gx, TPB, 0, ctx->stream>>>(plan.seg.p, plan.src.p, plan.nnz, vals, out, keep, nd);
    else  // about 5 (mass plus stiffness: the preconditioner matrix)
      k_segsum_wave<C, 1024><<<gx, TPB, 0, ctx->stream>>>(plan.seg.p, plan.src.p, plan.nnz, vals, out, keep, nd);
    FEEC_HIP(hipGetLastError());
  }, timed);
  if (!keep) return 0;
  unsigned long long h = 0;
  FEEC_HIP(hipMemcpyAsync(&h, nd, sizeof(h), hipMemcpyDeviceToHost, ctx->stream));
  ctx->sync();
  return (int64_t)h;
}

void coo_plan_apply(Ctx* ctx, const CooPlan& plan, const double* vals, bool zero_drop, Csr& out) {
  out.ctx = ctx;
  out.nrows = plan.nrows;
  out.ncols = plan.ncols;
  DBuf<double> v(ctx, plan.nnz);
  DBuf<uint8_t> keep;
  if (zero_drop) keep.alloc(ctx, plan.nnz);
  int64_t dropped = coo_plan_values(ctx, plan, vals, v.p, zero_drop ? keep.p : nullptr);
  if (dropped == 0) {
    out.nnz = plan.nnz;
    out.row_ptr.alloc(ctx, plan.nrows + 1);
    out.col.alloc(ctx, plan.nnz);
    FEEC_HIP(hipMemcpyAsync(out.row_ptr.p, plan.row_ptr.p, (plan.nrows + 1) * sizeof(int64_t),
                            hipMemcpyDeviceToDevice, ctx->stream));
    FEEC_HIP(hipMemcpyAsync(out.col.p, plan.col.p, plan.nnz * sizeof(int32_t),
                            hipMemcpyDeviceToDevice, ctx->stream));
    out.val = std::move(v);
    ctx->sync();
    return;
  }
  // Entries whose contributions were all exactly zero were never pushed by
  // the reference: compact them away.
  int64_t nnz = plan.nnz - dropped;
  DBuf<unsigned long long> k64(ctx, plan.nnz);
  k_u8_to_u64<<<grid_for(plan.nnz), TPB, 0, ctx->stream>>>(keep.p, plan.nnz, k64.p);
  DBuf<int64_t> pos(ctx, plan.nnz);
  exclusive_scan_u64_to_i64<int64_t>(ctx, k64.p, pos.p, plan.nnz);
  out.nnz = nnz;
  out.col.alloc(ctx, nnz);
  out.val.alloc(ctx, nnz);
  out.row_ptr.alloc(ctx, plan.nrows + 1);
  k_compact_entries<<<grid_for(plan.nnz), TPB, 0, ctx->stream>>>(plan.col.p, v.p, keep.p, pos.p,
                                                                 plan.nnz, out.col.p, out.val.p);
  k_compact_rows<<<grid_for(plan.nrows + 1), TPB, 0, ctx->stream>>>(
      plan.row_ptr.p, plan.nrows, pos.p, plan.nnz, nnz, out.row_ptr.p);
  FEEC_HIP(hipGetLastError());
  ctx->sync();
}

// ---------------------------------------------------------------------------
// sparse utilities
// ---------------------------------------------------------------------------
namespace {

__global__ void k_iota_u32(uint32_t* a, int64_t n, uint32_t base) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) a[i] = base + (uint32_t)i;
}

// ROW_LANES lanes share a row in the expansions below, so that a wavefront's
// stores fall on a few runs (one lane a row: 283 us for 7.4 M entries).
constexpr int ROW_LANES = 8;
inline unsigned row_grid(int64_t rows) { return grid_for(rows * ROW_LANES); }

__global__ void k_block_coo(const int64_t* row_ptr, const int32_t* col, int64_t nrows,
                            int64_t roff, int64_t coff, bool transpose, uint32_t src_base,
                            bool negate, int32_t* orow, int32_t* ocol, uint32_t* osrc) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, r = t / ROW_LANES;
  if (r >= nrows) return;
  const int64_t end = row_ptr[r + 1];
  for (int64_t p = row_ptr[r] + t % ROW_LANES; p < end; p += ROW_LANES) {
    int32_t a = (int32_t)r, b = col[p];
    orow[p] = (int32_t)((transpose ? b : a) + roff);
    ocol[p] = (int32_t)((transpose ? a : b) + coff);
    osrc[p] = (src_base + (uint32_t)p) | (negate ? NEG : 0u);
  }
}

// One block of a block matrix without transposes: row r of the block goes, in
// order, to its place in the wide row (`at`: where the row's entries of this
// block start), columns shifted, values scaled.
__global__ void k_block_place(const int64_t* row_ptr, const int32_t* col, const double* val, int64_t nrows,
                              int64_t coff, double s, const int64_t* at, int32_t* ocol, double* oval) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, r = t / ROW_LANES;
  if (r >= nrows) return;
  const int64_t b = row_ptr[r], end = row_ptr[r + 1], o = at[r] - b;
  for (int64_t p = b + t % ROW_LANES; p < end; p += ROW_LANES) {
    ocol[o + p] = (int32_t)(col[p] + coff);
    oval[o + p] = s == 1.0 ? val[p] : s == -1.0 ? -val[p] : s * val[p];
  }
}
// row lengths: len[r] += the block's row r (first: =); the exclusive scan of
// them is the row pointer, and `at` of a block what earlier blocks of the row hold
__global__ void k_block_len(const int64_t* row_ptr, int64_t nrows, unsigned long long* len) {
  const int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (r < nrows) len[r] += (unsigned long long)(row_ptr[r + 1] - row_ptr[r]);
}
__global__ void k_block_next(const int64_t* row_ptr, int64_t nrows, int64_t* at) {
  const int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (r < nrows) at[r] += row_ptr[r + 1] - row_ptr[r];
}
__global__ void k_zero_counts(unsigned long long* a, int64_t n) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) a[i] = 0;
}

// The sum of two CSRs with sorted, duplicate-free rows, ADD_LANES lanes a row.
// Count: fresh[p] = b's entries of the row before p whose column a has not (so
// an entry's place in the sum is its own index plus the other side's smaller
// columns), bit 31 set when a has p's column; cnt[r] = the sum's row length.
constexpr int ADD_LANES = 8;
constexpr uint32_t ADD_DUP = 0x80000000u;
__device__ __forceinline__ int64_t lower_col(const int32_t* col, int64_t lo, int64_t hi, int32_t c) {
  while (lo < hi) {
    const int64_t mid = (lo + hi) / 2;
    if (col[mid] < c)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}
// A row of the sum: the left row's entries and the right row's that it lacks,
// each found in the other by bisection: two reads of both operands in place of
// sorting all entries by (row, column), bound by bytes instead of by the sort's
// passes (hdif_gram(1) on 3D 40^3 with its two mass blocks: 2289 us sorted, 622).
__global__ void __launch_bounds__(TPB) k_add_count(const int64_t* arp, const int32_t* acol, const int64_t* brp,
                                                   const int32_t* bcol, int64_t nrows, uint32_t* fresh,
                                                   unsigned long long* cnt) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, r = t / ADD_LANES;
  const int lane = (int)(t % ADD_LANES);
  const bool live = r < nrows;
  const int64_t a0 = live ? arp[r] : 0, a1 = live ? arp[r + 1] : 0;
  const int64_t b0 = live ? brp[r] : 0, b1 = live ? brp[r + 1] : 0;
  uint32_t base = 0;
  const int shift = (int)(threadIdx.x & 63) / ADD_LANES * ADD_LANES;  // the group's lanes in the ballot
  for (int64_t p0 = b0; __any(p0 < b1); p0 += ADD_LANES) {
    const int64_t p = p0 + lane;
    const bool here = p0 < b1 && p < b1;
    bool dup = false;
    if (here) {
      const int32_t c = bcol[p];
      const int64_t q = lower_col(acol, a0, a1, c);
      dup = q < a1 && acol[q] == c;
    }
    const uint32_t mask = (uint32_t)(__ballot(here && !dup) >> shift) & ((1u << ADD_LANES) - 1);
    if (here) fresh[p] = (base + (uint32_t)__popc(mask & ((1u << lane) - 1))) | (dup ? ADD_DUP : 0u);
    base += (uint32_t)__popc(mask);
  }
  if (live && lane == 0) cnt[r] = (unsigned long long)(a1 - a0) + base;
  if (r == nrows && lane == 0) cnt[r] = 0;  // the scan ends on the total
}
// Fill: an entry of both is a's value plus b's, in that order.
__global__ void __launch_bounds__(TPB) k_add_fill(const int64_t* arp, const int32_t* acol, const double* aval,
                                                  const int64_t* brp, const int32_t* bcol, const double* bval,
                                                  int64_t nrows, const uint32_t* fresh, const int64_t* orp,
                                                  int32_t* ocol, double* oval) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, r = t / ADD_LANES;
  if (r >= nrows) return;
  const int lane = (int)(t % ADD_LANES);
  const int64_t a0 = arp[r], a1 = arp[r + 1], b0 = brp[r], b1 = brp[r + 1], o = orp[r];
  const int64_t nfresh = orp[r + 1] - o - (a1 - a0);
  for (int64_t p = a0 + lane; p < a1; p += ADD_LANES) {
    const int32_t c = acol[p];
    const int64_t q = lower_col(bcol, b0, b1, c);
    const int64_t at = o + (p - a0) + (q < b1 ? (int64_t)(fresh[q] & ~ADD_DUP) : nfresh);
    ocol[at] = c;
    oval[at] = q < b1 && bcol[q] == c ? aval[p] + bval[q] : aval[p];
  }
  for (int64_t p = b0 + lane; p < b1; p += ADD_LANES) {
    const uint32_t f = fresh[p];
    if (f & ADD_DUP) continue;
    const int32_t c = bcol[p];
    const int64_t at = o + (lower_col(acol, a0, a1, c) - a0) + f;
    ocol[at] = c;
    oval[at] = bval[p];
  }
}

__global__ void k_scale_copy(const double* a, int64_t n, double s, double* b) {
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) b[i] = (s == 1.0 || s == -1.0) ? a[i] : s * a[i];
}

__global__ void k_select_coo(const int64_t* row_ptr, const int32_t* col, int64_t nrows,
                             const int32_t* rmap, const int32_t* cmap, int32_t* orow,
                             int32_t* ocol, uint32_t* osrc) {
  int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (r >= nrows) return;
  int32_t nr = rmap ? rmap[r] : (int32_t)r;
  for (int64_t p = row_ptr[r]; p < row_ptr[r + 1]; ++p) {
    orow[p] = nr;
    ocol[p] = cmap ? cmap[col[p]] : col[p];
    osrc[p] = (uint32_t)p;
  }
}

// structural product: count terms per row of A, and the longest row
__global__ void k_mul_count(const int64_t* arp, const int32_t* acol, const int64_t* brp,
                            int64_t nrows, unsigned long long* cnt, unsigned long long* longest) {
  __shared__ unsigned long long top;
  if (threadIdx.x == 0) top = 0;
  __syncthreads();
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, r = t / ROW_LANES;
  unsigned long long c = 0;
  if (r < nrows)
    for (int64_t p = arp[r] + t % ROW_LANES; p < arp[r + 1]; p += ROW_LANES) c += brp[acol[p] + 1] - brp[acol[p]];
#pragma unroll
  for (int off = ROW_LANES / 2; off > 0; off >>= 1) c += __shfl_xor(c, off, 64);
  if (r <= nrows && t % ROW_LANES == 0) {
    cnt[r] = c;  // 0 at nrows: the scan ends on the total
    atomicMax(&top, c);
  }
  __syncthreads();
  if (threadIdx.x == 0 && top) atomicMax(longest, top);
}

// One row of the product per wavefront: its terms in the order of A's row go to
// LDS under keys (column, place), a bitonic sort brings equal columns together
// in that order, and each run's first lane adds it up from the left, as a
// stable sort of all terms by (row, column) and a segmented sum would. The rows
// come out at the terms' offsets; len[r] is what each kept. Rows of up to
// MUL_ROW terms (a 4D mass row times the coboundary has about 400): against the
// sort of all terms this reads and writes each one once instead of five times
// (a 4D 7^4 Hodge-Dirac assembly 4959 us with the sort, 3437 so).
constexpr int MUL_ROW = 512, MUL_BITS = 9;
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
__global__ void __launch_bounds__(TPB) k_mul_rows(const int64_t* arp, const int32_t* acol, const double* aval,
                                                  const int64_t* brp, const int32_t* bcol, const double* bval,
                                                  int64_t nrows, const int64_t* start, int32_t* tcol, double* tval,
                                                  unsigned long long* len) {
  __shared__ uint64_t keys_[TPB / 64][MUL_ROW];
  __shared__ double vals_[TPB / 64][MUL_ROW];
  uint64_t* keys = keys_[threadIdx.x / 64];
  double* vals = vals_[threadIdx.x / 64];
  const int lane = (int)(threadIdx.x & 63);
  const int64_t r = blockIdx.x * (int64_t)(TPB / 64) + threadIdx.x / 64;
  if (r > nrows) return;
  if (r == nrows) {
    if (lane == 0) len[r] = 0;
    return;
  }
  const int64_t o = start[r];
  const int m = (int)(start[r + 1] - o);
  const int64_t p1 = arp[r + 1];
  int at = 0;
  for (int64_t p0 = arp[r]; p0 < p1; p0 += 64) {
    const int64_t p = p0 + lane;
    const bool here = p < p1;
    const int32_t k = here ? acol[p] : 0;
    const double av = here ? aval[p] : 0.0;
    const int64_t q0 = here ? brp[k] : 0;
    const int n = here ? (int)(brp[k + 1] - q0) : 0;
    int before = n;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int up = __shfl_up(before, off, 64);
      if (lane >= off) before += up;
    }
    const int all = __shfl(before, 63, 64);
    int w = at + before - n;
    for (int i = 0; i < n; ++i, ++w) {
      keys[w] = (uint64_t)(uint32_t)bcol[q0 + i] << MUL_BITS | (uint64_t)w;
      vals[w] = av * bval[q0 + i];
    }
    at += all;
  }
  int size = 1;
  while (size < m) size <<= 1;
  for (int i = m + lane; i < size; i += 64) keys[i] = ~uint64_t(0);
  wave_lds_fence();
  for (int k = 2; k <= size; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int h = lane; h < size / 2; h += 64) {
        const int i = (h & (j - 1)) | (h & ~(j - 1)) << 1;  // the pair's lower place
        const uint64_t a = keys[i], b = keys[i | j];
        if ((a > b) == ((i & k) == 0)) {
          keys[i] = b;
          keys[i | j] = a;
        }
      }
      wave_lds_fence();
    }
  int kept = 0;
  for (int i0 = 0; i0 < m; i0 += 64) {
    const int i = i0 + lane;
    const uint64_t key = i < m ? keys[i] : 0;
    const bool head = i < m && (i == 0 || (keys[i - 1] ^ key) >> MUL_BITS);
    const uint64_t heads = __ballot(head);
    if (head) {
      double acc = vals[key & (MUL_ROW - 1)];
      for (int j = i + 1; j < m && ((keys[j] ^ key) >> MUL_BITS) == 0; ++j) acc += vals[keys[j] & (MUL_ROW - 1)];
      const int64_t w = o + kept + __popcll(heads & ((uint64_t(1) << lane) - 1));
      tcol[w] = (int32_t)(key >> MUL_BITS);
      tval[w] = acc;
    }
    kept += __popcll(heads);
  }
  if (lane == 0) len[r] = (unsigned long long)kept;
}
__global__ void k_mul_pack(const int64_t* start, const int32_t* tcol, const double* tval, int64_t nrows,
                           const int64_t* orp, int32_t* ocol, double* oval) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, r = t / ROW_LANES;
  if (r >= nrows) return;
  const int64_t o = orp[r], n = orp[r + 1] - o, s = start[r];
  for (int64_t i = t % ROW_LANES; i < n; i += ROW_LANES) {
    ocol[o + i] = tcol[s + i];
    oval[o + i] = tval[s + i];
  }
}

// The terms of the product, row by row in the order of A's row: ROW_LANES lanes
// a row take its entries in turn, each entry's terms after those of the entries
// before it (a prefix of the lanes' counts).
__global__ void __launch_bounds__(TPB) k_mul_terms(const int64_t* arp, const int32_t* acol, const double* aval,
                                                   const int64_t* brp, const int32_t* bcol, const double* bval,
                                                   int64_t nrows, const int64_t* start, int32_t* orow,
                                                   int32_t* ocol, uint32_t* osrc, double* oval) {
  const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, r = t / ROW_LANES;
  const int lane = (int)(t % ROW_LANES);
  const bool live = r < nrows;
  const int64_t p1 = live ? arp[r + 1] : 0;
  int64_t at = live ? start[r] : 0;
  for (int64_t p0 = live ? arp[r] : 0; __any(p0 < p1); p0 += ROW_LANES) {
    const int64_t p = p0 + lane;
    const bool here = p0 < p1 && p < p1;
    const int32_t k = here ? acol[p] : 0;
    const double av = here ? aval[p] : 0.0;
    const int64_t q0 = here ? brp[k] : 0;
    const int len = here ? (int)(brp[k + 1] - q0) : 0;
    int before = len;  // inclusive prefix over the group's lanes
#pragma unroll
    for (int off = 1; off < ROW_LANES; off <<= 1) {
      const int up = __shfl_up(before, off, ROW_LANES);
      if (lane >= off) before += up;
    }
    const int all = __shfl(before, ROW_LANES - 1, ROW_LANES);
    int64_t o = at + before - len;
    for (int i = 0; i < len; ++i, ++o) {
      orow[o] = (int32_t)r;
      ocol[o] = bcol[q0 + i];
      osrc[o] = (uint32_t)o;
      oval[o] = av * bval[q0 + i];
    }
    at += all;
  }
}

}  // namespace

void csr_block(Ctx* ctx, int nb, const BlockRef* blocks, const int64_t* row_sizes,
               const int64_t* col_sizes, Csr& out) {
  std::vector<int64_t> roff(nb + 1, 0), coff(nb + 1, 0);
  for (int i = 0; i < nb; ++i) {
    roff[i + 1] = roff[i] + row_sizes[i];
    coff[i + 1] = coff[i] + col_sizes[i];
  }
  int64_t total = 0;
  bool transposed = false;
  for (int i = 0; i < nb * nb; ++i)
    if (blocks[i].a) {
      total += blocks[i].a->nnz;
      transposed = transposed || (blocks[i].transpose && blocks[i].a->nnz);
    }
  require_entries(total);
  if (!transposed) {
    // the blocks' rows side by side: sorted already, no entry twice
    const int64_t n = roff[nb];
    out.ctx = ctx;
    out.nrows = n;
    out.ncols = coff[nb];
    out.nnz = total;
    out.row_ptr.alloc(ctx, n + 1);
    out.col.alloc(ctx, total);
    out.val.alloc(ctx, total);
    DBuf<unsigned long long> len(ctx, n + 1);
    DBuf<int64_t> at(ctx, std::max<int64_t>(n, 1));
    k_zero_counts<<<grid_for(n + 1), TPB, 0, ctx->stream>>>(len.p, n + 1);
    for (int i = 0; i < nb * nb; ++i)
      if (blocks[i].a && blocks[i].a->nnz)
        k_block_len<<<grid_for(blocks[i].a->nrows), TPB, 0, ctx->stream>>>(
            blocks[i].a->row_ptr.p, blocks[i].a->nrows, len.p + roff[i / nb]);
    exclusive_scan_u64_to_i64<int64_t>(ctx, len.p, out.row_ptr.p, n + 1);
    if (n)
      FEEC_HIP(hipMemcpyAsync(at.p, out.row_ptr.p, n * sizeof(int64_t), hipMemcpyDeviceToDevice, ctx->stream));
    for (int i = 0; i < nb * nb; ++i) {
      const BlockRef& b = blocks[i];
      if (!b.a || b.a->nnz == 0) continue;
      k_block_place<<<row_grid(b.a->nrows), TPB, 0, ctx->stream>>>(b.a->row_ptr.p, b.a->col.p, b.a->val.p,
                                                                   b.a->nrows, coff[i % nb], b.scale,
                                                                   at.p + roff[i / nb], out.col.p, out.val.p);
      k_block_next<<<grid_for(b.a->nrows), TPB, 0, ctx->stream>>>(b.a->row_ptr.p, b.a->nrows,
                                                                  at.p + roff[i / nb]);
    }
    FEEC_HIP(hipGetLastError());
    ctx->sync();
    return;
  }
  DBuf<int32_t> rows(ctx, total), cols(ctx, total);
  DBuf<uint32_t> srcs(ctx, total);
  DBuf<double> vals(ctx, total);
  int64_t at = 0;
  for (int bi = 0; bi < nb; ++bi)
    for (int bj = 0; bj < nb; ++bj) {
      const BlockRef& b = blocks[bi * nb + bj];
      if (!b.a || b.a->nnz == 0) continue;
      double s = b.scale;
      k_block_coo<<<row_grid(b.a->nrows), TPB, 0, ctx->stream>>>(
          b.a->row_ptr.p, b.a->col.p, b.a->nrows, roff[bi], coff[bj], b.transpose,
          (uint32_t)at, s == -1.0, rows.p + at, cols.p + at, srcs.p + at);
      k_scale_copy<<<grid_for(b.a->nnz), TPB, 0, ctx->stream>>>(b.a->val.p, b.a->nnz, s,
                                                                vals.p + at);
      at += b.a->nnz;
    }
  CooPlan plan;
  coo_plan_build(ctx, plan, roff[nb], coff[nb], total, rows.p, cols.p, srcs.p);
  coo_plan_apply(ctx, plan, vals.p, false, out);
}

// Exclusive prefix sum of n counts (n >= 1) into out[0..n).
void exclusive_scan_counts(Ctx* ctx, const unsigned long long* in, int64_t* out, int64_t n) {
  exclusive_scan_u64_to_i64<int64_t>(ctx, in, out, n);
}

void csr_transpose(const Csr& a, Csr& out) {
  BlockRef b{&a, 1.0, true};
  int64_t r = a.ncols, c = a.nrows;
  csr_block(a.ctx, 1, &b, &r, &c, out);
}

// a + b row by row (sorted rows without repeated columns, as every library CSR
// has them): a merge instead of a sort of both operands' entries.
void csr_add(const Csr& a, const Csr& b, Csr& out) {
  Ctx* ctx = a.ctx;
  const int64_t n = a.nrows;
  FEEC_REQUIRE(n == b.nrows && a.ncols == b.ncols, FEEC_E_ARG, "csr_add shape mismatch");
  require_entries(a.nnz + b.nnz);
  out.ctx = ctx;
  out.nrows = n;
  out.ncols = a.ncols;
  out.row_ptr.alloc(ctx, n + 1);
  DBuf<uint32_t> fresh(ctx, std::max<int64_t>(b.nnz, 1));
  DBuf<unsigned long long> cnt(ctx, n + 1);
  k_add_count<<<grid_for((n + 1) * ADD_LANES), TPB, 0, ctx->stream>>>(a.row_ptr.p, a.col.p, b.row_ptr.p, b.col.p, n,
                                                                      fresh.p, cnt.p);
  FEEC_HIP(hipGetLastError());
  exclusive_scan_u64_to_i64<int64_t>(ctx, cnt.p, out.row_ptr.p, n + 1);
  copy_to_host(ctx, &out.nnz, out.row_ptr.p + n, sizeof(int64_t));
  out.col.alloc(ctx, out.nnz);
  out.val.alloc(ctx, out.nnz);
  if (n)
    k_add_fill<<<grid_for(n * ADD_LANES), TPB, 0, ctx->stream>>>(a.row_ptr.p, a.col.p, a.val.p, b.row_ptr.p, b.col.p,
                                                                 b.val.p, n, fresh.p, out.row_ptr.p, out.col.p,
                                                                 out.val.p);
  FEEC_HIP(hipGetLastError());
  ctx->sync();
}

void csr_select(const Csr& a, const int32_t* row_map, int64_t nrows, const int32_t* col_map,
                int64_t ncols, Csr& out) {
  Ctx* ctx = a.ctx;
  DBuf<int32_t> rows(ctx, a.nnz), cols(ctx, a.nnz);
  DBuf<uint32_t> srcs(ctx, a.nnz);
  if (a.nnz)
    k_select_coo<<<grid_for(a.nrows), TPB, 0, ctx->stream>>>(a.row_ptr.p, a.col.p, a.nrows,
                                                             row_map, col_map, rows.p, cols.p,
                                                             srcs.p);
  CooPlan plan;
  coo_plan_build(ctx, plan, nrows, ncols, a.nnz, rows.p, cols.p, srcs.p);
  coo_plan_apply(ctx, plan, a.val.p, false, out);
}

void csr_mul(const Csr& a, const Csr& b, Csr& out) {
  Ctx* ctx = a.ctx;
  FEEC_REQUIRE(a.ncols == b.nrows, FEEC_E_ARG, "csr_mul shape mismatch");
  const int64_t n = a.nrows;
  DBuf<unsigned long long> cnt(ctx, n + 1), longest(ctx, 1);
  DBuf<int64_t> start(ctx, n + 1);
  k_zero_counts<<<1, TPB, 0, ctx->stream>>>(longest.p, 1);
  k_mul_count<<<row_grid(n + 1), TPB, 0, ctx->stream>>>(a.row_ptr.p, a.col.p, b.row_ptr.p, n, cnt.p, longest.p);
  FEEC_HIP(hipGetLastError());
  exclusive_scan_u64_to_i64<int64_t>(ctx, cnt.p, start.p, n + 1);
  int64_t total = 0;
  unsigned long long most = 0;
  FEEC_HIP(hipMemcpyAsync(&total, start.p + n, sizeof(int64_t), hipMemcpyDeviceToHost, ctx->stream));
  FEEC_HIP(hipMemcpyAsync(&most, longest.p, sizeof(most), hipMemcpyDeviceToHost, ctx->stream));
  ctx->sync();
  FEEC_REQUIRE(total < (int64_t(1) << 31), FEEC_E_ARG, "product too large");
  if (most <= MUL_ROW) {
    DBuf<int32_t> tcol(ctx, std::max<int64_t>(total, 1));
    DBuf<double> tval(ctx, std::max<int64_t>(total, 1));
    k_mul_rows<<<(unsigned)(n / (TPB / 64) + 1), TPB, 0, ctx->stream>>>(a.row_ptr.p, a.col.p, a.val.p, b.row_ptr.p,
                                                                       b.col.p, b.val.p, n, start.p, tcol.p, tval.p,
                                                                       cnt.p);
    FEEC_HIP(hipGetLastError());
    out.ctx = ctx;
    out.nrows = n;
    out.ncols = b.ncols;
    out.row_ptr.alloc(ctx, n + 1);
    exclusive_scan_u64_to_i64<int64_t>(ctx, cnt.p, out.row_ptr.p, n + 1);
    copy_to_host(ctx, &out.nnz, out.row_ptr.p + n, sizeof(int64_t));
    out.col.alloc(ctx, out.nnz);
    out.val.alloc(ctx, out.nnz);
    if (n)
      k_mul_pack<<<row_grid(n), TPB, 0, ctx->stream>>>(start.p, tcol.p, tval.p, n, out.row_ptr.p, out.col.p,
                                                       out.val.p);
    FEEC_HIP(hipGetLastError());
    ctx->sync();
    return;
  }
  DBuf<int32_t> rows(ctx, total), cols(ctx, total);
  DBuf<uint32_t> srcs(ctx, total);
  DBuf<double> vals(ctx, total);
  if (n)
    k_mul_terms<<<row_grid(a.nrows), TPB, 0, ctx->stream>>>(
        a.row_ptr.p, a.col.p, a.val.p, b.row_ptr.p, b.col.p, b.val.p, a.nrows, start.p, rows.p,
        cols.p, srcs.p, vals.p);
  CooPlan plan;
  coo_plan_build(ctx, plan, a.nrows, b.ncols, total, rows.p, cols.p, srcs.p);
  coo_plan_apply(ctx, plan, vals.p, false, out);
}

void csr_diagonal(const Csr& a, double* diag_dev) {
  int64_t n = std::min(a.nrows, a.ncols);
  k_diag<<<grid_for(n), TPB, 0, a.ctx->stream>>>(a.row_ptr.p, a.col.p, a.val.p, n, diag_dev);
  FEEC_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// element matrices -> Galerkin matrix
// ---------------------------------------------------------------------------
namespace {

// contributions of one element block, cell-major (t = cell * r * c + i * c + j),
// source index = SoA slot (i * c + j) * ncells + cell + base
__global__ void k_form_coo(const int32_t* faces_r, int nfr, const int32_t* faces_c, int nfc,
                           const int32_t* rmap, const int32_t* cmap, int64_t roff, int64_t coff,
                           int64_t nc, int r, int c, bool transpose, uint32_t base, bool negate,
                           int32_t* orow, int32_t* ocol, uint32_t* osrc) {
  int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  int64_t per = (int64_t)r * c;
  if (t >= nc * per) return;
  int64_t cell = t / per;
  int e = (int)(t % per);
  int i = e / c, j = e % c;
  int32_t gi = faces_r[cell * nfr + i];
  int32_t gj = faces_c[cell * nfc + j];
  if (rmap) gi = rmap[gi];
  if (cmap) gj = cmap[gj];
  bool ok = gi >= 0 && gj >= 0;
  int32_t R = ok ? (int32_t)(gi + roff) : -1, C = ok ? (int32_t)(gj + coff) : -1;
  orow[t] = transpose ? C : R;
  ocol[t] = transpose ? R : C;
  osrc[t] = (base + (uint32_t)((int64_t)e * nc + cell)) | (negate ? NEG : 0u);
}

}  // namespace

struct FormSide {
  int grade;
  int64_t offset;
};

// Contribution list of one element block of size r x c whose rows are the
// local faces of grade rg and columns of grade cg.
void form_contributions(Mesh& m, int bc, int rg, int cg, int r, int c, int64_t roff, int64_t coff,
                        bool transpose, uint32_t base, bool negate, int32_t* rows, int32_t* cols,
                        uint32_t* srcs) {
  int64_t nc = m.n[m.d];
  if (bc == FEEC_RELATIVE) m.ensure_interior();
  const int32_t* rmap = bc == FEEC_RELATIVE ? m.interior[rg].p : nullptr;
  const int32_t* cmap = bc == FEEC_RELATIVE ? m.interior[cg].p : nullptr;
  k_form_coo<<<grid_for(nc * r * c), TPB, 0, m.ctx->stream>>>(
      m.faces[rg].p, m.nfaces(rg), m.faces[cg].p, m.nfaces(cg), rmap, cmap, roff, coff, nc, r, c,
      transpose, base, negate, rows, cols, srcs);
  FEEC_HIP(hipGetLastError());
}

int64_t ndofs(Mesh& m, int bc, int k) {
  if (k < 0 || k > m.d) return 0;
  if (bc == FEEC_RELATIVE) {
    m.ensure_interior();
    return m.n_interior[k];
  }
  return m.n[k];
}

const CooPlan& form_plan(Mesh& m, int bc, int kind, int grade) {
  auto key = std::make_tuple(bc, kind, grade);
  {
    std::lock_guard<std::mutex> lock(m.mu);
    auto it = m.plans.find(key);
    if (it != m.plans.end()) return *it->second;
  }
  int tg = (kind == 2 || kind == 3) ? grade - 1 : grade;
  int rg = (kind == 1 || kind == 3) ? grade - 1 : grade;
  int r = element_rows(m.d, kind, grade), c = element_cols(m.d, kind, grade);
  int64_t nc = m.n[m.d];
  int64_t n = nc * r * c;
  auto plan = std::make_unique<CooPlan>();
  {
    DBuf<int32_t> rows(m.ctx, n), cols(m.ctx, n);
    DBuf<uint32_t> srcs(m.ctx, n);
    form_contributions(m, bc, tg, rg, r, c, 0, 0, false, 0, false, rows.p, cols.p, srcs.p);
    coo_plan_build(m.ctx, *plan, ndofs(m, bc, tg), ndofs(m, bc, rg), n, rows.p, cols.p, srcs.p);
  }
  std::lock_guard<std::mutex> lock(m.mu);
  auto& slot = m.plans[key];
  slot = std::move(plan);
  return *slot;
}

void assemble_form(Geom& g, int bc, int kind, int grade, Csr& out) {
  Mesh& m = *g.mesh;
  Ctx* ctx = m.ctx;
  out.ctx = ctx;
  if (kind == FEEC_HDIF_GRAM) {
    Csr a, b;
    assemble_form(g, bc, FEEC_MASS, grade, a);
    assemble_form(g, bc, FEEC_DIF_BOTH, grade + 1, b);
    csr_add(a, b, out);
    return;
  }
  int tg = (kind == 2 || kind == 3) ? grade - 1 : grade;
  int rg = (kind == 1 || kind == 3) ? grade - 1 : grade;
  int64_t nr = ndofs(m, bc, tg), ncl = ndofs(m, bc, rg);
  int r = element_rows(m.d, kind, grade), c = element_cols(m.d, kind, grade);
  // HilbertComplex::pairing (whitney_complex.rs:113-122): empty off the complex
  if (grade < 0 || grade > m.d || nr == 0 || ncl == 0 || r == 0 || c == 0) {
    out.nrows = nr;
    out.ncols = ncl;
    out.nnz = 0;
    out.row_ptr.alloc(ctx, nr + 1);
    FEEC_HIP(hipMemsetAsync(out.row_ptr.p, 0, (nr + 1) * sizeof(int64_t), ctx->stream));
    out.col.alloc(ctx, 0);
    out.val.alloc(ctx, 0);
    ctx->sync();
    return;
  }
  int64_t nc = m.n[m.d];
  DBuf<double> el(ctx, (size_t)nc * r * c);
  element_matrices_soa(g, kind, grade, el.p);
  const CooPlan& plan = form_plan(m, bc, kind, grade);
  coo_plan_apply(ctx, plan, el.p, true, out);
}

}  // namespace feec

namespace feec {

namespace {
__global__ void k_scatter_kept(const double* vals, const uint8_t* keep, const int64_t* pos,
                               int64_t n, double* out) {
  int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (e < n && keep[e]) out[pos[e]] = vals[e];
}
__global__ void k_keep_diff(const uint8_t* a, const uint8_t* b, int64_t n,
                            unsigned long long* cnt) {
  int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (e < n && a[e] != b[e]) atomicAdd(cnt, 1ull);
}
__global__ void k_dense_column(const int64_t* row_ptr, int64_t nrows, const double* v,
                               double* out) {
  int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (r >= nrows) return;
  int64_t b = row_ptr[r];
  out[r] = (row_ptr[r + 1] > b) ? v[b] : 0.0;
}
}  // namespace

void coo_plan_dense_column(Ctx* ctx, const CooPlan& plan, const double* vals, double* out) {
  DBuf<double> v(ctx, std::max<int64_t>(plan.nnz, 1));
  coo_plan_values(ctx, plan, vals, v.p, nullptr);
  k_dense_column<<<grid_for(plan.nrows), TPB, 0, ctx->stream>>>(plan.row_ptr.p, plan.nrows, v.p,
                                                                out);
  FEEC_HIP(hipGetLastError());
}

// Values of a plan into a CSR whose pattern is the plan's minus the entries
// whose contributions are all exactly zero. The first call (or a call where the
// set of such entries changed) rebuilds the compacted pattern and returns true.
bool assemble_compacted(Ctx* ctx, const CooPlan& plan, const double* vals, CompactMap& cm,
                        Csr& A) {
  const int64_t ns = plan.nnz;
  DBuf<double> v(ctx, ns);
  DBuf<uint8_t> keep(ctx, ns);
  int64_t dropped = coo_plan_values(ctx, plan, vals, v.p, keep.p);
  bool rebuild = !cm.valid;
  if (cm.valid) {
    DBuf<unsigned long long> cnt(ctx, 1);
    FEEC_HIP(hipMemsetAsync(cnt.p, 0, sizeof(unsigned long long), ctx->stream));
    if (ns)
      k_keep_diff<<<grid_for(ns), TPB, 0, ctx->stream>>>(keep.p, cm.keep.p, ns, cnt.p);
    unsigned long long h = 0;
    FEEC_HIP(hipMemcpyAsync(&h, cnt.p, sizeof(h), hipMemcpyDeviceToHost, ctx->stream));
    ctx->sync();
    rebuild = h != 0;
  }
  if (rebuild) {
    A.ctx = ctx;
    A.nrows = plan.nrows;
    A.ncols = plan.ncols;
    A.nnz = ns - dropped;
    A.row_ptr.alloc(ctx, plan.nrows + 1);
    A.col.alloc(ctx, A.nnz);
    A.val.alloc(ctx, A.nnz);
    cm.pos.alloc(ctx, ns);
    if (ns) {
      DBuf<unsigned long long> k64(ctx, ns);
      k_u8_to_u64<<<grid_for(ns), TPB, 0, ctx->stream>>>(keep.p, ns, k64.p);
      exclusive_scan_u64_to_i64<int64_t>(ctx, k64.p, cm.pos.p, ns);
    }
    if (ns)
      k_compact_entries<<<grid_for(ns), TPB, 0, ctx->stream>>>(plan.col.p, v.p, keep.p, cm.pos.p,
                                                               ns, A.col.p, A.val.p);
    k_compact_rows<<<grid_for(plan.nrows + 1), TPB, 0, ctx->stream>>>(
        plan.row_ptr.p, plan.nrows, cm.pos.p, ns, A.nnz, A.row_ptr.p);
    cm.keep = std::move(keep);
    cm.valid = true;
  } else if (ns) {
    k_scatter_kept<<<grid_for(ns), TPB, 0, ctx->stream>>>(v.p, cm.keep.p, cm.pos.p, ns, A.val.p);
  }
  FEEC_HIP(hipGetLastError());
  ctx->sync();
  return rebuild;
}

}  // namespace feec
