// Precompiled utility kernels (gfx950).  They replace the util module the
// reference builds with NVRTC in debug mode (CUDAAssembler.cpp:38-164,
// compiled with --device-debug per fem.cpp:210): zero fill, coefficient
// packing, set_bc, set_diagonal, plus the setup kernels of this engine
// (bs-unrolling of the CSR columns, offset tables, lifting entity lists).
#include <mutex>

#include "mf_internal.h"

namespace mf {
namespace {

constexpr int kBlock = 256;

inline uint32_t grid_for(int64_t n, int per_thread = 1) {
  int64_t g = (n + (int64_t)kBlock * per_thread - 1) / ((int64_t)kBlock * per_thread);
  if (g > 65535LL * 32) g = 65535LL * 32;
  return static_cast<uint32_t>(g < 1 ? 1 : g);
}

__global__ void fill_kernel(double* __restrict__ x, int64_t n, double v) {
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) x[i] = v;
}

// dst[map[k]] += src[k]: values of a matrix on the form's own pattern added
// into a caller's CSR whose pattern is a superset without the bs-unrolled
// block structure (map is injective, so no two threads share a target)
__global__ void scatter_add_kernel(double* __restrict__ dst, const double* __restrict__ src,
                                   const int32_t* __restrict__ map, int64_t n) {
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += stride)
    dst[map[k]] += src[k];
}

__global__ void fill_i32_kernel(int32_t* __restrict__ x, int64_t n, int32_t v) {
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) x[i] = v;
}

// Sum of the per-block partial sums of a scalar assembly, in a fixed order
// (one workgroup: strided per-thread sums, then a wave64 shuffle tree and a
// cross-wave LDS step), so repeated assemblies give bit-identical values.
__global__ void __launch_bounds__(kBlock) sum_partials_kernel(const double* __restrict__ p,
                                                              int64_t n, double* __restrict__ out,
                                                              int accumulate) {
  double acc = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += kBlock) acc += p[i];
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_down(acc, o, 64);
  __shared__ double red[kBlock / 64];
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int k = 0; k < kBlock / 64; ++k) t += red[k];
    out[0] = accumulate ? out[0] + t : t;
  }
}

// Same-map interpolation, one thread per target dof (node, component): the
// target node's value comes from its owning cell (c, local i),
// u1 = sum_k im[i][k] u0(dm0(c, k)), k ascending.
__global__ void interp_kernel(double* __restrict__ u1, const double* __restrict__ u0,
                              const int32_t* __restrict__ own, const int32_t* __restrict__ dm0,
                              const double* __restrict__ im, int64_t n, int n1, int n0, int bs) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int64_t node = t / bs;
  const int comp = static_cast<int>(t - node * bs);
  const int32_t ci = own[node];
  if (ci < 0) return;
  const int32_t c = ci / n1, i = ci - c * n1;
  const int32_t* d0 = dm0 + (int64_t)c * n0;
  const double* row = im + (int64_t)i * n0;
  double acc = 0.0;
  for (int k = 0; k < n0; ++k) acc += row[k] * u0[(int64_t)bs * d0[k] + comp];
  u1[t] = acc;
}

__global__ void mark_kernel(int8_t* __restrict__ m, int64_t ndofs, const int32_t* __restrict__ dofs,
                            int64_t nbc) {
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nbc; i += stride) {
    int32_t d = dofs[i];
    if (d >= 0 && d < ndofs) m[d] = 1;
  }
}

__global__ void cell_flags_kernel(uint8_t* __restrict__ flags, const int32_t* __restrict__ dm,
                                  int64_t ncells, int nd, const uint8_t* __restrict__ bits) {
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < ncells; c += stride) {
    uint8_t any = 0;
    for (int l = 0; l < nd; ++l) any |= bits[dm[c * nd + l]];
    flags[c] = any ? 1 : 0;
  }
}

__global__ void node_bits_kernel(uint8_t* __restrict__ bits, const int8_t* __restrict__ m,
                                 int64_t nnodes, int bs) {
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nnodes; i += stride) {
    uint8_t v = 0;
    for (int a = 0; a < bs; ++a) v |= (m[i * bs + a] ? 1 : 0) << a;
    bits[i] = v;
  }
}

// packed[c*W + off + k*bs + j] = values[bs*dofmap[c*nd + k] + j] for up to kPack
// coefficients of a form at once.  Threads run over the packed entries (cum: first
// entry of each coefficient among those packed), so a wave writes consecutive
// addresses whatever the widths, and a form's coefficients cost one launch.  N:
// number of coefficients, selected by compares; I: 32-bit indices where they do.
// Bound by launches at these sizes (4 to 7 us each): two P2 coefficients on 48
// thousand cells 10.6 -> 5.4 us.
constexpr int kPack = kPackItems;
template <int N>
struct PackArgs {
  const double* values[N];
  const int32_t* dofmap[N];
  int32_t nd[N], bs[N], off[N], cum[N + 1];
};

template <int N, class I>
__global__ void pack_kernel(double* __restrict__ packed, int64_t ncells, int W, const PackArgs<N> a) {
  const I width = a.cum[N], total = static_cast<I>(ncells) * width;
  const I stride = static_cast<I>(gridDim.x) * blockDim.x;
  for (I l = static_cast<I>(blockIdx.x) * blockDim.x + threadIdx.x; l < total; l += stride) {
    const I c = l / width;
    const int rr = static_cast<int>(l - c * width);
    const double* values = a.values[0];
    const int32_t* dofmap = a.dofmap[0];
    int nd = a.nd[0], bs = a.bs[0], off = a.off[0], first = 0;
#pragma unroll
    for (int g = 1; g < N; ++g)
      if (rr >= a.cum[g]) {
        values = a.values[g];
        dofmap = a.dofmap[g];
        nd = a.nd[g];
        bs = a.bs[g];
        off = a.off[g];
        first = a.cum[g];
      }
    const int r = rr - first, k = bs == 1 ? r : r / bs, j = r - k * bs;
    packed[static_cast<int64_t>(c) * W + off + r] =
        values[static_cast<int64_t>(bs) * dofmap[static_cast<int64_t>(c) * nd + k] + j];
  }
}

__global__ void set_bc_kernel(double* __restrict__ b, int64_t n, const int32_t* __restrict__ dofs,
                              int64_t nbc, const double* __restrict__ g,
                              const double* __restrict__ x0, double scale) {
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nbc; i += stride) {
    int32_t d = dofs[i];
    if (d < 0 || d >= n) continue;
    b[d] = scale * (g[d] - (x0 ? x0[d] : 0.0));
  }
}

// set_bc for up to 32 vectors in one launch: the groups' constrained dofs
// are numbered consecutively (start[g] .. start[g + 1]), every thread finds
// its group by a scan of the (at most 32) starts
struct SetBcBatchArgs {
  double* b[32];
  const int32_t* dofs[32];
  const double* g[32];
  int64_t n[32];
  int64_t start[33];
  int32_t ngroups;
};

__global__ void set_bc_batch_kernel(const SetBcBatchArgs a, double scale) {
  const int64_t total = a.start[a.ngroups];
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
    int grp = 0;
    while (grp + 1 < a.ngroups && a.start[grp + 1] <= i) ++grp;
    const int32_t d = a.dofs[grp][i - a.start[grp]];
    if (d < 0 || d >= a.n[grp]) continue;
    a.b[grp][d] = scale * a.g[grp][d];
  }
}

__device__ __forceinline__ int64_t search(const int32_t* __restrict__ cols, int64_t lo, int64_t hi,
                                          int32_t key) {
  // first position in [lo, hi) with cols[p] >= key
  while (lo < hi) {
    int64_t mid = lo + ((hi - lo) >> 1);
    if (cols[mid] < key) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

__global__ void set_diag_kernel(double* __restrict__ values, const int32_t* __restrict__ row_ptr,
                                const int32_t* __restrict__ cols, const int32_t* __restrict__ dofs,
                                int64_t nbc, int64_t nrows, double diag) {
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nbc; i += stride) {
    int32_t r = dofs[i];
    if (r < 0 || r >= nrows) continue;
    int64_t e = row_ptr[r + 1];
    int64_t p = search(cols, row_ptr[r], e, r);
    if (p < e && cols[p] == r) values[p] = diag;
  }
}

// One thread per blocked entry (r, k): writes the bs0*bs1 scalar columns.
__global__ void unroll_kernel(int32_t* __restrict__ cols, const int32_t* __restrict__ row_ptr,
                              const int32_t* __restrict__ rpb, const int32_t* __restrict__ colsb,
                              int64_t nrows_b, int bs0, int bs1) {
  int64_t nnzb = rpb[nrows_b];
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < nnzb; q += stride) {
    // row of q by binary search in rpb
    int64_t lo = 0, hi = nrows_b;
    while (hi - lo > 1) {
      int64_t mid = (lo + hi) >> 1;
      if (rpb[mid] <= q) lo = mid;
      else hi = mid;
    }
    int64_t r = lo, k = q - rpb[r];
    int32_t c = colsb[q];
    for (int a = 0; a < bs0; ++a) {
      int64_t base = (int64_t)row_ptr[r * bs0 + a] + k * bs1;
      for (int b = 0; b < bs1; ++b) cols[base + b] = bs1 * c + b;
    }
  }
}

__global__ void table_kernel(int32_t* __restrict__ table, const int32_t* __restrict__ ents,
                             int64_t nents, int stride, int ncell, const int32_t* __restrict__ dm0,
                             int nd0, const int32_t* __restrict__ dm1, int nd1, int bs0, int bs1,
                             const int32_t* __restrict__ row_ptr, const int32_t* __restrict__ rpb,
                             const int32_t* __restrict__ colsb, int32_t* __restrict__ missing) {
  const int NI = ncell * nd0, NJ = ncell * nd1;
  const int64_t total = nents * NI * NJ;
  int64_t gs = (int64_t)gridDim.x * blockDim.x;
  for (int64_t l = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; l < total; l += gs) {
    int64_t e = l / (NI * NJ);
    int ij = static_cast<int>(l - e * NI * NJ);
    int i = ij / NJ, j = ij - i * NJ;
    int32_t ci = ents[e * stride + 2 * (i / nd0)];
    int32_t cj = ents[e * stride + 2 * (j / nd1)];
    int32_t rn = dm0[(int64_t)ci * nd0 + (i % nd0)];
    int32_t cn = dm1[(int64_t)cj * nd1 + (j % nd1)];
    int64_t lo = rpb[rn], hi = rpb[rn + 1];
    int64_t p = search(colsb, lo, hi, cn);
    int32_t v = -1;
    if (p < hi && colsb[p] == cn)
      v = static_cast<int32_t>((int64_t)row_ptr[(int64_t)bs0 * rn] + (p - lo) * bs1);
    else
      atomicAdd(missing, 1);
    table[(e >> 6) * (int64_t)NI * NJ * 64 + (int64_t)ij * 64 + (e & 63)] = v;
  }
}

// Contributions of an integral to each blocked CSR entry q: fill == nullptr
// counts them (count[q]); otherwise count holds the next free place of q and
// fill gets each contribution's offset in the element-tensor workspace (entity
// e, local nodes i, j: plane (i bs0) NJ bs1 + j bs1 of the 64 entities of e).
__global__ void gather_plan_kernel(int32_t* __restrict__ count, int32_t* __restrict__ fill,
                                   const int32_t* __restrict__ ents, int64_t nents, int stride,
                                   int ncell, const int32_t* __restrict__ dm0, int nd0,
                                   const int32_t* __restrict__ dm1, int nd1, int bs0, int bs1,
                                   const int32_t* __restrict__ rpb,
                                   const int32_t* __restrict__ colsb, int32_t* __restrict__ missing) {
  const int NI = ncell * nd0, NJ = ncell * nd1;
  const int64_t total = nents * NI * NJ;
  const int64_t gs = (int64_t)gridDim.x * blockDim.x;
  for (int64_t l = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; l < total; l += gs) {
    const int64_t e = l / (NI * NJ);
    const int ij = static_cast<int>(l - e * NI * NJ);
    const int i = ij / NJ, j = ij - i * NJ;
    const int32_t ci = ents[e * stride + 2 * (i / nd0)], cj = ents[e * stride + 2 * (j / nd1)];
    const int32_t rn = dm0[(int64_t)ci * nd0 + (i % nd0)], cn = dm1[(int64_t)cj * nd1 + (j % nd1)];
    const int64_t hi = rpb[rn + 1], p = search(colsb, rpb[rn], hi, cn);
    if (p >= hi || colsb[p] != cn) {
      atomicAdd(missing, 1);
      continue;
    }
    const int32_t k = atomicAdd(&count[p], 1);
    if (fill) {
      const int64_t plane = (int64_t)i * bs0 * NJ * bs1 + (int64_t)j * bs1;
      const int64_t planes = (int64_t)NI * bs0 * NJ * bs1;
      fill[k] = static_cast<int32_t>(((e >> 6) * planes + plane) * 64 + (e & 63));
    }
  }
}

// Ascending order within every entry's contributions (a fixed order of
// summation), and the entry's place in the bs-unrolled CSR: pos[q] = (offset of
// its first value, length of its scalar rows).
__global__ void gather_sort_kernel(int32_t* __restrict__ fill, const int32_t* __restrict__ ptr,
                                   int2* __restrict__ pos, int64_t nq, int64_t nrows_b,
                                   const int32_t* __restrict__ rpb,
                                   const int32_t* __restrict__ row_ptr, int bs0, int bs1) {
  const int64_t gs = (int64_t)gridDim.x * blockDim.x;
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < nq; q += gs) {
    for (int32_t a = ptr[q] + 1; a < ptr[q + 1]; ++a) {
      const int32_t v = fill[a];
      int32_t b = a - 1;
      for (; b >= ptr[q] && fill[b] > v; --b) fill[b + 1] = fill[b];
      fill[b + 1] = v;
    }
    int64_t lo = 0, hi = nrows_b;                      // row of q
    while (hi - lo > 1) {
      const int64_t mid = (lo + hi) >> 1;
      if (rpb[mid] <= q) lo = mid;
      else hi = mid;
    }
    const int32_t r0 = row_ptr[lo * bs0];
    pos[q] = make_int2(r0 + static_cast<int32_t>(q - rpb[lo]) * bs1, row_ptr[lo * bs0 + 1] - r0);
  }
}

// values = sum of each entry's element-tensor contributions, in ascending order
// (0 where it has none): one thread per scalar value.  Bound by memory: the
// tensors (8 B) and their places (4 B) read once, the values written once.
// Workgroups of one XCD take a contiguous eighth of the entries, whose
// contributions lie close together in the workspace.
__global__ void __launch_bounds__(kBlock) gather_kernel(
    double* __restrict__ values, const double* __restrict__ ws, const int32_t* __restrict__ ptr,
    const int32_t* __restrict__ at, const int2* __restrict__ pos, int64_t nq, int bs0, int bs1,
    int row_stride) {
  const int64_t per = (gridDim.x + 7) / 8;
  const int64_t t = ((blockIdx.x % 8) * per + blockIdx.x / 8) * kBlock + threadIdx.x;
  const int bb = bs0 * bs1;
  const int64_t q = bb == 1 ? t : t / bb;
  if (q >= nq) return;
  const int ab = static_cast<int>(t - q * bb), a = ab / bs1, b = ab - a * bs1;
  const int32_t off = (a * row_stride + b) * 64;
  double sum = 0.0;
  int32_t k = ptr[q];
  const int32_t e = ptr[q + 1];
  for (; k + 3 < e; k += 4) {
    const int32_t k0 = at[k], k1 = at[k + 1], k2 = at[k + 2], k3 = at[k + 3];
    const double v0 = ws[k0 + off], v1 = ws[k1 + off], v2 = ws[k2 + off], v3 = ws[k3 + off];
    sum += v0;
    sum += v1;
    sum += v2;
    sum += v3;
  }
  for (; k < e; ++k) sum += ws[at[k] + off];
  if (bb == 1) {
    values[q] = sum;
  } else {
    const int2 p = pos[q];
    values[(int64_t)p.x + (int64_t)a * p.y + b] = sum;
  }
}

__global__ void block_table_kernel(int32_t* __restrict__ table, const int32_t* __restrict__ ents,
                                   int64_t nents, int stride, int ncell,
                                   const int32_t* __restrict__ dm0, int nd0,
                                   const int32_t* __restrict__ rmap0, int64_t off0, int bs0,
                                   const int32_t* __restrict__ dm1, int nd1,
                                   const int32_t* __restrict__ rmap1, int64_t off1, int bs1,
                                   const int32_t* __restrict__ row_ptr,
                                   const int32_t* __restrict__ cols, int32_t* __restrict__ missing) {
  const int NI = ncell * nd0, NJ = ncell * nd1;
  const int64_t total = nents * NI * NJ;
  int64_t gs = (int64_t)gridDim.x * blockDim.x;
  for (int64_t l = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; l < total; l += gs) {
    int64_t e = l / (NI * NJ);
    int ij = static_cast<int>(l - e * NI * NJ);
    int i = ij / NJ, j = ij - i * NJ;
    int32_t ci = ents[e * stride + 2 * (i / nd0)];
    int32_t cj = ents[e * stride + 2 * (j / nd1)];
    int32_t rn = dm0[(int64_t)ci * nd0 + (i % nd0)];
    int32_t cn = dm1[(int64_t)cj * nd1 + (j % nd1)];
    if (rmap0) rn = rmap0[rn];
    if (rmap1) cn = rmap1[cn];
    int32_t v = -1;
    if (rn >= 0 && cn >= 0) {
      const int64_t g = off0 + (int64_t)bs0 * rn;
      const int32_t key = static_cast<int32_t>(off1 + (int64_t)bs1 * cn);
      const int64_t lo = row_ptr[g], hi = row_ptr[g + 1];
      const int64_t p = search(cols, lo, hi, key);
      if (p < hi && cols[p] == key) v = static_cast<int32_t>(p);
      else atomicAdd(missing, 1);
    }
    table[(e >> 6) * (int64_t)NI * NJ * 64 + (int64_t)ij * 64 + (e & 63)] = v;
  }
}

__global__ void lift_list_kernel(int32_t* __restrict__ list, int32_t* __restrict__ count,
                                 const int32_t* __restrict__ ents, int64_t nents, int stride,
                                 int ncell, const int32_t* __restrict__ dm1, int nd1, int bs1,
                                 const int8_t* __restrict__ bc1) {
  int64_t gs = (int64_t)gridDim.x * blockDim.x;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < nents; e += gs) {
    bool has = false;
    for (int ci = 0; ci < ncell && !has; ++ci) {
      int32_t c = ents[e * stride + 2 * ci];
      for (int j = 0; j < nd1 && !has; ++j) {
        int32_t node = dm1[(int64_t)c * nd1 + j];
        for (int b = 0; b < bs1; ++b) has |= bc1[(int64_t)bs1 * node + b] != 0;
      }
    }
    if (has) list[atomicAdd(count, 1)] = static_cast<int32_t>(e);
  }
}

// Workgroups land on the 8 XCDs in turn; with this order (grid a multiple of 64)
// each XCD takes eight contiguous runs of the rows, every eighth one, so most of
// the part of x that they share stays in its own L2.  One run per XCD left XCDs
// idle where the entries lie in one part of the rows (P2 20^3, first half of the
// cells: 7.9 us, 5.9 with eight runs; eighth in the middle of 28^3: 27.2 and 6.6);
// four and sixteen runs are within 5% of eight.
constexpr int kXcdRuns = 8;
__device__ __forceinline__ int64_t xcd_block() {
  const int64_t run = gridDim.x / (8 * kXcdRuns), w = blockIdx.x / 8;
  return (w / run * 8 + blockIdx.x % 8) * run + w % run;
}

// y = A x for a CSR matrix (int32 row_ptr / cols, FP64 values): G lanes per
// row (G a power of two <= 64, so a wave holds 64 / G rows); each lane sums a
// strided part of its row and the lanes of a row combine with shuffles, in a
// fixed order (repeated products are bit-identical).
template <int G, bool PAIRS>
__global__ void __launch_bounds__(kBlock) spmv_kernel(int64_t nrows, const int32_t* __restrict__ rp,
                                                      const int32_t* __restrict__ cols,
                                                      const double* __restrict__ v,
                                                      const double* __restrict__ x,
                                                      double* __restrict__ y) {
  // short rows: the x gathers weigh most (P1 50^3 7.3 us in launch order, 6.3 in
  // XCD order; DG1 32^3 47.7 and 43.5); long rows stream their values (Q3 24^3: 2%
  // slower)
  const int64_t wg = G <= 8 ? xcd_block() : (int64_t)blockIdx.x;
  const int64_t row = (wg * kBlock + threadIdx.x) / G;
  const int lane = threadIdx.x & (G - 1);
  double acc = 0.0;
  if (row < nrows) {
    const int32_t e = rp[row + 1];
    int32_t k = rp[row] + lane;
    if (PAIRS) for (; k + G < e; k += 2 * G) {
      const double v0 = v[k], v1 = v[k + G];
      const double x0 = x[cols[k]], x1 = x[cols[k + G]];
      acc += v0 * x0;
      acc += v1 * x1;
    }
    for (; k < e; k += G) acc += v[k] * x[cols[k]];
  }
  for (int o = G / 2; o > 0; o >>= 1) acc += __shfl_xor(acc, o, G);
  if (row < nrows && lane == 0) y[row] = acc;
}

// y = A x for the bs-unrolled CSR of a BS-component space: the BS scalar rows of
// a blocked row hold the same columns, whole nodes at a time, so G lanes take
// the blocked row together, each x value is loaded once for BS rows and the
// columns come from the blocked pattern, 4 bytes per BS x BS values instead of
// 4 per value.  Bound by memory: (8 + 4 / BS^2) bytes per value.
template <int BS, int G>
__global__ void __launch_bounds__(kBlock) spmv_block_kernel(int64_t nrows_b,
                                                            const int32_t* __restrict__ rpb,
                                                            const int32_t* __restrict__ colsb,
                                                            const double* __restrict__ v,
                                                            const double* __restrict__ x,
                                                            double* __restrict__ y) {
  const int64_t row = ((int64_t)blockIdx.x * kBlock + threadIdx.x) / G;
  const int lane = threadIdx.x & (G - 1);
  double acc[BS];
#pragma unroll
  for (int a = 0; a < BS; ++a) acc[a] = 0.0;
  if (row < nrows_b) {
    const int32_t s = rpb[row], n = BS * (rpb[row + 1] - s);
    const double* vr = v + (int64_t)BS * BS * s;
    int32_t t = lane;
    for (; t + G < n; t += 2 * G) {
      const int32_t u = t + G;
      const double xt = x[(int64_t)BS * colsb[s + t / BS] + t % BS];
      const double xu = x[(int64_t)BS * colsb[s + u / BS] + u % BS];
      double vt[BS], vu[BS];
#pragma unroll
      for (int a = 0; a < BS; ++a) {
        vt[a] = vr[(int64_t)a * n + t];
        vu[a] = vr[(int64_t)a * n + u];
      }
#pragma unroll
      for (int a = 0; a < BS; ++a) acc[a] = acc[a] + vt[a] * xt + vu[a] * xu;
    }
    if (t < n) {
      const double xt = x[(int64_t)BS * colsb[s + t / BS] + t % BS];
#pragma unroll
      for (int a = 0; a < BS; ++a) acc[a] += vr[(int64_t)a * n + t] * xt;
    }
  }
#pragma unroll
  for (int a = 0; a < BS; ++a)
    for (int o = G / 2; o > 0; o >>= 1) acc[a] += __shfl_xor(acc[a], o, G);
  if (row < nrows_b) {
#pragma unroll
    for (int a = 0; a < BS; ++a)
      if (lane == a) y[(int64_t)BS * row + a] = acc[a];
  }
}

template <int BS>
void spmv_block(int64_t nrows_b, int64_t nnz_b, const int32_t* rpb, const int32_t* colsb,
                const double* v, const double* x, double* y, hipStream_t s) {
  // lanes per blocked row: about three of its columns each
  const double mean = (double)BS * nnz_b / (double)nrows_b;
  const int g = mean > 96 ? 64 : (mean > 48 ? 32 : (mean > 24 ? 16 : 8));
  const int64_t threads = nrows_b * g;
  MF_CHECK(threads / kBlock < (1LL << 31) - 16, MF_ESHAPE, "matrix too large for one SpMV launch");
  const uint32_t grid = static_cast<uint32_t>((threads + kBlock - 1) / kBlock);
  switch (g) {
    case 8: spmv_block_kernel<BS, 8><<<grid, kBlock, 0, s>>>(nrows_b, rpb, colsb, v, x, y); break;
    case 16: spmv_block_kernel<BS, 16><<<grid, kBlock, 0, s>>>(nrows_b, rpb, colsb, v, x, y); break;
    case 32: spmv_block_kernel<BS, 32><<<grid, kBlock, 0, s>>>(nrows_b, rpb, colsb, v, x, y); break;
    default: spmv_block_kernel<BS, 64><<<grid, kBlock, 0, s>>>(nrows_b, rpb, colsb, v, x, y); break;
  }
  MF_HIP(hipGetLastError());
}

// d[r] = A[r][r] (0 where the pattern has no diagonal entry); columns sorted.
__global__ void diag_kernel(int64_t nrows, const int32_t* __restrict__ rp,
                            const int32_t* __restrict__ cols, const double* __restrict__ v,
                            double* __restrict__ d) {
  const int64_t stride = (int64_t)gridDim.x * kBlock;
  for (int64_t r = (int64_t)blockIdx.x * kBlock + threadIdx.x; r < nrows; r += stride) {
    int32_t lo = rp[r], hi = rp[r + 1];
    while (lo < hi) {
      const int32_t mid = (lo + hi) >> 1;
      if (cols[mid] < r) lo = mid + 1;
      else hi = mid;
    }
    d[r] = (lo < rp[r + 1] && cols[lo] == r) ? v[lo] : 0.0;
  }
}

}  // namespace

void k_fill(double* x, int64_t n, double v, hipStream_t s) {
  if (n <= 0) return;
  fill_kernel<<<grid_for(n, 4), kBlock, 0, s>>>(x, n, v);
  MF_HIP(hipGetLastError());
}
void k_scatter_add(double* dst, const double* src, const int32_t* map, int64_t n, hipStream_t s) {
  if (n <= 0) return;
  scatter_add_kernel<<<grid_for(n, 4), kBlock, 0, s>>>(dst, src, map, n);
  MF_HIP(hipGetLastError());
}
void k_fill_i32(int32_t* x, int64_t n, int32_t v, hipStream_t s) {
  if (n <= 0) return;
  fill_i32_kernel<<<grid_for(n, 4), kBlock, 0, s>>>(x, n, v);
  MF_HIP(hipGetLastError());
}
void k_sum_partials(const double* partials, int64_t n, double* out, int accumulate, hipStream_t s) {
  sum_partials_kernel<<<1, kBlock, 0, s>>>(partials, n, out, accumulate);
  MF_HIP(hipGetLastError());
}
void k_interpolate(double* u1, const double* u0, const int32_t* own, const int32_t* dm0,
                   const double* im, int64_t nnodes1, int n1, int n0, int bs, hipStream_t s) {
  const int64_t n = nnodes1 * bs;
  if (n <= 0) return;
  interp_kernel<<<grid_for(n), kBlock, 0, s>>>(u1, u0, own, dm0, im, n, n1, n0, bs);
  MF_HIP(hipGetLastError());
}
void k_build_block_table(int32_t* table, const int32_t* ents, int64_t nents, int stride, int ncell,
                         const int32_t* dm0, int nd0, const int32_t* rmap0, int64_t off0, int bs0,
                         const int32_t* dm1, int nd1, const int32_t* rmap1, int64_t off1, int bs1,
                         const int32_t* row_ptr, const int32_t* cols, int32_t* missing,
                         hipStream_t s) {
  const int64_t total = nents * (int64_t)ncell * nd0 * ncell * nd1;
  if (total <= 0) return;
  block_table_kernel<<<grid_for(total, 4), kBlock, 0, s>>>(table, ents, nents, stride, ncell, dm0,
                                                           nd0, rmap0, off0, bs0, dm1, nd1, rmap1,
                                                           off1, bs1, row_ptr, cols, missing);
  MF_HIP(hipGetLastError());
}
void k_mark(int8_t* m, int64_t ndofs, const int32_t* dofs, int64_t nbc, hipStream_t s) {
  if (nbc <= 0) return;
  mark_kernel<<<grid_for(nbc), kBlock, 0, s>>>(m, ndofs, dofs, nbc);
  MF_HIP(hipGetLastError());
}
void k_cell_flags(uint8_t* flags, const int32_t* dm, int64_t ncells, int nd, const uint8_t* bits,
                  hipStream_t s) {
  if (ncells <= 0) return;
  cell_flags_kernel<<<grid_for(ncells), kBlock, 0, s>>>(flags, dm, ncells, nd, bits);
  MF_HIP(hipGetLastError());
}
void k_node_bits(uint8_t* bits, const int8_t* m, int64_t nnodes, int bs, hipStream_t s) {
  if (nnodes <= 0) return;
  node_bits_kernel<<<grid_for(nnodes), kBlock, 0, s>>>(bits, m, nnodes, bs);
  MF_HIP(hipGetLastError());
}
// N: room for coefficients, m of them given
template <int N>
static void pack_launch(double* packed, int64_t ncells, int W, const PackItem* items, int m, hipStream_t s) {
  PackArgs<N> a;
  a.cum[0] = 0;
  for (int g = 0; g < N; ++g) {
    const PackItem q = g < m ? items[g] : PackItem{nullptr, nullptr, 0, 1, 0};
    a.values[g] = q.values;
    a.dofmap[g] = q.dofmap;
    a.nd[g] = q.nd;
    a.bs[g] = q.bs;
    a.off[g] = q.off;
    a.cum[g + 1] = a.cum[g] + q.nd * q.bs;
  }
  const int64_t total = ncells * a.cum[N];
  // (a thread's index past the last entry stays below total + the grid's threads)
  if (total < (int64_t(1) << 31)) pack_kernel<N, uint32_t><<<grid_for(total), kBlock, 0, s>>>(packed, ncells, W, a);
  else pack_kernel<N, int64_t><<<grid_for(total), kBlock, 0, s>>>(packed, ncells, W, a);
  MF_HIP(hipGetLastError());
}
void k_pack(double* packed, int64_t ncells, int W, const PackItem* items, int n, hipStream_t s) {
  if (ncells <= 0) return;
  for (int i0 = 0; i0 < n; i0 += kPack) {
    const int m = std::min(n - i0, kPack);
    switch (m) {
      case 1: pack_launch<1>(packed, ncells, W, items + i0, m, s); break;
      case 2: pack_launch<2>(packed, ncells, W, items + i0, m, s); break;
      case 3: pack_launch<3>(packed, ncells, W, items + i0, m, s); break;
      case 4: pack_launch<4>(packed, ncells, W, items + i0, m, s); break;
      default: pack_launch<kPack>(packed, ncells, W, items + i0, m, s);
    }
  }
}
void k_set_bc_batch(const SetBcGroup* groups, int ngroups, double scale, hipStream_t s) {
  MF_CHECK(ngroups >= 0 && ngroups <= 32, MF_EINVAL, "at most 32 vectors per set_bc batch");
  SetBcBatchArgs a{};
  a.ngroups = ngroups;
  a.start[0] = 0;
  for (int g = 0; g < ngroups; ++g) {
    a.b[g] = groups[g].b;
    a.dofs[g] = groups[g].dofs;
    a.g[g] = groups[g].g;
    a.n[g] = groups[g].n;
    a.start[g + 1] = a.start[g] + std::max<int64_t>(0, groups[g].nbc);
  }
  if (ngroups == 0 || a.start[ngroups] == 0) return;
  set_bc_batch_kernel<<<grid_for(a.start[ngroups]), kBlock, 0, s>>>(a, scale);
  MF_HIP(hipGetLastError());
}
void k_set_bc(double* b, int64_t n, const int32_t* dofs, int64_t nbc, const double* g,
              const double* x0, double scale, hipStream_t s) {
  if (nbc <= 0) return;
  set_bc_kernel<<<grid_for(nbc), kBlock, 0, s>>>(b, n, dofs, nbc, g, x0, scale);
  MF_HIP(hipGetLastError());
}
void k_set_diagonal(double* values, const int32_t* row_ptr, const int32_t* cols,
                    const int32_t* dofs, int64_t nbc, int64_t nrows, double diag, hipStream_t s) {
  if (nbc <= 0) return;
  set_diag_kernel<<<grid_for(nbc), kBlock, 0, s>>>(values, row_ptr, cols, dofs, nbc, nrows, diag);
  MF_HIP(hipGetLastError());
}
void k_unroll_cols(int32_t* cols, const int32_t* row_ptr, const int32_t* rpb, const int32_t* colsb,
                   int64_t nrows_b, int bs0, int bs1, hipStream_t s) {
  unroll_kernel<<<grid_for(nrows_b * 32), kBlock, 0, s>>>(cols, row_ptr, rpb, colsb, nrows_b, bs0,
                                                          bs1);
  MF_HIP(hipGetLastError());
}
void k_gather_plan(int32_t* count, int32_t* fill, const int32_t* ents, int64_t nents, int stride,
                   int ncell, const int32_t* dm0, int nd0, const int32_t* dm1, int nd1, int bs0,
                   int bs1, const int32_t* rpb, const int32_t* colsb, int32_t* missing,
                   hipStream_t s) {
  const int64_t total = nents * (int64_t)ncell * nd0 * ncell * nd1;
  if (total <= 0) return;
  gather_plan_kernel<<<grid_for(total, 4), kBlock, 0, s>>>(count, fill, ents, nents, stride, ncell,
                                                           dm0, nd0, dm1, nd1, bs0, bs1, rpb, colsb,
                                                           missing);
  MF_HIP(hipGetLastError());
}
void k_gather_sort(int32_t* fill, const int32_t* ptr, int2* pos, int64_t nq, int64_t nrows_b,
                   const int32_t* rpb, const int32_t* row_ptr, int bs0, int bs1, hipStream_t s) {
  if (nq <= 0) return;
  gather_sort_kernel<<<grid_for(nq), kBlock, 0, s>>>(fill, ptr, pos, nq, nrows_b, rpb, row_ptr, bs0,
                                                     bs1);
  MF_HIP(hipGetLastError());
}
void k_gather(double* values, const double* ws, const int32_t* ptr, const int32_t* at,
              const int2* pos, int64_t nq, int bs0, int bs1, int row_stride, hipStream_t s) {
  const int64_t n = nq * bs0 * bs1;
  if (n <= 0) return;
  const int64_t blocks = (n + kBlock - 1) / kBlock;
  gather_kernel<<<static_cast<uint32_t>((blocks + 7) / 8 * 8), kBlock, 0, s>>>(
      values, ws, ptr, at, pos, nq, bs0, bs1, row_stride);
  MF_HIP(hipGetLastError());
}
void k_build_table(int32_t* table, const int32_t* ents, int64_t nents, int stride, int ncell,
                   const int32_t* dm0, int nd0, const int32_t* dm1, int nd1, int bs0, int bs1,
                   const int32_t* row_ptr, const int32_t* rpb, const int32_t* colsb,
                   int32_t* missing, hipStream_t s) {
  if (nents <= 0) return;
  int64_t total = nents * ncell * nd0 * ncell * nd1;
  table_kernel<<<grid_for(total, 4), kBlock, 0, s>>>(table, ents, nents, stride, ncell, dm0, nd0,
                                                     dm1, nd1, bs0, bs1, row_ptr, rpb, colsb,
                                                     missing);
  MF_HIP(hipGetLastError());
}
// Scratch of the allocation-free lifting entry point (mf_apply_lifting_noalloc):
// scratch[0] counts the entities of the list in scratch[64 ..].  One copy per
// device, loaded with the library's code object and held until the process
// ends.  Host code never passes `scratch` itself to a kernel: its device
// address comes from hipGetSymbolAddress, looked up once per device.
static __device__ __align__(256) int32_t scratch[kLiftScratchEntities + 64];

namespace {
std::mutex g_scratch_mutex;
int32_t* g_scratch_ptr[kMaxScratchDevices] = {};
}  // namespace

void lift_scratch_init(int device) {
  MF_CHECK(device >= 0 && device < kMaxScratchDevices, MF_EUNSUPPORTED, "device index too large");
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (g_scratch_ptr[device]) return;
  int cur = -1;
  MF_HIP(hipGetDevice(&cur));
  MF_CHECK(cur == device, MF_ESTATE, "the scratch lookup needs its device current");
  void* ptr = nullptr;
  MF_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
  MF_CHECK(ptr != nullptr, MF_EHIP, "no device address for the lifting scratch");
  g_scratch_ptr[device] = static_cast<int32_t*>(ptr);
}

int32_t* lift_scratch(int device) {
  MF_CHECK(device >= 0 && device < kMaxScratchDevices, MF_EUNSUPPORTED, "device index too large");
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  MF_CHECK(g_scratch_ptr[device] != nullptr, MF_ESTATE,
           "lifting scratch not set up on this device (create a context first)");
  return g_scratch_ptr[device];
}

void k_lift_list(int32_t* list, int32_t* count, const int32_t* ents, int64_t nents, int stride,
                 int ncell, const int32_t* dm1, int nd1, int bs1, const int8_t* bc1,
                 hipStream_t s) {
  if (nents <= 0) return;
  lift_list_kernel<<<grid_for(nents), kBlock, 0, s>>>(list, count, ents, nents, stride, ncell, dm1,
                                                      nd1, bs1, bc1);
  MF_HIP(hipGetLastError());
}


void k_spmv(int64_t nrows, int64_t nnz, const int32_t* rp, const int32_t* cols, const double* v,
            const double* x, double* y, hipStream_t s) {
  if (nrows <= 0) return;
  // lanes per row from the mean row length (about three entries per lane); two
  // loads of a lane in flight, but one where a lane has no more than two of a row's
  // entries and the pair only splits them (P1 48^3 6.2 us in pairs, 5.3 singly; DG1
  // 32^3, 20 entries a row, 39.8 and 45.2)
  const double mean = (double)nnz / (double)nrows;
  int g = 2;
  while (g < 64 && g * 3 < mean) g *= 2;
  const int64_t threads = nrows * g;
  MF_CHECK(threads / kBlock < (1LL << 31) - 8 * kXcdRuns, MF_ESHAPE,
           "matrix too large for one SpMV launch");
  const uint32_t grid = static_cast<uint32_t>((threads + kBlock - 1) / kBlock + 8 * kXcdRuns - 1) /
                        (8 * kXcdRuns) * (8 * kXcdRuns);
  switch (g) {
    case 2: spmv_kernel<2, true><<<grid, kBlock, 0, s>>>(nrows, rp, cols, v, x, y); break;
    case 4: spmv_kernel<4, true><<<grid, kBlock, 0, s>>>(nrows, rp, cols, v, x, y); break;
    case 8:
      if (mean > 16) spmv_kernel<8, true><<<grid, kBlock, 0, s>>>(nrows, rp, cols, v, x, y);
      else spmv_kernel<8, false><<<grid, kBlock, 0, s>>>(nrows, rp, cols, v, x, y);
      break;
    case 16: spmv_kernel<16, true><<<grid, kBlock, 0, s>>>(nrows, rp, cols, v, x, y); break;
    case 32: spmv_kernel<32, true><<<grid, kBlock, 0, s>>>(nrows, rp, cols, v, x, y); break;
    default: spmv_kernel<64, true><<<grid, kBlock, 0, s>>>(nrows, rp, cols, v, x, y); break;
  }
  MF_HIP(hipGetLastError());
}

bool k_spmv_block(int bs0, int bs1, int64_t nrows_b, int64_t nnz_b, const int32_t* rpb,
                  const int32_t* colsb, const double* v, const double* x, double* y, hipStream_t s) {
  if (bs0 != bs1 || (bs0 != 2 && bs0 != 3)) return false;
  if (nrows_b <= 0) return true;
  if (bs0 == 2) spmv_block<2>(nrows_b, nnz_b, rpb, colsb, v, x, y, s);
  else spmv_block<3>(nrows_b, nnz_b, rpb, colsb, v, x, y, s);
  return true;
}

void k_diagonal(int64_t nrows, const int32_t* rp, const int32_t* cols, const double* v, double* d,
                hipStream_t s) {
  if (nrows <= 0) return;
  diag_kernel<<<grid_for(nrows), kBlock, 0, s>>>(nrows, rp, cols, v, d);
  MF_HIP(hipGetLastError());
}

}  // namespace mf
