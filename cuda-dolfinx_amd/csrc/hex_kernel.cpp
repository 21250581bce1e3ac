// Matrix-core owner-computes kernel for kappa grad.grad - k^2 mass on Q_k
// hexahedra with trilinear (non-affine) geometry (HIP template, hipRTC).
//
// Per cell and quadrature point q the operator is a 4 x 4 block
//   D_q = [[kappa w_q |J_q| K_q K_q^T, 0], [0, -k^2 w_q |J_q|]]
// so A_ij = sum_{q, a, b} B_a(q, i) D_q[a][b] B_b(q, j), B_a the reference
// gradient components (a = x, y, z) and values (a = 0).  Written as
//   A[(cell, i), j] = sum_k F[(cell, i), k] * Bt[k, j],  k = (q, b),
//   F[(cell, i), (q, b)] = sum_a B_a(q, i) D_q[a][b],    Bt[(q, b), j] = B_b(q, j),
// the right factor Bt is the same for every cell, so one 16-row MFMA tile can
// hold rows of different cells: the workgroup packs all (cell, owned row)
// pairs of its CSR row chunk densely into tiles (no padding), contracts them
// against Bt with v_mfma_*_16x16x* (K loop over the quadrature points) and
// accumulates the 16 x (k+1)^3 result rows in the LDS copy of the chunk's CSR
// values (FP64, ds_add_f64), which is written out once.
//
// Precision variants (compile-time MF_HX_PREC): 32 = FP32 operands and
// accumulation (v_mfma_f32_16x16x4f32), 16 = BF16 operands with FP32
// accumulation (v_mfma_f32_16x16x16bf16_1k), 64 = FP64 on the vector ALUs
// (same tiles and pair packing; on MI355X the FP64 vector and matrix peaks
// are equal, 78.6 TFLOP/s, so FP64 matrix cores offer no higher ceiling, and
// the vector ALUs can contract over x, y and z in turn, 4.6 times fewer
// multiply-adds than the dense contraction: Q3 on 24^3 cubes 1,215 -> 435 us,
// 370 with what the kernel's comment below names).
// Geometry (J, det, K), D_q, and the CSR accumulation are FP64 in all three.
//
// Operand layouts (16x16xK, lane l): A[row l%16][k-slot l/16], B[k-slot
// l/16][col l%16], result rows 4*(l/16)+r, column l%16 (the FP32-result
// instructions; v_mfma_f64_16x16x4f64 places its result rows at l/16 + 4r).  The K index is
// (q, b) with b fastest, so one K-slot block covers one quadrature point.
#include "mf_internal.h"

namespace mf {

// Constrained columns of every cell as bits (bit j: local node j), for the
// assembly that follows: one wave per cell, lane = local node.
const char* kHexPrepTemplate = R"(
extern "C" __global__ void __launch_bounds__(256)
$KNAME(const int32_t n, const int32_t* __restrict__ ents, const int32_t* __restrict__ dm0,
       const uint8_t* __restrict__ nb0, uint64_t* __restrict__ cmask)
{
  static_assert(HX_ND == 64, "one lane per local node");
  const int e = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (e >= n) return;
  const int64_t c = ents[e];
  const uint64_t bits = __ballot(nb0[dm0[c * 64 + (threadIdx.x & 63)]] != 0);
  if ((threadIdx.x & 63) == 0) cmask[c] = bits;
}
)";

// Lifting over the hexahedra that touch a constrained dof: the element matrix
// is applied to the values to lift, v_j = scale (g_j - x0_j) at constrained
// columns and 0 elsewhere, without being formed.  One wave per listed cell:
// the gradient and the value of sum_j v_j phi_j at the quadrature points by
// contractions over x, y and z in turn, D_q applied at each point, and the
// transposed contractions back to the rows; stages pass through LDS.  About
// 5 thousand multiply-adds per cell at Q3 with 4 points per direction, against
// the 64 x 64 x 64 x 4 of the element tensor that the per-entity kernel builds
// in 34 KB of scratch per thread: 3,176 boundary cells (24^3 Q3) 86.6 ms
// with that kernel, 8.5 us here.  Bound by latency and by its FP64 atomics into
// b (25 G/s).
const char* kHexLiftTemplate = R"(
extern "C" __global__ void __launch_bounds__(64)
$KNAME(const int32_t nlist, const int32_t* __restrict__ nlist_dev, const int32_t* __restrict__ list,
       const int32_t* __restrict__ ents, const int32_t* __restrict__ geo,
       const double* __restrict__ xg, const int32_t* __restrict__ dm,
       const int8_t* __restrict__ bc1, const double* __restrict__ g,
       const double* __restrict__ x0, const double scale, double* __restrict__ b)
{
  constexpr int K1 = HX_K + 1, ND = HX_ND, M1 = HX_NQ1, NQ = M1 * M1 * M1;
  if ((int)blockIdx.x >= (nlist_dev ? *nlist_dev : nlist)) return;
  __shared__ double sx[24], sL[M1 * K1], sG[M1 * K1], sv[ND];
  __shared__ double a0[M1 * K1 * K1], a1[M1 * K1 * K1];             // x done: value, x-derivative
  __shared__ double bv[M1 * M1 * K1], bx[M1 * M1 * K1], by[M1 * M1 * K1];   // x and y done
  __shared__ double f0[NQ], f1[NQ], f2[NQ], f3[NQ];                 // D_q (gradient, value)
  const int lane = threadIdx.x;
  const int64_t c = ents[list[blockIdx.x]];
  for (int p = lane; p < M1 * K1; p += 64) {
    sL[p] = HX_L[p / K1][p % K1];
    sG[p] = HX_DL[p / K1][p % K1];
  }
  if (lane < 24) sx[lane] = xg[3 * (int64_t)geo[c * 8 + lane / 3] + lane % 3];
  for (int p = lane; p < ND; p += 64) {
    const int64_t col = dm[c * ND + p];
    sv[p] = bc1[col] ? scale * (g[col] - (x0 ? x0[col] : 0.0)) : 0.0;
  }
  __syncthreads();
  for (int p = lane; p < M1 * K1 * K1; p += 64) {
    const int q1 = p % M1, jj = p / M1;                             // jj = jb + K1 jc
    double u = 0.0, ux = 0.0;
    for (int j = 0; j < K1; ++j) {
      const double v = sv[j + K1 * jj];
      u += sL[q1 * K1 + j] * v;
      ux += sG[q1 * K1 + j] * v;
    }
    a0[p] = u;
    a1[p] = ux;
  }
  __syncthreads();
  for (int p = lane; p < M1 * M1 * K1; p += 64) {
    const int q1 = p % M1, q2 = (p / M1) % M1, jc = p / (M1 * M1);
    double u = 0.0, ux = 0.0, uy = 0.0;
    for (int j = 0; j < K1; ++j) {
      const int s = q1 + M1 * (j + K1 * jc);
      u += sL[q2 * K1 + j] * a0[s];
      ux += sL[q2 * K1 + j] * a1[s];
      uy += sG[q2 * K1 + j] * a0[s];
    }
    bv[p] = u;
    bx[p] = ux;
    by[p] = uy;
  }
  __syncthreads();
  for (int p = lane; p < NQ; p += 64) {
    const int q1 = p % M1, q2 = (p / M1) % M1, q3 = p / (M1 * M1);
    double u = 0.0, ux = 0.0, uy = 0.0, uz = 0.0;
    for (int j = 0; j < K1; ++j) {
      const int s = q1 + M1 * (q2 + M1 * j);
      u += sL[q3 * K1 + j] * bv[s];
      ux += sL[q3 * K1 + j] * bx[s];
      uy += sL[q3 * K1 + j] * by[s];
      uz += sG[q3 * K1 + j] * bv[s];
    }
    // trilinear geometry at this point (as in the matrix kernel)
    const double X = HX_X1[q1], Y = HX_X1[q2], Z = HX_X1[q3];
    double J[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
    for (int v = 0; v < 8; ++v) {
      const int a = v & 1, bb = (v >> 1) & 1, cc = v >> 2;
      const double fx = a ? X : 1 - X, fy = bb ? Y : 1 - Y, fz = cc ? Z : 1 - Z;
      const double d0 = (a ? 1.0 : -1.0) * fy * fz, d1 = fx * (bb ? 1.0 : -1.0) * fz;
      const double d2 = fx * fy * (cc ? 1.0 : -1.0);
      for (int i = 0; i < 3; ++i) {
        const double xv = sx[3 * v + i];
        J[i][0] += xv * d0; J[i][1] += xv * d1; J[i][2] += xv * d2;
      }
    }
    const double m00 = J[1][1] * J[2][2] - J[1][2] * J[2][1];
    const double m01 = J[0][2] * J[2][1] - J[0][1] * J[2][2];
    const double m02 = J[0][1] * J[1][2] - J[0][2] * J[1][1];
    const double det = J[0][0] * m00 + J[1][0] * m01 + J[2][0] * m02;
    const double id = 1.0 / det;
    double K[3][3];
    K[0][0] = m00 * id; K[0][1] = m01 * id; K[0][2] = m02 * id;
    K[1][0] = (J[1][2] * J[2][0] - J[1][0] * J[2][2]) * id;
    K[1][1] = (J[0][0] * J[2][2] - J[0][2] * J[2][0]) * id;
    K[1][2] = (J[0][2] * J[1][0] - J[0][0] * J[1][2]) * id;
    K[2][0] = (J[1][0] * J[2][1] - J[1][1] * J[2][0]) * id;
    K[2][1] = (J[0][1] * J[2][0] - J[0][0] * J[2][1]) * id;
    K[2][2] = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) * id;
    const double wq = HX_W1[q1] * HX_W1[q2] * HX_W1[q3] * fabs(det);
    const double s = HX_KAPPA * wq;
    // physical gradient K^T u, back to reference components K (K^T u)
    const double gx = K[0][0] * ux + K[1][0] * uy + K[2][0] * uz;
    const double gy = K[0][1] * ux + K[1][1] * uy + K[2][1] * uz;
    const double gz = K[0][2] * ux + K[1][2] * uy + K[2][2] * uz;
    f0[p] = s * (K[0][0] * gx + K[0][1] * gy + K[0][2] * gz);
    f1[p] = s * (K[1][0] * gx + K[1][1] * gy + K[1][2] * gz);
    f2[p] = s * (K[2][0] * gx + K[2][1] * gy + K[2][2] * gz);
    f3[p] = -HX_K2 * wq * u;
  }
  __syncthreads();
  for (int p = lane; p < M1 * M1 * K1; p += 64) {
    const int q1 = p % M1, q2 = (p / M1) % M1, ic = p / (M1 * M1);
    double r = 0.0, rx = 0.0, ry = 0.0;
    for (int q = 0; q < M1; ++q) {
      const int s = q1 + M1 * (q2 + M1 * q);
      r += sG[q * K1 + ic] * f2[s] + sL[q * K1 + ic] * f3[s];
      rx += sL[q * K1 + ic] * f0[s];
      ry += sL[q * K1 + ic] * f1[s];
    }
    bv[p] = r;
    bx[p] = rx;
    by[p] = ry;
  }
  __syncthreads();
  for (int p = lane; p < M1 * K1 * K1; p += 64) {
    const int q1 = p % M1, ib = (p / M1) % K1, ic = p / (M1 * K1);
    double r = 0.0, rx = 0.0;
    for (int q = 0; q < M1; ++q) {
      const int s = q1 + M1 * (q + M1 * ic);
      r += sG[q * K1 + ib] * by[s] + sL[q * K1 + ib] * bv[s];
      rx += sL[q * K1 + ib] * bx[s];
    }
    a0[p] = r;
    a1[p] = rx;
  }
  __syncthreads();
  for (int p = lane; p < ND; p += 64) {
    const int ia = p % K1, ii = p / K1;
    double r = 0.0;
    for (int q = 0; q < M1; ++q)
      r += sG[q * K1 + ia] * a1[q + M1 * ii] + sL[q * K1 + ia] * a0[q + M1 * ii];
    atomicAdd(&b[dm[c * ND + p]], -r);
  }
}
)";

// Source f v (f constant) on hexahedra in blocks of consecutive cells (the
// blocks, LDS sums and row atomics of mf_vblk_*): one wave per cell, its lanes
// the quadrature points, and the transposed contraction
//   b_abc = sum_q3 L(q3,c) sum_q2 L(q2,b) sum_q1 L(q1,a) f w |det J|
// over x, y and z in turn through LDS: at Q3 with 4 points per direction 12
// multiply-adds per lane after the geometry, where one thread per cell has
// 64 x 64 and the geometry of 64 points (13,824 cells, 216 waves for 1,024
// SIMDs).  Bound by latency: the chain entity -> vertices -> coordinates, loaded
// for the whole block at once, and the row atomics.  24^3 Q3, 389
// thousand rows: 79 -> 14 us.
const char* kHexSourceTemplate = R"(
extern "C" __global__ void __launch_bounds__(256)
$KNAME(const int32_t nblk, const int32_t* __restrict__ blk_ent, const int32_t* __restrict__ blk_ptr,
       const int32_t* __restrict__ blk_row, const uint16_t* __restrict__ slot,
       const int32_t* __restrict__ ents, const int32_t* __restrict__ geo,
       const double* __restrict__ xg, const double* __restrict__ coeffs,
       const double* __restrict__ consts, double* __restrict__ b)
{
  constexpr int K1 = HX_K + 1, ND = HX_ND, M1 = HX_NQ1, NQ = M1 * M1 * M1;
  constexpr int S0 = NQ > M1 * K1 * K1 ? NQ : M1 * K1 * K1;         // stage 0 and 2
  extern __shared__ double mf_acc[];
  __shared__ double sL[M1 * K1], sx[$HSC * 24];
  __shared__ double st[4][S0 + M1 * M1 * K1];
  const int k = mf_xcd_chunk(nblk);
  if (k < 0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int e0 = blk_ent[k], ne = blk_ent[k + 1] - e0, r0 = blk_ptr[k], len = blk_ptr[k + 1] - r0;
  for (int p = tid; p < ne * 24; p += 256)
    sx[p] = xg[3 * (int64_t)geo[(int64_t)ents[e0 + p / 24] * 8 + p % 24 / 3] + p % 3];
  for (int p = tid; p < M1 * K1; p += 256) sL[p] = HX_L[p / K1][p % K1];
  for (int p = tid; p < len; p += 256) mf_acc[p] = 0.0;
  const double fc = consts[HS_C];
  __syncthreads();
  double* A = st[wave];
  double* B = A + S0;
  for (int e = wave; e < ne; e += 4) {
    const uint16_t* sl = slot + (int64_t)(e0 + e) * ND;
    for (int p = lane; p < NQ; p += 64) {
      const int q1 = p % M1, q2 = (p / M1) % M1, q3 = p / (M1 * M1);
      const double X = HX_X1[q1], Y = HX_X1[q2], Z = HX_X1[q3];
      double J[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
#pragma unroll
      for (int v = 0; v < 8; ++v) {
        const double fx = v & 1 ? X : 1 - X, fy = v & 2 ? Y : 1 - Y, fz = v & 4 ? Z : 1 - Z;
        const double d0 = (v & 1 ? 1.0 : -1.0) * fy * fz, d1 = fx * (v & 2 ? 1.0 : -1.0) * fz;
        const double d2 = fx * fy * (v & 4 ? 1.0 : -1.0);
        for (int i = 0; i < 3; ++i) {
          const double xv = sx[24 * e + 3 * v + i];
          J[i][0] += xv * d0; J[i][1] += xv * d1; J[i][2] += xv * d2;
        }
      }
      const double det = J[0][0] * (J[1][1] * J[2][2] - J[1][2] * J[2][1])
                       + J[1][0] * (J[0][2] * J[2][1] - J[0][1] * J[2][2])
                       + J[2][0] * (J[0][1] * J[1][2] - J[0][2] * J[1][1]);
      A[p] = HX_W1[q1] * HX_W1[q2] * HX_W1[q3] * fabs(det) * fc;
    }
    // a wave's LDS accesses stay in order; the fences keep the compiler's too
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    for (int p = lane; p < M1 * M1 * K1; p += 64) {                 // over z
      const int q12 = p % (M1 * M1), c = p / (M1 * M1);
      double r = 0.0;
      for (int q = 0; q < M1; ++q) r += sL[q * K1 + c] * A[q12 + M1 * M1 * q];
      B[p] = r;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    for (int p = lane; p < M1 * K1 * K1; p += 64) {                 // over y
      const int q1 = p % M1, bb = (p / M1) % K1, c = p / (M1 * K1);
      double r = 0.0;
      for (int q = 0; q < M1; ++q) r += sL[q * K1 + bb] * B[q1 + M1 * (q + M1 * c)];
      A[p] = r;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    for (int p = lane; p < ND; p += 64) {                           // over x
      double r = 0.0;
      for (int q = 0; q < M1; ++q) r += sL[q * K1 + p % K1] * A[q + M1 * (p / K1)];
      atomicAdd(&mf_acc[sl[p]], r);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");          // A is written again
  }
  __syncthreads();
  for (int p = tid; p < len; p += 256) atomicAdd(&b[blk_row[r0 + p]], mf_acc[p]);
}
)";

const char* kHexOwnerTemplate = R"(
#if MF_HX_PREC == 64
// Sums over the four 16-lane rows of a wave, each row keeping another value:
// v_permlane32_swap exchanges a's upper half with b's lower half, so the sum
// of the two results is a's (lower lanes) and b's (upper lanes) total over the
// halves; v_permlane16_swap does the same for odd and even rows.
static __device__ __forceinline__ double mf_swap_add32(double a, double b)
{
  const auto l = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
  const auto h = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
  return __hiloint2double(h[0], l[0]) + __hiloint2double(h[1], l[1]);
}
static __device__ __forceinline__ double mf_swap_add16(double a, double b)
{
  const auto l = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
  const auto h = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
  return __hiloint2double(h[0], l[0]) + __hiloint2double(h[1], l[1]);
}
#endif
#if MF_HX_PREC == 16
typedef short mf_bf4 __attribute__((ext_vector_type(4)));
static __device__ __forceinline__ short mf_to_bf16(float f)
{
  // round to nearest even
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (short)(u >> 16);
}
#endif


extern "C" __global__ void __launch_bounds__($HBLOCK)
#if MF_HX_PREC != 64
__attribute__((amdgpu_waves_per_eu(4)))                // two workgroups of eight waves per CU
#endif
$KNAME(const int32_t nchunks, const int32_t* __restrict__ chunk_meta,
       const int32_t* __restrict__ item_cell, const int32_t* __restrict__ item_geo,
       const int32_t* __restrict__ pair_list, const uint16_t* __restrict__ pair_pos,
       const double* __restrict__ xg, const uint64_t* __restrict__ cmask,
       const int32_t* __restrict__ rpb,
       const int32_t* __restrict__ diag_pos, const uint8_t* __restrict__ nb0,
       double* __restrict__ values, const double diag, const int flags)
{
  constexpr int K1 = HX_K + 1, ND = HX_ND, M1 = HX_NQ1, NQ = M1 * M1 * M1;
  constexpr int NB = $HNB, CAP = $OCAP, MAXR = $OMAXR, MAXP = $OMAXP;
  constexpr int DS = 8;                              // D_q record: G00 G01 G02 G11 G12 G22 M pad
#if MF_HX_PREC == 64
  typedef double real;
  // planes of 16 points 130 doubles apart and cells 520: the four planes and
  // four cells that a wave reads at once lie in different LDS banks
  constexpr int DCELL = 520;
#define MF_DOFF(b, q) ((b) * DCELL + ((q) >> 4) * 130 + ((q) & 15) * DS)
#else
  typedef float real;
  constexpr int DCELL = NQ * DS;
#define MF_DOFF(b, q) ((b) * DCELL + (q) * DS)
#endif
  __shared__ __attribute__((aligned(16))) double acc[(CAP + 1) / 2 * 2];
  __shared__ int32_t lrp[MAXR + 1];
  __shared__ double sx[NB * 24];                     // vertex coordinates of the batch's cells
  __shared__ uint64_t smask[NB];                     // their constrained columns
  __shared__ __attribute__((aligned(16))) real sD[NB * DCELL];
  __shared__ int32_t spair[MAXP];
  // 1D basis values / derivatives at the 1D points, [q][n], in LDS: the
  // contraction reads them with lane-dependent n, which from constant memory
  // would be a global load (and a wait) per quadrature line
  __shared__ real sTL[M1 * K1], sTD[M1 * K1];

  // Persistent: the grid holds the resident workgroups (a multiple of 8); those
  // of XCD blockIdx % 8 walk its contiguous eighth of the chunks with stride
  // gridDim / 8.  Everything the next step (the chunk's next batch of cells, or
  // the next chunk) reads from memory is loaded into registers while this one
  // computes, its dependent loads issued a phase apart, and the accumulator is
  // cleared by the write-out.  24^3 cells, 47 M values, 0.38 GB: 370 us (FP64),
  // 510 us (FP32; 470 with chunks that end at full rounds of tiles) against 390
  // and 520 us with one workgroup per chunk, and 436 and 518 us when the
  // coordinates and dofs came from 464-byte cell records, rows were searched in
  // chunks and chunks were filled up.  What is left is the
  // arithmetic of the 4-5 tiles of a chunk (FP64 about 140 us of issue, FP32
  // 190 us of MFMA) and the geometry in two workgroups' phases per CU.
  constexpr int NTH = $HBLOCK;
  constexpr int PFX = (NB * 24 + NTH - 1) / NTH, PFP = (MAXP + NTH - 1) / NTH;
  constexpr int PFB = (NB + NTH - 1) / NTH, PFR = (MAXR + NTH) / NTH;   // one each unless a caller's shape has more
  const int tid = threadIdx.x, nt = NTH;
  const int lane = tid & 63, wave = tid >> 6, nwave = NTH >> 6;
  const int nx = 8, gx = gridDim.x / nx, per = (nchunks + nx - 1) / nx;
  const int kend = min(nchunks, ((int)blockIdx.x % nx + 1) * per);
  int k = ((int)blockIdx.x % nx) * per + (int)blockIdx.x / nx;
  if (k >= kend) return;
  const int4* meta = reinterpret_cast<const int4*>(chunk_meta);
  int4 m0 = meta[3 * k], m1 = meta[3 * k + 1], m2 = meta[3 * k + 2];
  if (tid < M1 * K1) {                                 // 16 of at least 64 threads
#if MF_HX_PREC == 64
    sTL[tid] = HX_L[tid / K1][tid % K1];
    sTD[tid] = HX_DL[tid / K1][tid % K1];
#else
    sTL[tid] = HX_LF[tid / K1][tid % K1];
    sTD[tid] = HX_DLF[tid / K1][tid % K1];
#endif
  }
  {
    mf_d2* a2 = reinterpret_cast<mf_d2*>(acc);
    const mf_d2 z = {0.0, 0.0};
    for (int p = tid; p < (CAP + 1) / 2; p += nt) a2[p] = z;
  }
  // registers of the step ahead: vertices (1), then coordinates and constrained
  // columns (2) of its cells; for a chunk also its pairs and its rows (row tid, ...)
  int pfv[PFX], pfc[PFB], pfp[PFP], pfr[PFR], pfd[PFR];
  double pfx[PFX];
  uint64_t pfm[PFB];
  auto fetch1 = [&](const int ib, const int nb, const int tid) {
#pragma clang loop unroll(full)
    for (int t = 0; t < PFX; ++t)                      // clamped, unconditional loads stay in registers
      pfv[t] = item_geo[(int64_t)ib * 8 + min(tid + t * NTH, max(nb * 24 - 1, 0)) / 3];
#pragma clang loop unroll(full)
    for (int t = 0; t < PFB; ++t)                      // (the lists are padded by one cell and pair)
      pfc[t] = item_cell[ib + min(tid + t * NTH, max(nb - 1, 0))];
  };
  auto fetch2 = [&](const int nb, const int tid) {
#pragma clang loop unroll(full)
    for (int t = 0; t < PFX; ++t)
      pfx[t] = xg[3 * (int64_t)pfv[t] + min(tid + t * NTH, max(nb * 24 - 1, 0)) % 3];
#pragma clang loop unroll(full)
    for (int t = 0; t < PFB; ++t) pfm[t] = cmask ? cmask[pfc[t]] : 0;
  };
  auto fetch_rows = [&](const int4 c0, const int4 c1, const int4 c2, const int tid) {
#pragma clang loop unroll(full)
    for (int t = 0; t < PFP; ++t) pfp[t] = pair_list[max(min(c2.x + tid + t * NTH, c2.y - 1), c2.x)];
#pragma clang loop unroll(full)
    for (int t = 0; t < PFR; ++t) {
      const int u = c0.x + tid + t * NTH;
      pfr[t] = rpb[min(u, c0.y)] - c1.x;               // rpb[c0.y] closes the last row
      // Dirichlet rows: position of their diagonal entry (-1: none)
      const int row = min(u, c0.y - 1);
      const int dp = diag_pos[row];
      const bool on = (flags & 2) && nb0 && nb0[row];
      pfd[t] = on && u < c0.y ? dp : -1;
    }
  };
  auto store_cells = [&](const int nb) {
#pragma clang loop unroll(full)
    for (int t = 0; t < PFX; ++t) {
      const int u = tid + t * NTH;
      if (u < nb * 24) sx[u] = pfx[t];
    }
#pragma clang loop unroll(full)
    for (int t = 0; t < PFB; ++t)
      if (tid + t * NTH < nb) smask[tid + t * NTH] = pfm[t];
  };
  auto store_rows = [&](const int4 c0, const int4 c2) {
#pragma clang loop unroll(full)
    for (int t = 0; t < PFP; ++t) {
      const int u = tid + t * NTH;
      if (u < c2.y - c2.x) spair[u] = pfp[t];
    }
#pragma clang loop unroll(full)
    for (int t = 0; t < PFR; ++t) {
      const int u = tid + t * NTH;
      if (u <= c0.y - c0.x) lrp[u] = pfr[t];
      // constrained rows get no contributions (their pairs are masked), so their
      // diagonal is set up front
      if (pfd[t] >= 0) acc[pfr[t] + pfd[t]] = diag;
    }
  };
  fetch1(m0.z, min(NB, m0.w - m0.z), tid);
  fetch_rows(m0, m1, m2, tid);
  fetch2(min(NB, m0.w - m0.z), tid);
  __syncthreads();                                     // accumulator cleared before a diagonal goes in
  store_cells(min(NB, m0.w - m0.z));
  store_rows(m0, m2);

  while (true) {
  const int32_t i0 = m0.z, i1 = m0.w, base = m1.z, seglen = m1.w, p0 = m2.x;
  const int npc = m2.y - m2.x;
  const int kn = k + gx;
  const bool more = kn < kend;
  const int4 n0 = meta[3 * (more ? kn : k)], n1 = meta[3 * (more ? kn : k) + 1], n2 = meta[3 * (more ? kn : k) + 2];
  int pb = 0;
  for (int ib = i0;; ib += NB) {                       // a chunk without cells takes one empty batch
    const int nb = min(NB, i1 - ib);
    const bool last = ib + NB >= i1;
    // the step ahead: its first item and how many cells it takes
    const int ibx = last ? n0.z : ib + NB, nbx = min(NB, (last ? n0.w : i1) - ibx);
    if (ib > i0) {
      __syncthreads();                                 // previous batch done with sx / sD
      store_cells(nb);
    }
    __syncthreads();                                   // lists and cells visible
    // the batch's serial part (pair range, FP64 geometry) holds every wave of
    // this workgroup at the next barrier, so it issues at a raised priority
    // over the other workgroup's contraction
    __builtin_amdgcn_s_setprio(2);
    int tid_ = tid;
#if MF_HX_PREC != 64
    // a thread's quadrature point is the same in every batch: keep the compiler
    // from holding what depends on it alone (24 basis derivatives) in registers
    // across the contraction, which would leave room for one workgroup per CU
    asm volatile("" : "+v"(tid_));
#endif
    fetch1(ibx, nbx, tid_);
    int pe;
    {
      int lo2 = pb, hi2 = npc;
      const int lim = ib - i0 + nb;
      while (lo2 < hi2) {
        const int mid = (lo2 + hi2) >> 1;
        if ((spair[mid] >> 16) < lim) lo2 = mid + 1;
        else hi2 = mid;
      }
      pe = lo2;
    }
    // geometry: D_q for every (cell, quadrature point), FP64
    for (int u = tid_; u < nb * NQ; u += nt) {
      const int b = u / NQ, q = u - b * NQ;
      const int q1 = q % M1, q2 = (q / M1) % M1, q3 = q / (M1 * M1);
      const double X = HX_X1[q1], Y = HX_X1[q2], Z = HX_X1[q3];
      double J[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
      for (int v = 0; v < 8; ++v) {
        const int a = v & 1, bb = (v >> 1) & 1, c = v >> 2;
        const double fx = a ? X : 1 - X, fy = bb ? Y : 1 - Y, fz = c ? Z : 1 - Z;
        const double gx = a ? 1.0 : -1.0, gy = bb ? 1.0 : -1.0, gz = c ? 1.0 : -1.0;
        const double d0 = gx * fy * fz, d1 = fx * gy * fz, d2 = fx * fy * gz;
        for (int i = 0; i < 3; ++i) {
          const double xv = sx[b * 24 + 3 * v + i];
          J[i][0] += xv * d0; J[i][1] += xv * d1; J[i][2] += xv * d2;
        }
      }
      const double m00 = J[1][1] * J[2][2] - J[1][2] * J[2][1];
      const double m01 = J[0][2] * J[2][1] - J[0][1] * J[2][2];
      const double m02 = J[0][1] * J[1][2] - J[0][2] * J[1][1];
      const double det = J[0][0] * m00 + J[1][0] * m01 + J[2][0] * m02;
      const double id = 1.0 / det;
      double K[3][3];
      K[0][0] = m00 * id; K[0][1] = m01 * id; K[0][2] = m02 * id;
      K[1][0] = (J[1][2] * J[2][0] - J[1][0] * J[2][2]) * id;
      K[1][1] = (J[0][0] * J[2][2] - J[0][2] * J[2][0]) * id;
      K[1][2] = (J[0][2] * J[1][0] - J[0][0] * J[1][2]) * id;
      K[2][0] = (J[1][0] * J[2][1] - J[1][1] * J[2][0]) * id;
      K[2][1] = (J[0][1] * J[2][0] - J[0][0] * J[2][1]) * id;
      K[2][2] = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) * id;
      const double wq = HX_W1[q1] * HX_W1[q2] * HX_W1[q3] * fabs(det);
      const double s = HX_KAPPA * wq;
      real* D = &sD[MF_DOFF(b, q)];
      D[0] = (real)(s * (K[0][0] * K[0][0] + K[0][1] * K[0][1] + K[0][2] * K[0][2]));
      D[1] = (real)(s * (K[0][0] * K[1][0] + K[0][1] * K[1][1] + K[0][2] * K[1][2]));
      D[2] = (real)(s * (K[0][0] * K[2][0] + K[0][1] * K[2][1] + K[0][2] * K[2][2]));
      D[3] = (real)(s * (K[1][0] * K[1][0] + K[1][1] * K[1][1] + K[1][2] * K[1][2]));
      D[4] = (real)(s * (K[1][0] * K[2][0] + K[1][1] * K[2][1] + K[1][2] * K[2][2]));
      D[5] = (real)(s * (K[2][0] * K[2][0] + K[2][1] * K[2][1] + K[2][2] * K[2][2]));
      D[6] = (real)(-HX_K2 * wq);
      D[7] = (real)0;
    }
    if (last) fetch_rows(n0, n1, n2, tid_);
    fetch2(nbx, tid_);
    __syncthreads();
    __builtin_amdgcn_s_setprio(0);
    // contraction: one wave per 16-pair tile, all 64 columns (4 tiles of 16)
    const int np = pe - pb;
    const int ntile = (np + 15) / 16;
    const int r = lane & 15, slot = lane >> 4;      // A row / K slot of this lane
    for (int t = wave; t < ntile; t += nwave) {
      const int pr = t * 16 + r;
      const bool valid = pr < np;
      const int pc = pb + (valid ? pr : 0);
      const int b = (spair[pc] >> 16) - (ib - i0), i = spair[pc] & 63;
      const int ia = i % K1, ib2 = (i / K1) % K1, ic = i / (K1 * K1);
#if MF_HX_PREC != 64
      const real* Db = &sD[b * DCELL];
#endif
#if MF_HX_PREC == 64
      // FP64 on the vector ALUs, sum-factorised: lane = (tile row r, slot).
      // The slot is the plane q3 of quadrature points whose row factors this
      // lane forms and contracts over x and y with all 16 (ja, jb), then the
      // column block jc whose sum over the planes it keeps:
      //   w[ja]     = sum_q1 F_x X' + F_m X,  F_y X,  F_z X
      //   YL[ja,jb] = sum_q2 w_xm Y + w_y Y',  YG = sum_q2 w_z Y
      //   A[ja,jb,jc] = sum_q3 YL Z + YG Z'
      // About 950 multiply-adds per row and lane against 4,350 when every
      // column's quadrature sum runs over all 64 points.
      const int jc = slot;
      // row-relative column positions of this pair (precomputed), 32 bytes,
      // loaded ahead of the arithmetic
      const uint4* pp = reinterpret_cast<const uint4*>(pair_pos + ((int64_t)p0 + pc) * ND + 16 * jc);
      const uint4 w0 = pp[0], w1 = pp[1];
      double Lx[4], Gx[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        Lx[m] = sTL[m * K1 + ia];
        Gx[m] = sTD[m * K1 + ia];
      }
      const double Lz = sTL[slot * K1 + ic], Gz = sTD[slot * K1 + ic];
      double YL[16], YG[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) YL[k] = YG[k] = 0.0;
      const double* Ds = &sD[MF_DOFF(b, 16 * slot)];
#pragma unroll
      for (int q2 = 0; q2 < 4; ++q2) {
        const double Ly = sTL[q2 * K1 + ib2], Gy = sTD[q2 * K1 + ib2];
        const double LyLz = Ly * Lz, GyLz = Gy * Lz, LyGz = Ly * Gz;
        double wx[4] = {0, 0, 0, 0}, wy[4] = {0, 0, 0, 0}, wz[4] = {0, 0, 0, 0};
#pragma unroll
        for (int q1 = 0; q1 < 4; ++q1) {
          const double* D = Ds + (q1 + 4 * q2) * DS;
          const double Bx = Gx[q1] * LyLz, By = Lx[q1] * GyLz, Bz = Lx[q1] * LyGz;
          const double fx = Bx * D[0] + By * D[1] + Bz * D[2];
          const double fy = Bx * D[1] + By * D[3] + Bz * D[4];
          const double fz = Bx * D[2] + By * D[4] + Bz * D[5];
          const double fm = Lx[q1] * LyLz * D[6];
#pragma unroll
          for (int ja = 0; ja < 4; ++ja) {
            wx[ja] += fx * HX_DL[q1][ja] + fm * HX_L[q1][ja];
            wy[ja] += fy * HX_L[q1][ja];
            wz[ja] += fz * HX_L[q1][ja];
          }
        }
#pragma unroll
        for (int jb = 0; jb < 4; ++jb)
#pragma unroll
          for (int ja = 0; ja < 4; ++ja) {
            YL[ja + 4 * jb] += wx[ja] * HX_L[q2][jb] + wy[ja] * HX_DL[q2][jb];
            YG[ja + 4 * jb] += wz[ja] * HX_L[q2][jb];
          }
      }
      double Zl[4], Zd[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        Zl[m] = sTL[slot * K1 + m];
        Zd[m] = sTD[slot * K1 + m];
      }
      double cacc[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        double z[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) z[m] = YL[k] * Zl[m] + YG[k] * Zd[m];
        cacc[k] = mf_swap_add16(mf_swap_add32(z[0], z[2]), mf_swap_add32(z[1], z[3]));
      }
      {
        if (valid) {
          const uint64_t mask = smask[b];
          if (!((mask >> i) & 1u)) {                   // not a Dirichlet row
            const int lo = lrp[(spair[pc] >> 6) & 1023];
            const uint32_t cbits = (uint32_t)(mask >> (16 * jc)) & 0xFFFFu;
            const uint32_t pw[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
            int pos[16];
#pragma unroll
            for (int jj = 0; jj < 16; ++jj) pos[jj] = lo + (int)((pw[jj >> 1] >> (16 * (jj & 1))) & 0xFFFFu);
#pragma unroll
            for (int jj = 0; jj < 16; ++jj)
              if (!((cbits >> jj) & 1u)) atomicAdd(&acc[pos[jj]], cacc[jj]);
          }
        }
      }
#else
      // column factors of this lane: j = 16 * tile + (lane % 16), tile = jc
      const int ja = (lane & 15) % K1, jb = (lane & 15) / K1;
      typedef float acc4 __attribute__((ext_vector_type(4)));
      acc4 C[4];
      for (int jt = 0; jt < 4; ++jt) C[jt] = (acc4){0, 0, 0, 0};
#if MF_HX_PREC == 16
      // K slot block of 16 = 4 quadrature points; lane holds points q0 + slot, b = 0..3
      for (int qb = 0; qb < NQ; qb += 4) {
        const int q = qb + slot;
        const int q1 = q % M1, q2 = (q / M1) % M1, q3 = q / (M1 * M1);
        const real* D = &Db[q * DS];
        const double Lx = sTL[(q1) * K1 + (ia)], Ly = sTL[(q2) * K1 + (ib2)], Lz = sTL[(q3) * K1 + (ic)];
        const double Gx = sTD[(q1) * K1 + (ia)], Gy = sTD[(q2) * K1 + (ib2)], Gz = sTD[(q3) * K1 + (ic)];
        const double B0 = Lx * Ly * Lz, Bx = Gx * Ly * Lz, By = Lx * Gy * Lz, Bz = Lx * Ly * Gz;
        float f[4];
        f[0] = (float)(Bx * D[0] + By * D[1] + Bz * D[2]);
        f[1] = (float)(Bx * D[1] + By * D[3] + Bz * D[4]);
        f[2] = (float)(Bx * D[2] + By * D[4] + Bz * D[5]);
        f[3] = (float)(B0 * D[6]);
        mf_bf4 av;
        for (int h = 0; h < 4; ++h) av[h] = valid ? mf_to_bf16(f[h]) : (short)0;
        const double cLx = sTL[(q1) * K1 + (ja)], cLy = sTL[(q2) * K1 + (jb)];
        const double cGx = sTD[(q1) * K1 + (ja)], cGy = sTD[(q2) * K1 + (jb)];
        for (int jt = 0; jt < 4; ++jt) {
          const double cLz = sTL[(q3) * K1 + (jt)], cGz = sTD[(q3) * K1 + (jt)];
          mf_bf4 bv;
          bv[0] = mf_to_bf16((float)(cGx * cLy * cLz));
          bv[1] = mf_to_bf16((float)(cLx * cGy * cLz));
          bv[2] = mf_to_bf16((float)(cLx * cLy * cGz));
          bv[3] = mf_to_bf16((float)(cLx * cLy * cLz));
          C[jt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, bv, C[jt], 0, 0, 0);
        }
      }
#else
      // FP32: operands built in FP32.  Column factors of this lane (column
      // ja + 4 jb + 16 jt, component `slot`) are lane constants; row factors
      // of the tile row are loaded once per tile.
      float cx[4], cy[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        cx[m] = slot == 0 ? sTD[(m) * K1 + (ja)] : sTL[(m) * K1 + (ja)];
        cy[m] = slot == 1 ? sTD[(m) * K1 + (jb)] : sTL[(m) * K1 + (jb)];
      }
      // which D entries combine into this lane's K slot (slot 3: the mass entry)
      const int c0 = slot == 0 ? 0 : (slot == 1 ? 1 : (slot == 2 ? 2 : 6));
      const int c1 = slot == 0 ? 1 : (slot == 1 ? 3 : 4);
      const int c2 = slot == 0 ? 2 : (slot == 1 ? 4 : 5);
      // one branch-free formula for every slot:
      //   fa = P(q1) LyLz D[c0] + Q(q1) (GyLz D[c1] + LyGz D[c2])
      // slots 0-2: P = Gx, Q = Lx (the gradient row); slot 3: P = Lx, Q = 0
      // (the mass entry b0 D[6]); invalid rows are zeroed through P and Q
      const float vmask = valid ? 1.0f : 0.0f;
      float P[4], Q[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const float Lx = sTL[m * K1 + ia], Gx = sTD[m * K1 + ia];
        P[m] = (slot == 3 ? Lx : Gx) * vmask;
        Q[m] = (slot == 3 ? 0.0f : Lx) * vmask;
      }
#pragma unroll 1
      for (int q3 = 0; q3 < M1; ++q3) {
        const float Lz = sTL[(q3) * K1 + (ic)], Gz = sTD[(q3) * K1 + (ic)];
        float cz[4];
#pragma unroll
        for (int jt = 0; jt < 4; ++jt)
          cz[jt] = slot == 2 ? sTD[(q3) * K1 + (jt)] : sTL[(q3) * K1 + (jt)];
#pragma unroll
        for (int q2 = 0; q2 < 4; ++q2) {
          const float Ly = sTL[(q2) * K1 + (ib2)], Gy = sTD[(q2) * K1 + (ib2)];
          const float LyLz = Ly * Lz, GyLz = Gy * Lz, LyGz = Ly * Gz;
          const float* Dq = &Db[(4 * (q2 + 4 * q3)) * DS];
          float d0[4], d1[4], d2[4];
#pragma unroll
          for (int q1 = 0; q1 < 4; ++q1) {
            d0[q1] = Dq[q1 * DS + c0];
            d1[q1] = Dq[q1 * DS + c1];
            d2[q1] = Dq[q1 * DS + c2];
          }
#pragma unroll
          for (int q1 = 0; q1 < 4; ++q1) {
            const float fa = P[q1] * LyLz * d0[q1] + Q[q1] * (GyLz * d1[q1] + LyGz * d2[q1]);
            const float cxy = cx[q1] * cy[q2];
#pragma unroll
            for (int jt = 0; jt < 4; ++jt)
              C[jt] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa, cxy * cz[jt], C[jt], 0, 0, 0);
          }
        }
      }
#endif
      // scatter the 16 x 64 tile into the LDS segment: all 16 positions of
      // the lane first (independent searches), then the adds
      {
        int pos[4][4];
        bool ok[4][4];
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
          const int prr = t * 16 + slot * 4 + rr;
          const bool rv = prr < np;
          const int pcc = pb + (rv ? prr : 0);
          const int iq = spair[pcc] & 63;
          const uint64_t mask = smask[(spair[pcc] >> 16) - (ib - i0)];
          const bool rowok = rv && !((mask >> iq) & 1u);                  // Dirichlet row
          const int lo = lrp[(spair[pcc] >> 6) & 1023];
          const uint16_t* pp = pair_pos + ((int64_t)p0 + pcc) * ND;   // precomputed positions
#pragma unroll
          for (int jt = 0; jt < 4; ++jt) {
            const int j = jt * 16 + (lane & 15);
            ok[rr][jt] = rowok && !((mask >> j) & 1u);                    // Dirichlet column
            pos[rr][jt] = lo + (int)pp[j];
          }
        }
#pragma unroll
        for (int rr = 0; rr < 4; ++rr)
#pragma unroll
          for (int jt = 0; jt < 4; ++jt)
            if (ok[rr][jt]) atomicAdd(&acc[pos[rr][jt]], (double)C[jt][rr]);
      }
#endif
    }
    pb = pe;
    if (last) break;
  }
  __syncthreads();                                     // all contributions in acc
  __builtin_amdgcn_s_setprio(2);
  // write the segment and clear what was read
  double* out = values + (int64_t)(uint32_t)base;
  if (flags & 1) {
    const int h = min(base & 1, seglen);               // peel to a 16-byte boundary
    if (h && tid == 0) {
      __builtin_nontemporal_store(acc[0], &out[0]);
      acc[0] = 0.0;
    }
    mf_d2* o2 = reinterpret_cast<mf_d2*>(out + h);
    for (int p = tid; p < (seglen - h) >> 1; p += nt) {
      const mf_d2 v = {acc[h + 2 * p], acc[h + 2 * p + 1]};
      __builtin_nontemporal_store(v, &o2[p]);
      acc[h + 2 * p] = 0.0;
      acc[h + 2 * p + 1] = 0.0;
    }
    if (((seglen - h) & 1) && tid == 0) {
      __builtin_nontemporal_store(acc[seglen - 1], &out[seglen - 1]);
      acc[seglen - 1] = 0.0;
    }
  } else {
    for (int p = tid; p < seglen; p += nt) {
      out[p] += acc[p];
      acc[p] = 0.0;
    }
  }
  if (!more) break;
  if ((flags & 2) && nb0) __syncthreads();             // cleared before a diagonal goes in
  store_cells(min(NB, n0.w - n0.z));
  store_rows(n0, n2);
  m0 = n0; m1 = n1; m2 = n2;
  k = kn;
  }
}
#undef MF_DOFF
)";

}  // namespace mf
