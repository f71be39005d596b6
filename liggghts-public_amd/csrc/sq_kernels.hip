// Superquadric contact points on the GPU: the FP64 Newton solve for many
// independent pose pairs (eight lanes each), and the contact-point network
// that warm-starts it -- an 18 -> 64 -> 64 -> 3 tanh MLP whose forward and
// backward passes run on BF16 matrix cores (v_mfma_f32_16x16x16_bf16) with
// FP32 accumulation, trained here with Adam on FP32 master weights.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>

#include "sq_device.h"
#include "sq_group.h"
#include "sq_kernels.h"

namespace sqk {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kBlk = 256;

// ---------------------------------------------------------------------------
// contact-point solve
// ---------------------------------------------------------------------------

// mode 0: fresh contacts (homotopy from spheres); mode 1: one solve from
// init[k], and the homotopy when that one fails or stops without meeting the
// merit tolerance (the plain start then judges and replaces it).
struct SolveSource {
  const SolveArgs &a;
  int64_t k;
  __device__ bool next(sqd::QTask &t) {
    k = sqd::q_take(a.queue, a.n);
    if (k < 0) return false;
    t.start = a.mode == 0 ? sqd::kStartFresh : sqd::kStartGiven;
    for (int c = 0; c < 3; c++) {
      t.est[c] = a.mode == 0 ? 0.0 : a.init[3 * k + c];
      t.cp[c] = 0.0;
    }
    return true;
  }
  __device__ void pose(double *p) const {
    const double *src = ((threadIdx.x & 8) ? a.pose_b : a.pose_a) + 12 * k;
    for (int c = 0; c < 12; c++) p[c] = src[c];
  }
  __device__ void put(const sqd::QResult &r, const double *cp) const {
    if (!sqd::q_leader()) return;
    for (int c = 0; c < 3; c++) a.point[3 * k + c] = cp[c];
    a.fi[k] = r.fi;
    a.fj[k] = r.fj;
    a.iters[k] = r.iters;
    a.fail[k] = r.fail | (r.fallback << 1);
  }
};

__global__ __launch_bounds__(sqd::kGroupBlock, 2) void k_sq_solve(SolveArgs a) {
  __shared__ sqd::GroupLds lds;
  SolveSource src{a, 0};
  sqd::q_solve_all(src, a.max_iter, lds);
}

__global__ void k_zero_queue(unsigned *queue) { *queue = 0u; }

// the optional refinement of a finished solve, one thread per pair
__global__ __launch_bounds__(kBlk) void k_sq_polish(SolveArgs a) {
  const int64_t k = (int64_t)blockIdx.x * kBlk + threadIdx.x;
  if (k >= a.n || (a.fail[k] & 1)) return;
  sqd::Sq A, B;
  sqd::init(A, a.pose_a + 12 * k);
  sqd::init(B, a.pose_b + 12 * k);
  double cp[3] = {a.point[3 * k], a.point[3 * k + 1], a.point[3 * k + 2]};
  double fi = a.fi[k], fj = a.fj[k];
  a.iters[k] += sqd::polish(A, B, cp, fi, fj, a.polish);
  for (int c = 0; c < 3; c++) a.point[3 * k + c] = cp[c];
  a.fi[k] = fi;
  a.fj[k] = fj;
}

// SurfaceModel<SURFACE_SUPERQUADRIC>::checkSurfaceIntersect
// (surface_model_superquadric.h:108-205): OBB pre-check unless the pair
// intersected last step, the contact point (homotopy for a pair far apart
// last step, else from the previous point moved by the mass-weighted contact
// velocity, calc_contact_point_using_prev_step, math_extra_liggghts_superquadric.cpp:
// 1434-1466), and for intersecting surfaces the normal from the two gradients
// and the overlap along it (extended_overlap_algorithm, :1489-1504). With
// init, a pair far apart last step starts from the network's point instead of
// the homotopy, which remains the fallback. Three launches: the pre-check and
// the start point (one thread per pair), the solves (eight lanes per pair),
// the overlap (one thread per pair). Between them a pair's start kind waits in
// flags (kNoSolve: boxes apart), its start point in en, the gradients at the
// contact point in cp_i and cp_j.
constexpr int kNoSolve = 8;

__global__ __launch_bounds__(kBlk) void k_sq_check_start(CheckArgs a) {
  const int64_t k = (int64_t)blockIdx.x * kBlk + threadIdx.x;
  if (k >= a.n) return;
  sqd::Sq A, B;
  sqd::init(A, a.pose_a + 12 * k);
  sqd::init(B, a.pose_b + 12 * k);
  double *h = a.hist + kHist * k;
  const int state = (int)(h[0] + 0.5);
  int start = (int)(h[1] + 0.5);
  const int obb = state == 2 ? 1 : sqd::obb_intersect(A, B, start);
  h[1] = (double)start;
  if (!obb) {
    a.flags[k] = kNoSolve;
    return;
  }
  const double cp[3] = {h[2], h[3], h[4]};
  double est[3] = {cp[0], cp[1], cp[2]};
  int kind = sqd::kStartOnly;
  if (state == 0) {
    kind = a.init ? sqd::kStartGiven : sqd::kStartFresh;
    if (a.init)
      for (int c = 0; c < 3; c++) est[c] = a.init[3 * k + c];
  } else if (a.vel && a.mass) {
    const double *v = a.vel + 12 * k;
    const double mi = a.mass[2 * k], mj = a.mass[2 * k + 1];
    const double xci[3] = {cp[0] - A.center[0], cp[1] - A.center[1], cp[2] - A.center[2]};
    const double xcj[3] = {cp[0] - B.center[0], cp[1] - B.center[1], cp[2] - B.center[2]};
    const double *wi = v + 6, *wj = v + 9;
    const double ri_[3] = {wi[1] * xci[2] - wi[2] * xci[1], wi[2] * xci[0] - wi[0] * xci[2],
                           wi[0] * xci[1] - wi[1] * xci[0]};
    const double rj_[3] = {wj[1] * xcj[2] - wj[2] * xcj[1], wj[2] * xcj[0] - wj[0] * xcj[2],
                           wj[0] * xcj[1] - wj[1] * xcj[0]};
    for (int c = 0; c < 3; c++) {
      const double vi = v[c] + ri_[c], vj = v[3 + c] + rj_[c];
      const double veff = (vi * mi + vj * mj) / (mi + mj);
      est[c] = cp[c] + veff * a.dt;
    }
  }
  a.flags[k] = kind;
  for (int c = 0; c < 3; c++) a.en[3 * k + c] = est[c];
}

struct CheckSource {
  const CheckArgs &a;
  int64_t k;
  __device__ bool next(sqd::QTask &t) {
    do {
      k = sqd::q_take(a.queue, a.n);
      if (k < 0) return false;
      t.start = a.flags[k];
    } while (t.start == kNoSolve);
    for (int c = 0; c < 3; c++) {
      t.est[c] = a.en[3 * k + c];
      t.cp[c] = a.hist[kHist * k + 2 + c];
    }
    return true;
  }
  __device__ void pose(double *p) const {
    const double *src = ((threadIdx.x & 8) ? a.pose_b : a.pose_a) + 12 * k;
    for (int c = 0; c < 12; c++) p[c] = src[c];
  }
  __device__ void put(const sqd::QResult &r, const double *cp) const {
    if (!sqd::q_leader()) return;
    for (int c = 0; c < 3; c++) {
      a.point[3 * k + c] = cp[c];
      a.cp_i[3 * k + c] = r.gA[c];
      a.cp_j[3 * k + c] = r.gB[c];
    }
    a.fi[k] = r.fi;
    a.fj[k] = r.fj;
    a.iters[k] = r.iters;
    a.flags[k] = r.fail | (r.fallback << 1);
  }
};

__global__ __launch_bounds__(sqd::kGroupBlock, 2) void k_sq_check_solve(CheckArgs a) {
  __shared__ sqd::GroupLds lds;
  CheckSource src{a, 0};
  sqd::q_solve_all(src, a.max_iter, lds);
}

__global__ __launch_bounds__(kBlk) void k_sq_check_finish(CheckArgs a) {
  const int64_t k = (int64_t)blockIdx.x * kBlk + threadIdx.x;
  if (k >= a.n) return;
  double *h = a.hist + kHist * k;
  double en[3] = {0.0, 0.0, 0.0}, dn = 0.0, cpa[3] = {0.0, 0.0, 0.0}, cpb[3] = {0.0, 0.0, 0.0};
  int contact = 0;
  if (a.flags[k] == kNoSolve) {
    for (int c = 0; c < 3; c++) a.point[3 * k + c] = h[2 + c];
    a.fi[k] = a.fj[k] = 0.0;
    a.iters[k] = 0;
    a.flags[k] = 1 << 2;
    h[0] = 0.0;
  } else {
    const double cp[3] = {a.point[3 * k], a.point[3 * k + 1], a.point[3 * k + 2]};
    const double fi = a.fi[k], fj = a.fj[k];
    contact = (fi > fj ? fi : fj) < 0.0;
    if (contact) {
      sqd::Sq A, B;
      sqd::init(A, a.pose_a + 12 * k);
      sqd::init(B, a.pose_b + 12 * k);
      sqd::overlap_along_normal(A, B, cp, a.cp_i + 3 * k, a.cp_j + 3 * k, en, h[5], h[6], cpa, cpb);
      dn = fabs(h[5]) + fabs(h[6]);
    }
    h[0] = contact ? 2.0 : 1.0;
    for (int c = 0; c < 3; c++) h[2 + c] = cp[c];
  }
  a.contact[k] = contact;
  for (int c = 0; c < 3; c++) {
    a.en[3 * k + c] = en[c];
    a.cp_i[3 * k + c] = cpa[c];
    a.cp_j[3 * k + c] = cpb[c];
  }
  a.deltan[k] = dn;
}

// ---------------------------------------------------------------------------
// network inputs and outputs (the encoding of superquadrics.py)
// ---------------------------------------------------------------------------
__device__ __forceinline__ void rot_of(const double *q, double *R) {
  const double w = q[0], i = q[1], j = q[2], kk = q[3];
  R[0] = w * w + i * i - j * j - kk * kk;
  R[1] = 2 * i * j - 2 * kk * w;
  R[2] = 2 * j * w + 2 * i * kk;
  R[3] = 2 * i * j + 2 * kk * w;
  R[4] = w * w - i * i + j * j - kk * kk;
  R[5] = 2 * j * kk - 2 * i * w;
  R[6] = 2 * i * kk - 2 * j * w;
  R[7] = 2 * j * kk + 2 * i * w;
  R[8] = w * w - i * i - j * j + kk * kk;
}

__global__ __launch_bounds__(kBlk) void k_sq_features(const double *pa, const double *pb, int64_t n,
                                                       float *X) {
  const int64_t k = (int64_t)blockIdx.x * kBlk + threadIdx.x;
  if (k >= n) return;
  const double *A = pa + 12 * k, *B = pb + 12 * k;
  const double rA = cbrt(A[7] * A[8] * A[9]), rB = cbrt(B[7] * B[8] * B[9]);
  const double L = rA + rB;
  double R[9];
  rot_of(A + 3, R);
  const double d[3] = {B[0] - A[0], B[1] - A[1], B[2] - A[2]};
  float *x = X + 18 * k;
  for (int c = 0; c < 3; c++) x[c] = (float)((R[c] * d[0] + R[3 + c] * d[1] + R[6 + c] * d[2]) / L);
  // conj(qA) * qB
  const double w1 = A[3], x1 = -A[4], y1 = -A[5], z1 = -A[6];
  const double w2 = B[3], x2 = B[4], y2 = B[5], z2 = B[6];
  double qr[4] = {w1 * w2 - x1 * x2 - y1 * y2 - z1 * z2, w1 * x2 + x1 * w2 + y1 * z2 - z1 * y2,
                  w1 * y2 - x1 * z2 + y1 * w2 + z1 * x2, w1 * z2 + x1 * y2 - y1 * x2 + z1 * w2};
  const double sg = qr[0] < 0.0 ? -1.0 : 1.0;
  for (int c = 0; c < 4; c++) x[3 + c] = (float)(qr[c] * sg);
  for (int c = 0; c < 3; c++) x[7 + c] = (float)(A[7 + c] / rA);
  x[10] = (float)(A[10] / 8.0);
  x[11] = (float)(A[11] / 8.0);
  for (int c = 0; c < 3; c++) x[12 + c] = (float)(B[7 + c] / rB);
  x[15] = (float)(B[10] / 8.0);
  x[16] = (float)(B[11] / 8.0);
  x[17] = (float)(rA / (rA + rB));
}

// global contact points from outputs (to_point), or targets from points (from_point)
__global__ __launch_bounds__(kBlk) void k_sq_frame(const double *pa, const double *pb, int64_t n,
                                                    const float *Y, double *P, const double *Pin,
                                                    float *T) {
  const int64_t k = (int64_t)blockIdx.x * kBlk + threadIdx.x;
  if (k >= n) return;
  const double *A = pa + 12 * k, *B = pb + 12 * k;
  const double L = cbrt(A[7] * A[8] * A[9]) + cbrt(B[7] * B[8] * B[9]);
  double R[9];
  rot_of(A + 3, R);
  if (Y) {
    const double y[3] = {(double)Y[3 * k] * L, (double)Y[3 * k + 1] * L, (double)Y[3 * k + 2] * L};
    for (int c = 0; c < 3; c++) P[3 * k + c] = A[c] + (R[3 * c] * y[0] + R[3 * c + 1] * y[1] + R[3 * c + 2] * y[2]);
  } else {
    const double d[3] = {Pin[3 * k] - A[0], Pin[3 * k + 1] - A[1], Pin[3 * k + 2] - A[2]};
    for (int c = 0; c < 3; c++) T[3 * k + c] = (float)((R[c] * d[0] + R[3 + c] * d[1] + R[6 + c] * d[2]) / L);
  }
}

// ---------------------------------------------------------------------------
// the network on matrix cores
//
// v_mfma_f32_16x16x16_bf16 lane layout (64 lanes, l = lane, r = l % 16,
// q = l / 16): A (16 x 16, M x K) element A[r][4q + j] in slot j of the lane's
// bf16x4; B (K x N) element B[4q + j][r]; the FP32 result D[4q + j][r] in
// slot j. One wavefront owns a tile of 16 samples and computes every layer
// transposed, H^T = W^T X^T: a layer's result (feature 4q + j of sample r) is
// then the next layer's B operand as it stands, so activations and deltas pass
// from product to product in registers, and the weights are A operands read
// from the L2 as the lane's own 8 bytes. Only the weight gradients, whose
// products run over the samples, take their operands through LDS.
// ---------------------------------------------------------------------------
__device__ __forceinline__ unsigned short to_bf16(float f) { return pack_bf16(f); }

__device__ __forceinline__ floatx4 mfma(bf16x4 a, bf16x4 b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ bf16x4 pack4(const floatx4 &v) {
  bf16x4 o;
  for (int j = 0; j < 4; j++) o[j] = (short)to_bf16(v[j]);
  return o;
}

// A operand: tile t of a packed weight array
__device__ __forceinline__ bf16x4 ld_w(const unsigned short *w, int t) {
  return *(const bf16x4 *)(w + ((size_t)t * 64 + (threadIdx.x & 63)) * 4);
}

constexpr int kTilesHid = kHid / 16, kTilesIn = kInPad / 16;

// activations of a tile: FP32 and the BF16 operands the products read
struct Hidden {
  bf16x4 x[kTilesIn], b1[kTilesHid], b2[kTilesHid];
  floatx4 h1[kTilesHid], h2[kTilesHid];
};

// forward pass of one 16-sample tile; row: this lane's sample (r), valid or a
// zero input. Returns output 4q + j of sample r.
__device__ __forceinline__ floatx4 forward_tile(const NetDev &net, const float *X, int64_t row, bool valid,
                                                Hidden &hid) {
  const int q = (threadIdx.x & 63) >> 4;
  for (int ks = 0; ks < kTilesIn; ks++) {
    floatx4 v = {0.f, 0.f, 0.f, 0.f};
    for (int j = 0; j < 4; j++) {
      const int k = 16 * ks + 4 * q + j;
      if (valid && k < kIn) v[j] = X[row * kIn + k];
    }
    hid.x[ks] = pack4(v);
  }
#pragma unroll
  for (int nt = 0; nt < kTilesHid; nt++) {
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int ks = 0; ks < kTilesIn; ks++) acc = mfma(ld_w(net.w1f, nt * kTilesIn + ks), hid.x[ks], acc);
    const float *b = net.b1 + 16 * nt + 4 * q;
    for (int j = 0; j < 4; j++) hid.h1[nt][j] = tanhf(acc[j] + b[j]);
    hid.b1[nt] = pack4(hid.h1[nt]);
  }
#pragma unroll
  for (int nt = 0; nt < kTilesHid; nt++) {
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int ks = 0; ks < kTilesHid; ks++) acc = mfma(ld_w(net.w2f, nt * kTilesHid + ks), hid.b1[ks], acc);
    const float *b = net.b2 + 16 * nt + 4 * q;
    for (int j = 0; j < 4; j++) hid.h2[nt][j] = tanhf(acc[j] + b[j]);
    hid.b2[nt] = pack4(hid.h2[nt]);
  }
  floatx4 y = {0.f, 0.f, 0.f, 0.f};
  for (int ks = 0; ks < kTilesHid; ks++) y = mfma(ld_w(net.w3f, ks), hid.b2[ks], y);
  for (int j = 0; j < 4; j++) y[j] += net.b3[4 * q + j];
  return y;
}

__global__ __launch_bounds__(kBlk) void k_mlp_forward(NetDev net, const float *X, int64_t n, float *Y) {
  const int l = threadIdx.x & 63, r = l & 15, q = l >> 4;
  const int64_t row = ((int64_t)blockIdx.x * (kBlk / 64) + (threadIdx.x >> 6)) * 16 + r;
  Hidden hid;
  const floatx4 y = forward_tile(net, X, row, row < n, hid);
  if (q == 0 && row < n)
    for (int j = 0; j < kOut; j++) Y[row * kOut + j] = y[j];
}

// sample k of a batch
__device__ __forceinline__ int64_t picked_row(const RowPick &p, int64_t k) {
  if (p.n <= 0) return k;
  uint64_t z = p.seed + 0x9e3779b97f4a7c15ull * (uint64_t)(k + 1);  // splitmix64
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  z ^= z >> 31;
  return (int64_t)(z % (uint64_t)p.n);
}

// A tile's operands of the weight-gradient products, sample by sample: rows
// padded by 8 bytes so that the 16 lanes of a write fall in different banks.
constexpr int kActStride = kHid + 4, kXStride = kInPad + 4, kYStride = kOutPad + 4;
struct WaveLds {
  unsigned short x[16 * kXStride], h1[16 * kActStride], h2[16 * kActStride], d1[16 * kActStride],
      d2[16 * kActStride], dy[16 * kYStride];
};
struct GradLds {
  WaveLds wave[kBlk / 64];
  float part[kBlk / 64][kNumParams];  // each wavefront's parameter gradients
  float loss[kBlk / 64];
};

// features 16t + 4q .. + 3 of sample r
__device__ __forceinline__ void put_act(unsigned short *m, int stride, int t, bf16x4 v) {
  const int l = threadIdx.x & 63;
  *(bf16x4 *)(m + (l & 15) * stride + 16 * t + 4 * (l >> 4)) = v;
}

// feature 16t + r of samples 4q .. + 3: the A operand (rows features) and the B
// operand (columns features) of a product over the samples
__device__ __forceinline__ bf16x4 get_act(const unsigned short *m, int stride, int t) {
  const int l = threadIdx.x & 63;
  const unsigned short *p = m + 4 * (l >> 4) * stride + 16 * t + (l & 15);
  bf16x4 v;
  for (int j = 0; j < 4; j++) v[j] = (short)p[j * stride];
  return v;
}

template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}

// Sums over the row of 16 lanes (the tile's samples), valid in its lane 0: four
// samples one after another, then the four groups in pairs. The order is part
// of the result: the parameters after some hundred Adam steps depend on the
// rounding of each sum.
constexpr int kDppShl4 = 0x104, kDppShl8 = 0x108;  // the value of lane i + 4, i + 8
__device__ __forceinline__ float quad_sum(float v) {
  return ((v + dpp<0x55>(v)) + dpp<0xaa>(v)) + dpp<0xff>(v);  // quad_perm: the quad's lanes 1, 2, 3
}
// (group 0 + group 1) + (group 2 + group 3)
__device__ __forceinline__ float row_sum(float v) {
  v = quad_sum(v);
  v += dpp<kDppShl4>(v);
  return v + dpp<kDppShl8>(v);
}
// (group 0 + group 2) + (group 1 + group 3)
__device__ __forceinline__ float row_sum_across(float v) {
  v = quad_sum(v);
  v += dpp<kDppShl8>(v);
  return v + dpp<kDppShl4>(v);
}

// one gradient pass: every wavefront takes one 16-sample tile of the batch,
// runs forward and backward with the products on matrix cores, and the block
// writes the sum of its four tiles' parameter gradients to part[block][] (in a
// fixed order, so the result does not depend on timing). Loss = mean over the
// batch of |y - t|^2; BF16 copies feed every product: inputs, weights, hidden
// activations, and the output and hidden-layer deltas. Bound by the latency of
// one tile's chain (32 tanh a lane, 80 products): 8,192 samples in 21 us on
// half the chip's CUs; with the weights staged in LDS two bytes at a time and
// the activations passed through it 30 us.
__global__ __launch_bounds__(kBlk) void k_mlp_grad(NetDev net, const float *X, const float *T, RowPick pick,
                                                    int64_t batch, float *part, float *loss_part) {
  __shared__ GradLds s;
  const int wv = threadIdx.x >> 6, l = threadIdx.x & 63, r = l & 15, q = l >> 4;
  WaveLds &w = s.wave[wv];
  float *out = s.part[wv];
  const int64_t k = ((int64_t)blockIdx.x * (kBlk / 64) + wv) * 16 + r;
  const bool valid = k < batch;
  const int64_t row = valid ? picked_row(pick, k) : 0;
  Hidden hid;
  const floatx4 y = forward_tile(net, X, row, valid, hid);
  const float scale = 2.0f / (float)batch;
  floatx4 d = {0.f, 0.f, 0.f, 0.f}, sq = d;
  if (valid && q == 0)
    for (int j = 0; j < kOut; j++) {
      const float e = y[j] - T[row * kOut + j];
      sq[j] = e * e;
      d[j] = scale * e;
    }
  const bf16x4 dyb = pack4(d);
  for (int t = 0; t < kTilesIn; t++) put_act(w.x, kXStride, t, hid.x[t]);
  for (int t = 0; t < kTilesHid; t++) {
    put_act(w.h1, kActStride, t, hid.b1[t]);
    put_act(w.h2, kActStride, t, hid.b2[t]);
  }
  put_act(w.dy, kYStride, 0, dyb);
  const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
  // dZ2 = (dY W3^T) * (1 - h2^2), dZ1 = (dZ2 W2^T) * (1 - h1^2), transposed
  bf16x4 d2b[kTilesHid];
#pragma unroll
  for (int t = 0; t < kTilesHid; t++) {
    floatx4 v = mfma(ld_w(net.w3t, t), dyb, zero);
    for (int j = 0; j < 4; j++) v[j] *= 1.0f - hid.h2[t][j] * hid.h2[t][j];
    d2b[t] = pack4(v);
    put_act(w.d2, kActStride, t, d2b[t]);
    for (int j = 0; j < 4; j++) {
      const float b = row_sum(v[j]);
      if (r == 0) out[kOffB2 + 16 * t + 4 * q + j] = b;
    }
  }
#pragma unroll
  for (int t = 0; t < kTilesHid; t++) {
    floatx4 v = zero;
    for (int ks = 0; ks < kTilesHid; ks++) v = mfma(ld_w(net.w2t, t * kTilesHid + ks), d2b[ks], v);
    for (int j = 0; j < 4; j++) v[j] *= 1.0f - hid.h1[t][j] * hid.h1[t][j];
    put_act(w.d1, kActStride, t, pack4(v));
    for (int j = 0; j < 4; j++) {
      const float b = row_sum(v[j]);
      if (r == 0) out[kOffB1 + 16 * t + 4 * q + j] = b;
    }
  }
  for (int j = 0; j < 4; j++) {
    const float b = row_sum(d[j]);
    if (l == 0 && j < kOut) out[kOffB3 + j] = b;
  }
  static_assert(kOut == 3, "the loss adds the outputs 0 and 2 first");
  const float lsum = (row_sum_across(sq[0]) + row_sum_across(sq[2])) + row_sum_across(sq[1]);
  if (l == 0) s.loss[wv] = lsum;
  __syncthreads();  // the tile's operands are in LDS
  // dW3 = H2^T dY, dW2 = H1^T dZ2, dW1 = X^T dZ1 (rows >= kIn are padding)
  {
    const bf16x4 b = get_act(w.dy, kYStride, 0);
    for (int mt = 0; mt < kTilesHid; mt++) {
      const floatx4 g = mfma(get_act(w.h2, kActStride, mt), b, zero);
      if (r < kOut)
        for (int j = 0; j < 4; j++) out[kOffW3 + (mt * 16 + 4 * q + j) * kOut + r] = g[j];
    }
  }
  bf16x4 ah[kTilesHid], ax[kTilesIn];
  for (int mt = 0; mt < kTilesHid; mt++) ah[mt] = get_act(w.h1, kActStride, mt);
  for (int mt = 0; mt < kTilesIn; mt++) ax[mt] = get_act(w.x, kXStride, mt);
#pragma unroll
  for (int nt = 0; nt < kTilesHid; nt++) {
    const bf16x4 b2 = get_act(w.d2, kActStride, nt), b1 = get_act(w.d1, kActStride, nt);
    for (int mt = 0; mt < kTilesHid; mt++) {
      const floatx4 g = mfma(ah[mt], b2, zero);
      for (int j = 0; j < 4; j++) out[kOffW2 + (mt * 16 + 4 * q + j) * kHid + nt * 16 + r] = g[j];
    }
    for (int mt = 0; mt < kTilesIn; mt++) {
      const floatx4 g = mfma(ax[mt], b1, zero);
      for (int j = 0; j < 4; j++) {
        const int m = mt * 16 + 4 * q + j;
        if (m < kIn) out[kOffW1 + m * kHid + nt * 16 + r] = g[j];
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kNumParams; i += kBlk) {
    float v = 0.f;
    for (int p = 0; p < kBlk / 64; p++) v += s.part[p][i];
    part[(int64_t)blockIdx.x * kNumParams + i] = v;
  }
  if (threadIdx.x == 0) {
    float v = 0.f;
    for (int p = 0; p < kBlk / 64; p++) v += s.loss[p];
    loss_part[blockIdx.x] = v;
  }
}

// sums the blocks' gradient partials one after another, then one Adam step on
// the FP32 master parameters and a refresh of the copies the matrix cores read.
// ad.apply = 0: only the summed gradient is written. 64 parameters a block: its
// 1,024 threads load 256 partials of each together, one wavefront adds them in
// order out of LDS. The last block sums the batch loss. Bound by that chain of
// additions, about 1 us for the 128 partials of 8,192 samples: a training step
// takes 24.7 us (16,384 samples: 27.2); with the partials added in 16 slices,
// another order, 24.1 (25.9), with one thread a parameter loading them in a
// row 67 (103).
constexpr int kAdamParams = 64, kAdamSlices = 16, kAdamRows = 256, kAdamBatch = 32;
__global__ __launch_bounds__(kAdamParams * kAdamSlices)
    __attribute__((amdgpu_waves_per_eu(4, 4))) void k_mlp_adam(NetDev net, const float *part, int nparts, float *grad,
                                                               AdamArgs ad) {
  __shared__ float stage[kAdamRows][kAdamParams];
  const int c = threadIdx.x % kAdamParams, sl = threadIdx.x / kAdamParams;
  const bool loss = blockIdx.x == gridDim.x - 1;
  const int i = blockIdx.x * kAdamParams + c;
  const int at = i < kNumParams ? i : kNumParams - 1;
  // what the update needs is under way while the partials are summed
  float m0 = 0.f, v0 = 0.f, p0 = 0.f;
  if (sl == 0 && ad.apply) {
    m0 = net.m[at];
    v0 = net.v[at];
    p0 = net.params[at];
  }
  float gsum = 0.f;
  for (int b0 = 0; b0 < nparts; b0 += kAdamRows) {
    const int rows = nparts - b0 < kAdamRows ? nparts - b0 : kAdamRows;
    const int padded = (rows + kAdamBatch - 1) / kAdamBatch * kAdamBatch;
    if (b0 > 0) __syncthreads();
    if (loss) {
      if ((int)threadIdx.x < padded) stage[threadIdx.x][0] = (int)threadIdx.x < rows ? ad.loss_part[b0 + threadIdx.x] : 0.f;
    } else {
      // independent loads, the last row again past it
      float v[kAdamRows / kAdamSlices];
#pragma unroll
      for (int u = 0; u < kAdamRows / kAdamSlices; u++) {
        const int r = u * kAdamSlices + sl;
        if (u * kAdamSlices < rows) v[u] = part[(int64_t)(b0 + (r < rows ? r : rows - 1)) * kNumParams + at];
      }
#pragma unroll
      for (int u = 0; u < kAdamRows / kAdamSlices; u++) {
        const int r = u * kAdamSlices + sl;
        if (u * kAdamSlices < padded) stage[r][c] = r < rows ? v[u] : 0.f;
      }
    }
    __syncthreads();
    if (sl == 0) {
      // the zeros behind the last row change no sum; the next rows are read
      // while these are added
      float v[kAdamBatch], w[kAdamBatch];
      const auto read = [&](float(&q)[kAdamBatch], int r) {
#pragma unroll
        for (int u = 0; u < kAdamBatch; u++) q[u] = stage[r + u][c];
        __builtin_amdgcn_sched_barrier(0);
      };
      const auto add = [&](const float(&q)[kAdamBatch]) {
#pragma unroll
        for (int u = 0; u < kAdamBatch; u++) gsum += q[u];
      };
      read(v, 0);
      for (int r = 0; r < rows; r += 2 * kAdamBatch) {
        read(w, r + kAdamBatch < padded ? r + kAdamBatch : 0);
        add(v);
        if (r + kAdamBatch >= rows) break;
        read(v, r + 2 * kAdamBatch < padded ? r + 2 * kAdamBatch : 0);
        add(w);
      }
    }
  }
  if (sl != 0) return;
  if (loss) {
    if (c == 0 && ad.loss_out) *ad.loss_out = gsum / (float)ad.batch;
    return;
  }
  if (i >= kNumParams) return;
  grad[i] = gsum;
  if (!ad.apply) return;
  const float m = ad.beta1 * m0 + (1.0f - ad.beta1) * gsum;
  const float v2 = ad.beta2 * v0 + (1.0f - ad.beta2) * gsum * gsum;
  net.m[i] = m;
  net.v[i] = v2;
  const float mh = m / ad.bc1, vh = v2 / ad.bc2;
  const float p = p0 - ad.lr * mh / (sqrtf(vh) + ad.eps);
  net.params[i] = p;
  write_packed(net, i, p);
}

__global__ __launch_bounds__(kBlk) void k_mlp_pack(NetDev net) {
  const int i = blockIdx.x * kBlk + threadIdx.x;
  if (i < kNumParams) write_packed(net, i, net.params[i]);
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static inline unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

// wavefronts of a solve: the pairs spread eight to a wavefront, as far as the
// chip holds them at once (1,024 SIMDs, two wavefronts each by registers)
static inline unsigned solve_blocks(int64_t n) {
  const int64_t b = (n + sqd::kGroupsPerBlock - 1) / sqd::kGroupsPerBlock;
  return (unsigned)(b < 2048 ? b : 2048);
}

hipError_t launch_solve(const SolveArgs &a, hipStream_t s) {
  if (a.n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_zero_queue, dim3(1), dim3(1), 0, s, a.queue);
  hipLaunchKernelGGL(k_sq_solve, dim3(solve_blocks(a.n)), dim3(sqd::kGroupBlock), 0, s, a);
  if (a.polish > 0) hipLaunchKernelGGL(k_sq_polish, dim3(nblk(a.n, kBlk)), dim3(kBlk), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_check(const CheckArgs &a, hipStream_t s) {
  if (a.n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_sq_check_start, dim3(nblk(a.n, kBlk)), dim3(kBlk), 0, s, a);
  hipLaunchKernelGGL(k_zero_queue, dim3(1), dim3(1), 0, s, a.queue);
  hipLaunchKernelGGL(k_sq_check_solve, dim3(solve_blocks(a.n)), dim3(sqd::kGroupBlock), 0, s, a);
  hipLaunchKernelGGL(k_sq_check_finish, dim3(nblk(a.n, kBlk)), dim3(kBlk), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_features(const double *pa, const double *pb, int64_t n, float *X, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_sq_features, dim3(nblk(n, kBlk)), dim3(kBlk), 0, s, pa, pb, n, X);
  return hipGetLastError();
}

hipError_t launch_to_point(const double *pa, const double *pb, int64_t n, const float *Y, double *P,
                           hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_sq_frame, dim3(nblk(n, kBlk)), dim3(kBlk), 0, s, pa, pb, n, Y, P,
                     (const double *)nullptr, (float *)nullptr);
  return hipGetLastError();
}

hipError_t launch_to_target(const double *pa, const double *pb, int64_t n, const double *P, float *T,
                            hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_sq_frame, dim3(nblk(n, kBlk)), dim3(kBlk), 0, s, pa, pb, n,
                     (const float *)nullptr, (double *)nullptr, P, T);
  return hipGetLastError();
}

hipError_t launch_mlp_forward(const NetDev &net, const float *X, int64_t n, float *Y, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_mlp_forward, dim3(nblk(n, kBlk / 4)), dim3(kBlk), 0, s, net, X, n, Y);
  return hipGetLastError();
}

int grad_blocks(int64_t batch) { return (int)nblk(batch, kBlk / 4); }

// Workspace of the allocation-free gradient entry point: k_mlp_grad's
// per-block gradient partials ([blocks][kNumParams]) followed by its per-block
// loss partials, for batches of up to kGradScratchMaxBatch samples. Every
// block writes its whole partial, so nothing needs clearing between calls.
// Each device holds its own copy until the process ends.
constexpr int kGradScratchBlocks = (int)((kGradScratchMaxBatch + kBlk / 4 - 1) / (kBlk / 4));
static __device__ __align__(256) float scratch[(size_t)kGradScratchBlocks * (kNumParams + 1)];

// Device address of this device's scratch copy (the array's name is only a
// host-side stand-in). Resolved once per device with that device current.
hipError_t grad_scratch(int device, float **part, float **loss_part) {
  static std::mutex mu;
  static float *addr[kMaxScratchDevices] = {};
  if (device < 0 || device >= kMaxScratchDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(mu);
  if (!addr[device]) {
    float *p = nullptr;
    const hipError_t e = hipGetSymbolAddress((void **)&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    addr[device] = p;
  }
  *part = addr[device];
  *loss_part = addr[device] + (size_t)kGradScratchBlocks * kNumParams;
  return hipSuccess;
}

hipError_t launch_mlp_grad(const NetDev &net, const float *X, const float *T, const RowPick &pick,
                           int64_t batch, float *part, float *loss_part, hipStream_t s) {
  if (batch <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_mlp_grad, dim3(grad_blocks(batch)), dim3(kBlk), 0, s, net, X, T, pick, batch, part,
                     loss_part);
  return hipGetLastError();
}

hipError_t launch_mlp_adam(const NetDev &net, const float *part, int nparts, float *grad, const AdamArgs &ad,
                           hipStream_t s) {
  hipLaunchKernelGGL(k_mlp_adam, dim3(nblk(kNumParams, kAdamParams) + 1), dim3(kAdamParams * kAdamSlices), 0, s, net,
                     part, nparts, grad, ad);
  return hipGetLastError();
}

hipError_t launch_mlp_pack(const NetDev &net, hipStream_t s) {
  hipLaunchKernelGGL(k_mlp_pack, dim3(nblk(kNumParams, kBlk)), dim3(kBlk), 0, s, net);
  return hipGetLastError();
}

}  // namespace sqk
