// Coordinate MLP of the learned warm start (include/usg_mlp.h) on gfx950:
// every product is v_mfma_f32_16x16x32_bf16 (BF16 operands, FP32
// accumulation).
//
// Operand layout of one 16x16x32 MFMA in a 64-lane wave (lane l):
//   A (16 x 32): row l % 16, k = 8 * (l / 16) .. +7      (8 bf16 in a lane)
//   B (32 x 16): column l % 16, k = 8 * (l / 16) .. +7
//   C (16 x 16): column l % 16, rows 4 * (l / 16) .. +3  (4 floats)
// (checked against the CPU by usg_mlp_mfma_check).  Activations are kept
// twice: as rows in LDS (the A operand of the forward and data-gradient
// products, 8 consecutive k per lane) and in memory as operands of the
// weight-gradient product, which reduces over points (8 consecutive points per
// lane).  Every operand load is one 16-byte load.
//
// A training step is two launches: k_net (batch assembly, forward pass, loss,
// data gradients) and k_weights (weight and bias gradients, Adam); for a small
// network on a large batch k_apply (Adam) is a third.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/usg_mlp.h"

namespace usgmlp {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint16_t bf16;  // raw bits

constexpr int kWave = 64;
constexpr int kChunk = 256;  // points per partial sum of the weight and bias gradients

thread_local std::string g_err;
int fail(int code, const std::string &m) {
  g_err = m;
  return code;
}
#define HIPCHK(x)                                                                        \
  do {                                                                                   \
    hipError_t e_ = (x);                                                                 \
    if (e_ != hipSuccess) return fail(-3, std::string(#x) + ": " + hipGetErrorString(e_)); \
  } while (0)

// FP32 -> BF16, round to nearest even (finite inputs)
__host__ __device__ __forceinline__ bf16 to_bf16(float f) {
  uint32_t u;
  std::memcpy(&u, &f, 4);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (bf16)(u >> 16);
}
__host__ __device__ __forceinline__ float from_bf16(bf16 h) {
  uint32_t u = (uint32_t)h << 16;
  float f;
  std::memcpy(&f, &u, 4);
  return f;
}
__device__ __forceinline__ float sigmoid(float z) { return 1.0f / (1.0f + expf(-z)); }

__device__ __forceinline__ bf16x8 load8(const bf16 *p) { return *reinterpret_cast<const bf16x8 *>(p); }

// ---------------------------------------------------------------------------
// The network as the kernels see it.  Weights come as MFMA operands: `wf` the
// B fragments of the forward product (reduction over k), `wb` those of the
// data gradient (reduction over n), each fragment 64 lanes x 8 values in lane
// order, so that a wave loads one with a single contiguous kilobyte.  Layers
// follow one another in every array; where a layer begins is arithmetic on
// the shape (a table would put a dependent load before each layer).
// ---------------------------------------------------------------------------
constexpr int kOut = 32;   // padded outputs of the last layer
struct Net {
  int nl, W, K0, nin, nout;  // layers, width, padded and real inputs, outputs
  long P;                    // points (training; a multiple of 128)
  bf16 *wf, *wb;
  bf16 *in;                  // input of each layer, P x K (pt_index; training)
  bf16 *dz;                  // output gradient of each layer, P x N (pt_index; training)
  bf16 *h;                   // rows of each hidden output [P][W] that LDS cannot hold (training)
  float *w, *b;              // FP32 masters, compact
  __host__ __device__ int K(int l) const { return l == 0 ? K0 : W; }
  __host__ __device__ int N(int l) const { return l == nl - 1 ? kOut : W; }
  __host__ __device__ int k(int l) const { return l == 0 ? nin : W; }
  __host__ __device__ int n(int l) const { return l == nl - 1 ? nout : W; }
  __host__ __device__ long frag(int l) const { return l == 0 ? 0 : (long)K0 * W + (long)(l - 1) * W * W; }
  __host__ __device__ long inp(int l) const { return l == 0 ? 0 : P * K0 + (l - 1) * P * W; }
  __host__ __device__ long out(int l) const { return l * P * W; }
  __host__ __device__ long ow(int l) const { return l == 0 ? 0 : (long)nin * W + (long)(l - 1) * W * W; }
  __host__ __device__ long ob(int l) const { return (long)l * W; }
  __host__ __device__ long weights() const { return ow(nl - 1) + (long)W * nout; }
  __host__ __device__ long params() const { return weights() + ob(nl - 1) + nout; }
};
__host__ __device__ __forceinline__ size_t wf_index(int k, int n, int N) {
  return ((size_t)((k / 32) * (N / 16) + n / 16) * 64 + (k % 32) / 8 * 16 + n % 16) * 8 + k % 8;
}
__host__ __device__ __forceinline__ size_t wb_index(int k, int n, int K) {
  return ((size_t)((n / 32) * (K / 16) + k / 16) * 64 + (n % 32) / 8 * 16 + k % 16) * 8 + n % 8;
}

// Inputs and output gradients for the weight gradient, in MFMA operand order
// too: the fragment of points 32 q .. 32 q + 31 and columns 16 c .. 16 c + 15
// (width N) is the kilobyte q * N / 16 + c, its lanes 16 columns of each
// 8-point block in turn.  (8-point blocks of all columns, whose quarters of a
// fragment lie 4 KB apart, met in the same few L2 channels.)
__host__ __device__ __forceinline__ size_t pt_index(long p, int n, int N) {
  return ((size_t)(p / 32) * (N / 16) + n / 16) * 512 + ((p % 32) / 8 * 16 + n % 16) * 8 + p % 8;
}

// Where a pass takes its points from: rows idx[0..nv) of the resident set
// (bf16 inputs padded to K0, fp32 targets), or nv rows of x and y as the
// caller gave them.
struct Points {
  const bf16 *xs;
  const float *ys;
  const int *idx;
  const float *x;
  const float *y;
  int nv;
};

// exp by extended-precision reduction (Cody and Waite): x log2(e) as a rounded
// product and its remainder, 2^n times 2^f with |f| <= 1/2.  |x| <= 87, where
// neither end of the range is near.
__device__ __forceinline__ float exp_mid(float x) {
  const float c = 1.44269504088896340736f, c2 = (float)(1.44269504088896340736 - (double)c);
  const float t = x * c;
  const float lo = __builtin_fmaf(x, c2, __builtin_fmaf(x, c, -t));
  const float n = __builtin_rintf(t);
  return __builtin_ldexpf(__builtin_amdgcn_exp2f((t - n) + lo), (int)n);
}
// 1 / x for 1 <= x < 2^126: two Newton steps on the approximate reciprocal, the
// second on the quotient's remainder.  From a start within one unit they give
// the rounded quotient, but for a mantissa of all ones, where the start has to
// be it already, or the result is one unit below.  With gfx950's v_rcp_f32 no
// x of the range differs from the quotient (all compared).  No operand needs
// the scaling of a general division.
__device__ __forceinline__ float recip_mid(float x) {
  float r = __builtin_amdgcn_rcpf(x);
  r = __builtin_fmaf(__builtin_fmaf(-x, r, 1.0f), r, r);
  return __builtin_fmaf(__builtin_fmaf(-x, r, 1.0f), r, r);
}
// sigmoid of eight values: 16 instructions each where |z| <= 87, against 24 of
// expf and a division, which the rest take.  sigmoid_mid does the common ones
// without a branch (matrix instructions can go among them) and says whether
// they were all.
__device__ __forceinline__ bool sigmoid_mid(const float (&z)[2][4], float (&s)[2][4]) {
  float top = 0.0f;
  for (int t = 0; t < 2; t++)
    for (int r = 0; r < 4; r++) {
      s[t][r] = recip_mid(1.0f + exp_mid(-z[t][r]));
      top = fmaxf(top, fabsf(z[t][r]));
    }
  return top <= 87.0f;
}
__device__ __forceinline__ void sigmoid_rest(const float (&z)[2][4], float (&s)[2][4]) {
  for (int t = 0; t < 2; t++)
    for (int r = 0; r < 4; r++) s[t][r] = sigmoid(z[t][r]);
}
typedef bf16 bf16x4u __attribute__((ext_vector_type(4)));
// four FP32 -> BF16, round to nearest even (as to_bf16)
__device__ __forceinline__ bf16x4u to_bf16x4(const float (&f)[4]) {
  typedef float floatx2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const uint32_t a = __builtin_bit_cast(uint32_t, __builtin_convertvector((floatx2{f[0], f[1]}), bf16x2));
  const uint32_t b = __builtin_bit_cast(uint32_t, __builtin_convertvector((floatx2{f[2], f[3]}), bf16x2));
  return bf16x4u{(bf16)a, (bf16)(a >> 16), (bf16)b, (bf16)(b >> 16)};
}

constexpr int kTile = 32;  // points per block of k_net
constexpr int kPad = 8;    // bf16 added to a row in LDS: 16 rows then start in different banks

// The B fragments of two n tiles of a product of `steps` k steps (a shorter
// one loads its last step again).  No branch: a load in a branch would make
// every later wait one for all loads.
template <int T>
__device__ __forceinline__ void load_frags(bf16x8 *b, const bf16 *w, int steps, int tiles, int tile) {
  const int lane = threadIdx.x % kWave;
#pragma unroll
  for (int s = 0; s < T; s++)
    for (int t = 0; t < 2; t++)
      b[2 * s + t] = load8(w + ((size_t)(min(s, steps - 1) * tiles + tile + t) * 64 + lane) * 8);
}

// acc[n tile] of one wave: 16 points x 32 outputs, A rows in LDS
template <int T>
__device__ __forceinline__ void product(floatx4 (&acc)[2], const bf16 *a, int lda, const bf16x8 *b, int steps) {
  const int lane = threadIdx.x % kWave;
  for (int t = 0; t < 2; t++) acc[t] = floatx4{0, 0, 0, 0};
  const bf16 *r = a + (lane % 16) * lda + (lane / 16) * 8;
#pragma unroll
  for (int s = 0; s < T; s++) {
    if (s >= steps) continue;
    const bf16x8 x = load8(r + s * 32);
    for (int t = 0; t < 2; t++) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, b[2 * s + t], acc[t], 0, 0, 0);
  }
}
// N matrix instructions among the vector ones around them, one after every 10
// (a wave's activations of one half are 11 of them per matrix instruction).
template <int N>
__device__ __forceinline__ void interleave() {
#pragma unroll
  for (int i = 0; i < N; i++) {
    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x2, 10, 0);
  }
}

// Four values of one column n for points p, p+1, p+2, p+3 of the block (p a
// multiple of 4): into rows in LDS, and into the operand of the weight gradient.
__device__ __forceinline__ void put4(bf16 *rows, int ld, bf16 *op, int p0, int N, int p, int n,
                                     bf16x4u v) {
  for (int r = 0; r < 4; r++) rows[(p + r) * ld + n] = v[r];
  if (op) *reinterpret_cast<bf16x4u *>(op + pt_index(p0, 0, N) + pt_index(p, n, N)) = v;
}

// ---------------------------------------------------------------------------
// k_net: the whole network on kTile points per block.
//   PREDICT: the outputs of every point.
//   TRAIN: the forward pass, the loss and the data gradients back to the first
//   layer; the inputs and output gradients of every layer go to memory as
//   operands of k_weights.
// W is the width; W / 32 waves, each 32 outputs of a layer.  Activations stay
// in LDS as rows, all layers' in training (118 KB at 8 x 256; a deeper
// network's lower layers go through memory): the backward pass forms each
// pre-activation again from them, with the forward pass's own product, which
// costs a third more matrix work but no 4-byte value per activation to memory
// and back.  A layer's weights come from L2 into registers while the previous
// layer's activation is in work.
// Bound by the vector instructions of the SiLU and its derivative: they issue
// in 40 % of the SIMDs' cycles in training, whose two waves per SIMD wait for
// data or a barrier a third of their time, and in 63 % in inference; matrix
// instructions take 14 and 18 %.  Measured at 8 x 256 on 16384 points: 116 us,
// against 350 us for a launch per product (and one each for the batch, the loss
// and the last layer).  Inference of 12576 points takes 36 us, against 98 us, with the two
// halves of a block's points one behind the other (125 VGPRs: two blocks to a
// CU; both at once took 179 VGPRs and 45 us).
// ---------------------------------------------------------------------------
template <int W, bool TRAIN>
__global__ __launch_bounds__(2 * W) void k_net(const Net m, int slots, const Points pt, float *__restrict__ out,
                                               float *__restrict__ lossp) {
  constexpr int KS = W / 32, ld = W + kPad, kThreads = 2 * W;
  constexpr int KM = KS > 4 ? KS : 4;  // the first layer has up to 128 inputs
  extern __shared__ __align__(16) bf16 sm[];
  const int nl = m.nl, K0 = m.K0, nin = m.nin, nout = m.nout, ld0 = K0 + kPad;
  bf16 *sx = sm;                                 // [kTile][ld0]
  bf16 *sd = sx + kTile * ld0;                   // training: output gradients, 2 x [kTile][ld]
  bf16 *sh = sd + (TRAIN ? 2 * kTile * ld : 0);  // slots x [kTile][ld]
  float *sy = reinterpret_cast<float *>(sh + (size_t)slots * kTile * ld);  // training: targets, [kTile][nout]
  const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave;
  const int lp = lane / 16 * 4, ln = lane % 16;  // a lane's first point and column of a 16 x 16 result
  const int p0 = blockIdx.x * kTile;
  auto rows = [&](int j) { return sh + (size_t)(j % slots) * kTile * ld; };  // output of layer j

  bf16x8 b[2 * KM];
  load_frags<4>(b, m.wf, K0 / 32, W / 16, 2 * wave);

  // inputs and targets; every load of a round trip is made before the first is
  // waited for
  const int nx = kTile * K0 / 8, ny = kTile * nout;
  if (pt.xs) {
    constexpr int NI = (kTile * 128 / 8 + kThreads - 1) / kThreads;
    int q[NI], qy = 0;
#pragma unroll
    for (int j = 0; j < NI; j++) q[j] = pt.idx[min(p0 + min(tid + j * kThreads, nx - 1) / (K0 / 8), pt.nv - 1)];
    if (TRAIN) qy = pt.idx[min(p0 + min(tid, ny - 1) / nout, pt.nv - 1)];
    bf16x8 v[NI];
#pragma unroll
    for (int j = 0; j < NI; j++)
      v[j] = load8(pt.xs + (size_t)q[j] * K0 + min(tid + j * kThreads, nx - 1) % (K0 / 8) * 8);
    const float y = TRAIN ? pt.ys[(size_t)qy * nout + tid % nout] : 0.0f;
#pragma unroll
    for (int j = 0; j < NI; j++) {
      const int i = tid + j * kThreads, p = i / (K0 / 8), c = i % (K0 / 8) * 8;
      if (i < nx) *reinterpret_cast<bf16x8 *>(sx + p * ld0 + c) = p0 + p < pt.nv ? v[j] : bf16x8{};
    }
    if (TRAIN && tid < ny) sy[tid] = p0 + tid / nout < pt.nv ? y : 0.0f;
  } else {
    constexpr int NI = (kTile * 128 + kThreads - 1) / kThreads;
    float v[NI];
#pragma unroll
    for (int j = 0; j < NI; j++) {
      const int i = min(tid + j * kThreads, kTile * K0 - 1);
      v[j] = pt.x[(size_t)min(p0 + i / K0, pt.nv - 1) * nin + min(i % K0, nin - 1)];
    }
#pragma unroll
    for (int j = 0; j < NI; j++) {
      const int i = tid + j * kThreads, p = i / K0, c = i % K0;
      if (i < kTile * K0) sx[p * ld0 + c] = p0 + p < pt.nv && c < nin ? to_bf16(v[j]) : (bf16)0;
    }
  }
  if (TRAIN)
    for (int i = tid + (pt.xs ? kThreads : 0); i < ny; i += kThreads) {
      const int p = p0 + i / nout;
      float v = 0.0f;
      if (p < pt.nv) v = pt.xs ? pt.ys[(size_t)pt.idx[p] * nout + i % nout] : pt.y[(size_t)p0 * nout + i];
      sy[i] = v;
    }
  __syncthreads();
  if (TRAIN) {
    bf16 *xb = m.in;
    for (int i = tid; i < kTile / 8 * K0; i += kThreads) {
      const int q = i / K0, c = i % K0;
      bf16x8 v;
      for (int e = 0; e < 8; e++) v[e] = __builtin_bit_cast(__bf16, sx[(q * 8 + e) * ld0 + c]);
      *reinterpret_cast<bf16x8 *>(xb + pt_index(p0 + q * 8, c, K0)) = v;
    }
  }

  // forward: hidden layers
  for (int l = 0; l < nl - 1; l++) {
    float bl[2];
    for (int t = 0; t < 2; t++) bl[t] = m.b[l * W + wave * 32 + t * 16 + ln];
    const bf16 *in = l == 0 ? sx : rows(l - 1);
    bf16 *h = rows(l), *hb = TRAIN ? m.in + m.inp(l + 1) : nullptr;
    const bool last = l == nl - 2;  // (of the last layer every wave loads the two n tiles there are)
    const bf16 *wn = m.wf + m.frag(l + 1);
    // the second half's product runs among the first half's activations
    floatx4 acc[2][2];
    float z[2][4], s[2][4];
    auto pre = [&](int i) {
      for (int t = 0; t < 2; t++)
        for (int r = 0; r < 4; r++) z[t][r] = acc[i][t][r] + bl[t];
    };
    auto put = [&](int i, bool mid) {
      if (!mid) sigmoid_rest(z, s);
      for (int t = 0; t < 2; t++) {
        float v[4];
        for (int r = 0; r < 4; r++) v[r] = z[t][r] * s[t][r];
        put4(h, ld, hb, p0, W, i * 16 + lp, wave * 32 + t * 16 + ln, to_bf16x4(v));
      }
    };
    bool mid;
    if (l == 0) {
      product<4>(acc[0], in, ld0, b, K0 / 32);
      product<4>(acc[1], in + 16 * ld0, ld0, b, K0 / 32);
      pre(0);
      mid = sigmoid_mid(z, s);
    } else {
      product<KS>(acc[0], in, ld, b, KS);
      pre(0);
      product<KS>(acc[1], in + 16 * ld, ld, b, KS);
      mid = sigmoid_mid(z, s);
      interleave<2 * KS>();
    }
    load_frags<KS>(b, wn, KS, last ? kOut / 16 : W / 16, last ? 0 : 2 * wave);
    put(0, mid);
    pre(1);
    mid = sigmoid_mid(z, s);
    put(1, mid);
    __syncthreads();
    if (TRAIN && l + slots <= nl - 2)
      for (int i = tid; i < kTile * W / 8; i += kThreads) {
        const int p = i / (W / 8), c = i % (W / 8) * 8;
        *reinterpret_cast<bf16x8 *>(m.h + m.out(l) + (size_t)(p0 + p) * W + c) = load8(h + p * ld + c);
      }
  }

  // last layer: wave 0 the first 16 points, wave 1 the others
  float *sq = reinterpret_cast<float *>(sd + kTile * ld);  // squared errors, [kTile * kOut]
  if (wave < 2) {
    floatx4 o[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
    const bf16 *r = rows(nl - 2) + (wave * 16 + ln) * ld + (lane / 16) * 8;
#pragma unroll
    for (int s = 0; s < KS; s++) {
      const bf16x8 a = load8(r + s * 32);
      for (int t = 0; t < 2; t++) o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[2 * s + t], o[t], 0, 0, 0);
    }
    for (int t = 0; t < 2; t++) {
      const int n = t * 16 + ln;
      const float bn = n < nout ? m.b[(nl - 1) * W + n] : 0.0f;
      float v[4];
      for (int q = 0; q < 4; q++) {
        const int p = wave * 16 + lp + q;
        const bool real = p0 + p < pt.nv && n < nout;
        const float z = o[t][q] + bn;
        if (!TRAIN) {
          if (real) out[(size_t)(p0 + p) * nout + n] = z;
          continue;
        }
        // loss = mean of squares; dZ = bf16(2 (z - y) / (nv nout)), zero on padding
        float e2 = 0, g = 0;
        if (real) {
          const float e = z - sy[p * nout + n];
          e2 = e * e;
          g = 2.0f * e / ((float)pt.nv * (float)nout);
        }
        v[q] = g;
        sq[p * kOut + n] = e2;
      }
      if (TRAIN) put4(sd, ld, m.dz + m.out(nl - 1), p0, kOut, wave * 16 + lp, n, to_bf16x4(v));
    }
  }
  if (!TRAIN) return;
  bf16x8 c[2 * KS];
  load_frags<1>(c, m.wb + m.frag(nl - 1), 1, W / 16, 2 * wave);
  load_frags<KM>(b, m.wf + m.frag(nl - 2), m.K(nl - 2) / 32, W / 16, 2 * wave);
  __syncthreads();
  // the sums of squares of 8 points each, by a fixed tree
  for (int w = 128; w > 0; w >>= 1) {
    for (int i = tid; i < kTile / 8 * w; i += kThreads) {
      float *s = sq + i / w * 256 + i % w;
      s[0] += s[w];
    }
    __syncthreads();
  }
  if (tid < kTile / 8) lossp[blockIdx.x * (kTile / 8) + tid] = sq[tid * 256];
  __syncthreads();  // the second gradient buffer holds the squares no longer

  // backward: dZ of layer l - 1 from dZ of layer l
  for (int l = nl - 1; l >= 1; l--) {
    const bf16 *cur = sd + ((nl - 1 - l) & 1) * kTile * ld;
    bf16 *nxt = sd + ((nl - l) & 1) * kTile * ld;
    if (l >= 2 && l - 2 + slots <= nl - 2) {  // the input rows of layer l - 1 have left LDS
      bf16 *h = rows(l - 2);
      for (int i = tid; i < kTile * W / 8; i += kThreads) {
        const int p = i / (W / 8), k = i % (W / 8) * 8;
        *reinterpret_cast<bf16x8 *>(h + p * ld + k) = load8(m.h + m.out(l - 2) + (size_t)(p0 + p) * W + k);
      }
      __syncthreads();
    }
    float bl[2];
    for (int t = 0; t < 2; t++) bl[t] = m.b[(l - 1) * W + wave * 32 + t * 16 + ln];
    floatx4 acc[2][2], z4[2][2];
    for (int i = 0; i < 2; i++) {
      if (l == nl - 1)
        product<1>(acc[i], cur + i * 16 * ld, ld, c, 1);
      else
        product<KS>(acc[i], cur + i * 16 * ld, ld, c, KS);
      if (l == 1)
        product<4>(z4[i], sx + i * 16 * ld0, ld0, b, K0 / 32);
      else
        product<KS>(z4[i], rows(l - 2) + i * 16 * ld, ld, b, KS);
    }
    const int j = max(l - 2, 0);  // (the last round loads what it does not use)
    load_frags<KS>(c, m.wb + m.frag(j + 1), m.N(j + 1) / 32, W / 16, 2 * wave);
    load_frags<KM>(b, m.wf + m.frag(j), m.K(j) / 32, W / 16, 2 * wave);
    for (int i = 0; i < 2; i++) {
      float z[2][4], s[2][4];
      for (int t = 0; t < 2; t++)
        for (int r = 0; r < 4; r++) z[t][r] = z4[i][t][r] + bl[t];
      if (!sigmoid_mid(z, s)) sigmoid_rest(z, s);
      for (int t = 0; t < 2; t++) {
        float v[4];
        for (int r = 0; r < 4; r++) v[r] = acc[i][t][r] * (s[t][r] * (1.0f + z[t][r] * (1.0f - s[t][r])));
        put4(nxt, ld, m.dz + m.out(l - 1), p0, W, i * 16 + lp, wave * 32 + t * 16 + ln, to_bf16x4(v));
      }
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// k_weights: weight and bias gradients of every layer from the inputs and
// output gradients, and Adam on them (or the gradients themselves).
// A block owns 32 k x 64 n (32 k x 32 n of the last layer) over all points,
// a wave 32 k x 32 n: partial products of kChunk points (32 at a time, in
// MFMA order), added in chunk order, so the result does not depend on the
// launch.  Operands go straight from memory to registers, kFlight steps of 32
// points ahead.  The bias sums are blocks of their own (beside a block's
// products they took as long again).  Blocks of one layer share an XCD (block
// b: XCD b % 8, layer b % 8 of each eight), so its L2 reads each operand once.
// Adam runs on the sum while it is in registers: FP32 master weights, then the
// BF16 fragments of the next step's products.
// Bound by the operands' way from L2 into the CUs, 8 KB per block and 32
// points (with every block on the same 16 steps it takes 5 us less; 8 to 24
// steps in flight make no difference).  Measured at 8 x 256, 16384 points: 60
// us, against 192 us for a launch per layer for the partial products, the bias
// sums and each update, with the partial products in memory.
// A network of few such blocks leaves CUs idle, and its one walk over the points
// of a large batch is the time: the points are then split over `splits` rows of
// blocks (each a whole number of kSplit steps), which leave partial gradients
// in memory, and k_apply adds these up in order and takes Adam's step
// (weight_splits).  A training step, one walk -> split: 64 x 2 layers, 16 384
// points 99 -> 64 us, 131 072 points 474 -> 179 us; 128 x 2, 400 000 points 1890
// -> 653 us; 256 x 3, 32 768 points 223 -> 183 us.
// ---------------------------------------------------------------------------
struct WeightTile {
  int layer, k0, n0;  // layer -1: no work; k0 -1: the bias sums of 16 columns
};
struct AdamStep {
  float lr, c1, c2;
};
struct Moments {
  float *m1, *m2, *m1b, *m2b;
};
constexpr int kFlight = 16;
constexpr int kSplit = 64;  // steps (of 32 points): 8 chunks, an iteration of bias_sums
constexpr int kSplitSteps = 512;

// One Adam step on parameter p[o].
__device__ __forceinline__ float adam(float *p, float *m1, float *m2, size_t o, float g, const AdamStep &st) {
  const float a = 0.9f * m1[o] + 0.1f * g;
  const float v = 0.999f * m2[o] + 0.001f * g * g;
  m1[o] = a;
  m2[o] = v;
  const float x = p[o] - st.lr * (a / st.c1) / (sqrtf(v / st.c2) + 1e-8f);
  p[o] = x;
  return x;
}

// Bias gradients of columns n0 .. n0 + 15 of layer l (two waves): a lane takes
// one column of one chunk, sums the 8-point blocks j, j + 8, ... of the chunk
// for each j, then the eight sums, and the chunks add up in order.
// (steps first .. end - 1 of 32 points, four 8-point blocks each)
template <bool ADAM>
__device__ __forceinline__ void bias_sums(const Net &m, int l, int n0, int first, int end, const AdamStep &st,
                                          const Moments &mo, float *gb) {
  __shared__ float part[8][16];
  const int tid = threadIdx.x, N = m.N(l), c0 = tid / 16, nblk = end * 4;
  const bf16 *d = m.dz + m.out(l);
  float sum = 0.0f;
  for (int b0 = first * 4; b0 < nblk; b0 += 8 * (kChunk / 8)) {
    const int b = b0 + c0 * (kChunk / 8);
    float s[8];
#pragma unroll
    for (int j = 0; j < 8; j++) s[j] = 0.0f;
#pragma unroll
    for (int i = 0; i < kChunk / 64; i++)
      if (b + 8 * i < nblk) {
        bf16x8 v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = load8(d + pt_index((long)(b + 8 * i + j) * 8, n0 + tid % 16, N));
#pragma unroll
        for (int j = 0; j < 8; j++)
          for (int e = 0; e < 8; e++) s[j] += (float)v[j][e];
      }
    float t = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; j++) t += s[j];
    part[c0][tid % 16] = t;
    __syncthreads();
    if (tid < 16)
      for (int c = 0; c < 8; c++)
        if (b0 + c * (kChunk / 8) < nblk) sum += part[c][tid];
    __syncthreads();
  }
  if (tid >= 16 || n0 + tid >= m.n(l)) return;
  const size_t o = m.ob(l) + n0 + tid;
  if (ADAM)
    adam(m.b, mo.m1b, mo.m2b, o, sum, st);
  else
    gb[o] = sum;
}

template <bool ADAM>
__global__ __launch_bounds__(128, 1) void k_weights(const Net m, const WeightTile *__restrict__ tiles,
                                                    const AdamStep st, const Moments mo, float *__restrict__ gw,
                                                    float *__restrict__ gb) {
  // row r of blocks: the tiles of a layer one XCD further on than row r - 1's
  const int row = blockIdx.y, rows = gridDim.y;
  const WeightTile tl = tiles[blockIdx.x / 8 * 8 + (blockIdx.x + 8 - row % 8) % 8];
  const int units = (int)((m.P / 32 + kSplit - 1) / kSplit);
  const int first = units * row / rows * kSplit, end = min(units * (row + 1) / rows * kSplit, (int)(m.P / 32));
  if (rows > 1) {
    gw += (size_t)row * m.params();
    gb += (size_t)row * m.params();
  }
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int l = tl.layer, n0 = tl.n0 + wave * 32;
  if (l < 0) return;
  if (tl.k0 < 0) {
    bias_sums<ADAM>(m, l, tl.n0, first, end, st, mo, gb);
    return;
  }
  const int K = m.K(l), N = m.N(l), rk = m.k(l), rn = m.n(l);
  if (n0 >= N) return;
  const int nstep = end - first;  // a multiple of 4
  // the step to load next (its last one again past the end): uniform bases
  // and a lane's offset, so that a step costs a few scalar additions
  const bf16 *x = m.in + m.inp(l) + (size_t)first * 32 * K + tl.k0 / 16 * 512,
             *d = m.dz + m.out(l) + (size_t)first * 32 * N + n0 / 16 * 512;
  int left = nstep - 1;
  bf16x8 a[kFlight][2], b[kFlight][2];
  auto fetch = [&](int slot) {
    for (int t = 0; t < 2; t++) {
      a[slot][t] = load8(x + lane * 8 + t * 512);
      b[slot][t] = load8(d + lane * 8 + t * 512);
    }
    x += left > 0 ? 32 * K : 0;
    d += left > 0 ? 32 * N : 0;
    left--;
  };
  floatx4 acc[2][2], sum[2][2];
  for (int i = 0; i < 2; i++)
    for (int t = 0; t < 2; t++) acc[i][t] = sum[i][t] = floatx4{0, 0, 0, 0};
#pragma unroll
  for (int i = 0; i < kFlight; i++) fetch(i);
  for (int s0 = 0; s0 < nstep; s0 += kFlight) {
#pragma unroll
    for (int g = 0; g < kFlight / 4; g++) {
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int i = g * 4 + q;
        if (s0 + g * 4 < nstep)
          for (int u = 0; u < 2; u++)
            for (int t = 0; t < 2; t++)
              acc[u][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i][u], b[i][t], acc[u][t], 0, 0, 0);
        fetch(i);
      }
      const int done = s0 + g * 4 + 4;  // steps done
      if (done <= nstep && (done % (kChunk / 32) == 0 || done == nstep)) {
        for (int u = 0; u < 2; u++)
          for (int t = 0; t < 2; t++)
            for (int r = 0; r < 4; r++) {
              sum[u][t][r] += acc[u][t][r];
              acc[u][t][r] = 0.0f;
            }
      }
    }
  }
  for (int u = 0; u < 2; u++)
    for (int t = 0; t < 2; t++)
      for (int r = 0; r < 4; r++) {
        const int k = tl.k0 + u * 16 + lane / 16 * 4 + r, n = n0 + t * 16 + lane % 16;
        if (k >= rk || n >= rn) continue;
        const size_t o = m.ow(l) + (size_t)k * rn + n;
        const float gi = sum[u][t][r];
        if (!ADAM) {
          gw[o] = gi;
          continue;
        }
        const bf16 h = to_bf16(adam(m.w, mo.m1, mo.m2, o, gi, st));
        m.wf[m.frag(l) + wf_index(k, n, N)] = h;
        m.wb[m.frag(l) + wb_index(k, n, K)] = h;
      }
}

// The gradients of layer blockIdx.y: the sums over the splits' partial ones, in
// order, and Adam's step on them (or the gradients themselves).
template <bool ADAM>
__global__ __launch_bounds__(256) void k_apply(const Net m, int splits, const float *__restrict__ part,
                                               const AdamStep st, const Moments mo, float *__restrict__ gw,
                                               float *__restrict__ gb) {
  const int l = blockIdx.y, rk = m.k(l), rn = m.n(l), nw = rk * rn;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= nw + rn) return;
  const size_t o = i < nw ? m.ow(l) + i : m.ob(l) + (i - nw);
  const float *p = part + (i < nw ? o : m.weights() + o);
  float g = p[0];
  for (int q = 1; q < splits; q++) g += p[(size_t)q * m.params()];
  if (!ADAM) {
    (i < nw ? gw : gb)[o] = g;
  } else if (i >= nw) {
    adam(m.b, mo.m1b, mo.m2b, o, g, st);
  } else {
    const int k = i / rn, n = i % rn;
    const bf16 h = to_bf16(adam(m.w, mo.m1, mo.m2, o, g, st));
    m.wf[m.frag(l) + wf_index(k, n, m.N(l))] = h;
    m.wb[m.frag(l) + wb_index(k, n, m.K(l))] = h;
  }
}

// Batch losses of an epoch, one block per step: scale * (sum of the step's n
// partials), thread t summing t, t + 256, ... then a fixed tree (reproducible).
__global__ __launch_bounds__(256) void k_losses(const float *__restrict__ part, int n, float scale, float scale_last,
                                                float *__restrict__ out) {
  __shared__ double sh[256];
  part += (size_t)blockIdx.x * n;
  double a = 0;
  for (int i = threadIdx.x; i < n; i += 256) a += part[i];
  sh[threadIdx.x] = a;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[blockIdx.x] = (float)(sh[0] * (blockIdx.x == gridDim.x - 1 ? scale_last : scale));
}

__global__ void k_mfma_check(const bf16 *a, const bf16 *b, float *d) {
  const int lane = threadIdx.x;
  bf16x8 av, bv;
  for (int e = 0; e < 8; e++) {
    const int k = (lane / 16) * 8 + e;
    uint16_t ab = a[(lane % 16) * 32 + k], bb = b[k * 16 + lane % 16];
    av[e] = __builtin_bit_cast(__bf16, ab);
    bv[e] = __builtin_bit_cast(__bf16, bb);
  }
  floatx4 c = {0, 0, 0, 0};
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, c, 0, 0, 0);
  for (int r = 0; r < 4; r++) d[((lane / 16) * 4 + r) * 16 + lane % 16] = c[r];
}

// BF16 fragments of the weights of layers l0 + blockIdx.y from the FP32 masters;
// the padding stays zero.
constexpr int kPackLayers = 32768;  // (a launch has at most 65536 blocks along y)
__global__ __launch_bounds__(256) void k_pack(const Net m, int l0) {
  const int l = l0 + blockIdx.y, i = blockIdx.x * 256 + threadIdx.x;
  if (i >= m.k(l) * m.n(l)) return;
  const int k = i / m.n(l), n = i % m.n(l);
  const bf16 h = to_bf16(m.w[m.ow(l) + i]);
  m.wf[m.frag(l) + wf_index(k, n, m.N(l))] = h;
  m.wb[m.frag(l) + wb_index(k, n, m.K(l))] = h;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// A device buffer that grows and is kept for the next call.
struct Buf {
  void *p = nullptr;
  size_t bytes = 0;
};

}  // namespace usgmlp

using namespace usgmlp;

struct usg_mlp {
  usg_mlp_desc d{};
  long nw = 0, nb = 0;
  Net net{};
  Moments mo{};
  hipStream_t s = nullptr;
  std::vector<void *> allocs;
  long step = 0;
  WeightTile *d_tiles = nullptr;
  int ntiles = 0, nwork = 0;  // blocks of k_weights, and those of them with work
  int cus = 0;
  int slots = 0;              // layers whose rows LDS holds in training
  size_t lds_train = 0, lds_predict = 0;
  // training buffers for `cap` points (Net's in, dz and h)
  int cap = 0;
  std::vector<void *> bufs;
  Buf x, y, g, part, lossp, losses, idx;
  // resident training set
  bf16 *xs = nullptr;
  float *ys = nullptr;
  long nset = 0;
};

namespace usgmlp {

template <typename T>
int dalloc(std::vector<void *> &v, T **p, size_t n) {
  void *q = nullptr;
  HIPCHK(hipMalloc(&q, std::max<size_t>(n, 1) * sizeof(T)));
  v.push_back(q);
  *p = (T *)q;
  return 0;
}

int grow(usg_mlp *m, Buf &b, size_t bytes) {
  if (bytes <= b.bytes) return 0;
  HIPCHK(hipStreamSynchronize(m->s));
  if (b.p) hipFree(b.p);
  b.p = nullptr;
  b.bytes = 0;
  HIPCHK(hipMalloc(&b.p, bytes));
  b.bytes = bytes;
  return 0;
}

int round_up(int a, int b) { return (a + b - 1) / b * b; }

// Training buffers for P points (a multiple of 128).
int ensure_cap(usg_mlp *m, int P) {
  Net &t = m->net;
  t.P = P;
  if (P <= m->cap) return 0;
  HIPCHK(hipStreamSynchronize(m->s));
  for (void *p : m->bufs) hipFree(p);
  m->bufs.clear();
  m->cap = 0;
  int rc = 0;
  if ((rc = dalloc(m->bufs, &t.in, (size_t)t.inp(t.nl))) ||
      (rc = dalloc(m->bufs, &t.dz, (size_t)t.out(t.nl - 1) + (size_t)P * kOut)) ||
      (m->slots < t.nl - 1 && (rc = dalloc(m->bufs, &t.h, (size_t)t.out(t.nl - 1)))))
    return rc;
  m->cap = P;
  return 0;
}

template <int W>
int net_lds(usg_mlp *m, int limit) {
  const size_t row = (size_t)kTile * (W + kPad) * sizeof(bf16), x = (size_t)kTile * (m->net.K0 + kPad) * sizeof(bf16),
               y = (size_t)kTile * m->d.nout * sizeof(float);
  m->slots = std::min<int>(m->net.nl - 1, (int)(((size_t)limit - x - y) / row) - 2);
  m->slots = std::max(m->slots, 2);
  m->lds_train = x + y + (2 + m->slots) * row;
  m->lds_predict = x + 2 * row;
  // what is set holds for every network of this width: the device's most
  for (const void *f :
       {reinterpret_cast<const void *>(&k_net<W, true>), reinterpret_cast<const void *>(&k_net<W, false>)})
    HIPCHK(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, limit));
  return 0;
}

template <int W>
void launch_net(usg_mlp *m, bool train, int blocks, const Points &pt, float *out, float *lossp) {
  if (train)
    hipLaunchKernelGGL((k_net<W, true>), dim3(blocks), dim3(2 * W), m->lds_train, m->s, m->net, m->slots, pt, out,
                       lossp);
  else
    hipLaunchKernelGGL((k_net<W, false>), dim3(blocks), dim3(2 * W), m->lds_predict, m->s, m->net, 2, pt, out, lossp);
}

void net(usg_mlp *m, bool train, int blocks, const Points &pt, float *out, float *lossp) {
  switch (m->d.width) {
    case 64: launch_net<64>(m, train, blocks, pt, out, lossp); break;
    case 128: launch_net<128>(m, train, blocks, pt, out, lossp); break;
    case 192: launch_net<192>(m, train, blocks, pt, out, lossp); break;
    default: launch_net<256>(m, train, blocks, pt, out, lossp); break;
  }
}

// The blocks of k_weights: block b works on a layer l with l % 8 == b % 8, so
// that a layer's blocks run on one XCD.
int build_tiles(usg_mlp *m) {
  std::vector<WeightTile> by[8], all;
  for (int l = 0; l < m->net.nl; l++)
    for (int k0 = 0; k0 < m->net.K(l); k0 += 32)
      for (int n0 = 0; n0 < m->net.N(l); n0 += 64) by[l % 8].push_back({l, k0, n0});
  for (int l = 0; l < m->net.nl; l++)
    for (int n0 = 0; n0 < m->net.n(l); n0 += 16) by[l % 8].push_back({l, -1, n0});
  size_t most = 0;
  for (auto &v : by) {
    most = std::max(most, v.size());
    m->nwork += (int)v.size();
  }
  for (size_t i = 0; i < most; i++)
    for (auto &v : by) all.push_back(i < v.size() ? v[i] : WeightTile{-1, 0, 0});
  m->ntiles = (int)all.size();
  if (int rc = dalloc(m->allocs, &m->d_tiles, all.size())) return rc;
  HIPCHK(hipMemcpy(m->d_tiles, all.data(), all.size() * sizeof(WeightTile), hipMemcpyHostToDevice));
  return 0;
}

// Rows of blocks that k_weights splits a batch's points over: as many as the
// CUs take beside one another, if the second launch is repaid.  Split from 64
// steps on, training gained at every size (8192 points: 84 -> 69 us), but the
// gradients of one batch lost (4096 points: 109 -> 130 us, 8192: 147 -> 159,
// 16 384: 227 -> 224).
int weight_splits(const usg_mlp *m) {
  const int steps = (int)(m->net.P / 32), units = (steps + kSplit - 1) / kSplit;
  return steps < kSplitSteps ? 1 : std::max(1, std::min(units, m->cus / m->nwork));
}

// The partial gradients' memory, before a step's first launch.
int ensure_parts(usg_mlp *m) {
  const int splits = weight_splits(m);
  return splits > 1 ? grow(m, m->part, (size_t)splits * m->net.params() * sizeof(float)) : 0;
}

// Weight and bias gradients of the points k_net went through, and Adam on them
// (or the gradients themselves, into gw and gb).
template <bool ADAM>
void weights(usg_mlp *m, const AdamStep &st, float *gw, float *gb) {
  const int splits = weight_splits(m);
  if (splits == 1) {
    hipLaunchKernelGGL((k_weights<ADAM>), dim3(m->ntiles), dim3(128), 0, m->s, m->net, m->d_tiles, st, m->mo, gw, gb);
    return;
  }
  float *part = (float *)m->part.p;
  hipLaunchKernelGGL((k_weights<false>), dim3(m->ntiles, splits), dim3(128), 0, m->s, m->net, m->d_tiles, st, m->mo,
                     part, part + m->nw);
  const int most = (std::max(m->d.nin, m->d.width) + 1) * m->d.width;
  hipLaunchKernelGGL((k_apply<ADAM>), dim3((most + 255) / 256, m->net.nl), dim3(256), 0, m->s, m->net, splits, part, st,
                     m->mo, gw, gb);
}

}  // namespace usgmlp

extern "C" {

const char *usg_mlp_last_error(void) { return usgmlp::g_err.c_str(); }

int usg_mlp_sizes(const usg_mlp_desc *d, long *nw, long *nb) {
  if (!d || !nw || !nb) return fail(-1, "null argument");
  if (d->nin < 1 || d->nin > 128 || d->width < 64 || d->width > 256 || d->width % 64 || d->nlayer < 2 ||
      d->nout < 1 || d->nout > 16)
    return fail(-1, "network shape out of range (nin <= 128, width multiple of 64 <= 256, nout <= 16)");
  *nw = (long)d->nin * d->width + (long)(d->nlayer - 2) * d->width * d->width + (long)d->width * d->nout;
  *nb = (long)(d->nlayer - 1) * d->width + d->nout;
  return 0;
}

int usg_mlp_destroy(usg_mlp *m) {
  if (!m) return 0;
  if (m->s) hipStreamSynchronize(m->s);
  for (void *p : m->bufs) hipFree(p);
  for (void *p : m->allocs) hipFree(p);
  for (Buf *b : {&m->x, &m->y, &m->g, &m->part, &m->lossp, &m->losses, &m->idx})
    if (b->p) hipFree(b->p);
  if (m->xs) hipFree(m->xs);
  if (m->ys) hipFree(m->ys);
  if (m->s) hipStreamDestroy(m->s);
  delete m;
  return 0;
}

static int create(usg_mlp *m) {
  const usg_mlp_desc &d = m->d;
  HIPCHK(hipStreamCreate(&m->s));
  Net &t = m->net;
  t.nl = d.nlayer;
  t.W = d.width;
  t.K0 = round_up(d.nin, 64);
  t.nin = d.nin;
  t.nout = d.nout;
  const size_t frags = t.frag(t.nl - 1) + (size_t)t.W * kOut;
  int rc = 0, dev = 0, limit = 0;
  if ((rc = dalloc(m->allocs, &t.wf, frags)) || (rc = dalloc(m->allocs, &t.wb, frags)) ||
      (rc = dalloc(m->allocs, &t.w, m->nw)) || (rc = dalloc(m->allocs, &t.b, m->nb)) ||
      (rc = dalloc(m->allocs, &m->mo.m1, m->nw)) || (rc = dalloc(m->allocs, &m->mo.m2, m->nw)) ||
      (rc = dalloc(m->allocs, &m->mo.m1b, m->nb)) || (rc = dalloc(m->allocs, &m->mo.m2b, m->nb)) ||
      (rc = build_tiles(m)))
    return rc;
  for (bf16 *p : {t.wf, t.wb}) HIPCHK(hipMemsetAsync(p, 0, frags * sizeof(bf16), m->s));
  HIPCHK(hipGetDevice(&dev));
  HIPCHK(hipDeviceGetAttribute(&limit, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
  HIPCHK(hipDeviceGetAttribute(&m->cus, hipDeviceAttributeMultiprocessorCount, dev));
  switch (d.width) {
    case 64: return net_lds<64>(m, limit);
    case 128: return net_lds<128>(m, limit);
    case 192: return net_lds<192>(m, limit);
    default: return net_lds<256>(m, limit);
  }
}

int usg_mlp_create(const usg_mlp_desc *d, usg_mlp **out) {
  long nw, nb;
  if (!out) return fail(-1, "null argument");
  *out = nullptr;
  int rc = usg_mlp_sizes(d, &nw, &nb);
  if (rc) return rc;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return fail(-2, "no GPU visible");
  usg_mlp *m = new usg_mlp();
  m->d = *d;
  m->nw = nw;
  m->nb = nb;
  // zero parameters until set
  std::vector<float> w(nw, 0.0f), b(nb, 0.0f);
  if ((rc = create(m)) || (rc = usg_mlp_set_params(m, w.data(), b.data()))) {
    usg_mlp_destroy(m);
    return rc;
  }
  *out = m;
  return 0;
}

int usg_mlp_set_params(usg_mlp *m, const float *w, const float *b) {
  if (!m || !w || !b) return fail(-1, "null argument");
  HIPCHK(hipMemcpyAsync(m->net.w, w, m->nw * sizeof(float), hipMemcpyHostToDevice, m->s));
  HIPCHK(hipMemcpyAsync(m->net.b, b, m->nb * sizeof(float), hipMemcpyHostToDevice, m->s));
  for (float *p : {m->mo.m1, m->mo.m2}) HIPCHK(hipMemsetAsync(p, 0, m->nw * sizeof(float), m->s));
  for (float *p : {m->mo.m1b, m->mo.m2b}) HIPCHK(hipMemsetAsync(p, 0, m->nb * sizeof(float), m->s));
  const int most = std::max(m->d.nin, m->d.width) * m->d.width;
  for (int l0 = 0; l0 < m->net.nl; l0 += kPackLayers)
    hipLaunchKernelGGL(k_pack, dim3((most + 255) / 256, std::min(m->net.nl - l0, kPackLayers)), dim3(256), 0, m->s,
                       m->net, l0);
  HIPCHK(hipGetLastError());
  m->step = 0;
  HIPCHK(hipStreamSynchronize(m->s));
  return 0;
}

int usg_mlp_get_params(usg_mlp *m, float *w, float *b) {
  if (!m || !w || !b) return fail(-1, "null argument");
  HIPCHK(hipMemcpyAsync(w, m->net.w, m->nw * sizeof(float), hipMemcpyDeviceToHost, m->s));
  HIPCHK(hipMemcpyAsync(b, m->net.b, m->nb * sizeof(float), hipMemcpyDeviceToHost, m->s));
  HIPCHK(hipStreamSynchronize(m->s));
  return 0;
}

// The caller's rows on the device.
static int upload_points(usg_mlp *m, const float *x, const float *y, int n, Points &pt) {
  const size_t bx = (size_t)n * m->d.nin * sizeof(float), by = (size_t)n * m->d.nout * sizeof(float);
  int rc = grow(m, m->x, bx);
  if (rc || (rc = grow(m, m->y, by))) return rc;
  HIPCHK(hipMemcpyAsync(m->x.p, x, bx, hipMemcpyHostToDevice, m->s));
  if (y) HIPCHK(hipMemcpyAsync(m->y.p, y, by, hipMemcpyHostToDevice, m->s));
  pt = Points{nullptr, nullptr, nullptr, (const float *)m->x.p, y ? (const float *)m->y.p : nullptr, n};
  return 0;
}

int usg_mlp_predict(usg_mlp *m, const float *x, long n, float *y) {
  if (!m || !x || !y || n < 0) return fail(-1, "bad argument");
  const int step = 262144;  // bounds the device copies of x and y
  const int nout = m->d.nout;
  for (long a = 0; a < n; a += step) {
    const int cnt = (int)std::min<long>(step, n - a);
    Points pt;
    if (int rc = upload_points(m, x + a * m->d.nin, nullptr, cnt, pt)) return rc;
    net(m, false, (cnt + kTile - 1) / kTile, pt, (float *)m->y.p, nullptr);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(y + a * nout, m->y.p, (size_t)cnt * nout * sizeof(float), hipMemcpyDeviceToHost, m->s));
  }
  HIPCHK(hipStreamSynchronize(m->s));
  return 0;
}

int usg_mlp_gradients(usg_mlp *m, const float *x, const float *y, int n, float *loss, float *dw, float *db) {
  if (!m || !x || !y || n <= 0) return fail(-1, "bad argument");
  const int P = round_up(n, 128), nbl = P / 8;
  int rc = ensure_cap(m, P);
  if (rc || (rc = ensure_parts(m)) || (rc = grow(m, m->lossp, nbl * sizeof(float))) ||
      (rc = grow(m, m->g, (m->nw + m->nb) * sizeof(float))))
    return rc;
  Points pt;
  if ((rc = upload_points(m, x, y, n, pt))) return rc;
  float *gw = (float *)m->g.p, *gb = gw + m->nw;
  net(m, true, P / kTile, pt, nullptr, (float *)m->lossp.p);
  weights<false>(m, AdamStep{}, gw, gb);
  HIPCHK(hipGetLastError());
  std::vector<float> lp(loss ? nbl : 0);
  if (loss) HIPCHK(hipMemcpyAsync(lp.data(), m->lossp.p, nbl * sizeof(float), hipMemcpyDeviceToHost, m->s));
  if (dw) HIPCHK(hipMemcpyAsync(dw, gw, m->nw * sizeof(float), hipMemcpyDeviceToHost, m->s));
  if (db) HIPCHK(hipMemcpyAsync(db, gb, m->nb * sizeof(float), hipMemcpyDeviceToHost, m->s));
  HIPCHK(hipStreamSynchronize(m->s));
  if (loss) {
    double s = 0;
    for (float v : lp) s += v;
    *loss = (float)(s / ((double)n * m->d.nout));
  }
  return 0;
}

int usg_mlp_set_data(usg_mlp *m, const float *x, const float *y, long n) {
  if (!m || !x || !y || n <= 0) return fail(-1, "bad argument");
  // the old set is gone from here on: a failure below leaves no data set
  m->nset = 0;
  if (m->xs || m->ys) {
    HIPCHK(hipStreamSynchronize(m->s));
    if (m->xs) hipFree(m->xs);
    if (m->ys) hipFree(m->ys);
    m->xs = nullptr;
    m->ys = nullptr;
  }
  const int K0 = m->net.K0, nin = m->d.nin, nout = m->d.nout;
  std::vector<bf16> X((size_t)n * K0, 0);
  for (long p = 0; p < n; p++)
    for (int k = 0; k < nin; k++) X[(size_t)p * K0 + k] = to_bf16(x[(size_t)p * nin + k]);
  HIPCHK(hipMalloc(&m->xs, X.size() * 2));
  HIPCHK(hipMalloc(&m->ys, (size_t)n * nout * 4));
  HIPCHK(hipMemcpyAsync(m->xs, X.data(), X.size() * 2, hipMemcpyHostToDevice, m->s));
  HIPCHK(hipMemcpyAsync(m->ys, y, (size_t)n * nout * 4, hipMemcpyHostToDevice, m->s));
  HIPCHK(hipStreamSynchronize(m->s));
  m->nset = n;
  return 0;
}

int usg_mlp_train_epoch(usg_mlp *m, const int *perm, long n, int batch, float lr, float *loss_out) {
  if (!m || !perm || n <= 0 || batch <= 0) return fail(-1, "bad argument");
  if (n != m->nset) return fail(-1, "perm length differs from the training set");
  for (long i = 0; i < n; i++)
    if (perm[i] < 0 || perm[i] >= n) return fail(-1, "perm entry out of range");
  const int P = round_up(batch, 128), nbl = P / 8;
  const long nsteps = (n + batch - 1) / batch;
  int rc = ensure_cap(m, P);
  if (rc || (rc = ensure_parts(m)) || (rc = grow(m, m->idx, n * sizeof(int))) ||
      (rc = grow(m, m->lossp, (size_t)nsteps * nbl * sizeof(float))) || (rc = grow(m, m->losses, nsteps * sizeof(float))))
    return rc;
  HIPCHK(hipMemcpyAsync(m->idx.p, perm, n * sizeof(int), hipMemcpyHostToDevice, m->s));
  float *lossp = (float *)m->lossp.p;
  int nv = 0;
  for (long q = 0; q < nsteps; q++) {
    nv = (int)std::min<long>(batch, n - q * batch);
    net(m, true, P / kTile, Points{m->xs, m->ys, (const int *)m->idx.p + q * batch, nullptr, nullptr, nv}, nullptr,
        lossp + q * nbl);
    m->step++;
    const AdamStep st{lr, 1.0f - std::pow(0.9f, (float)m->step), 1.0f - std::pow(0.999f, (float)m->step)};
    weights<true>(m, st, nullptr, nullptr);
  }
  hipLaunchKernelGGL(k_losses, dim3((unsigned)nsteps), dim3(256), 0, m->s, lossp, nbl,
                     (float)(1.0 / ((double)batch * m->d.nout)), (float)(1.0 / ((double)nv * m->d.nout)),
                     (float *)m->losses.p);
  HIPCHK(hipGetLastError());
  std::vector<float> lb(nsteps);
  HIPCHK(hipMemcpyAsync(lb.data(), m->losses.p, nsteps * sizeof(float), hipMemcpyDeviceToHost, m->s));
  HIPCHK(hipStreamSynchronize(m->s));
  double lsum = 0;
  for (float v : lb) lsum += v;
  if (loss_out) *loss_out = (float)(lsum / nsteps);
  return 0;
}

int usg_mlp_mfma_check(const float *a, const float *b, float *d) {
  if (!a || !b || !d) return fail(-1, "null argument");
  // device buffers released on every return
  struct Bufs {
    void *p[3] = {nullptr, nullptr, nullptr};
    ~Bufs() {
      for (void *q : p)
        if (q) (void)hipFree(q);
    }
  } bufs;
  std::vector<bf16> ha(16 * 32), hb(32 * 16);
  for (int i = 0; i < 16 * 32; i++) {
    ha[i] = to_bf16(a[i]);
    hb[i] = to_bf16(b[i]);
  }
  HIPCHK(hipMalloc(&bufs.p[0], ha.size() * 2));
  HIPCHK(hipMalloc(&bufs.p[1], hb.size() * 2));
  HIPCHK(hipMalloc(&bufs.p[2], 256 * 4));
  bf16 *da = (bf16 *)bufs.p[0], *db = (bf16 *)bufs.p[1];
  float *dd = (float *)bufs.p[2];
  HIPCHK(hipMemcpy(da, ha.data(), ha.size() * 2, hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(db, hb.data(), hb.size() * 2, hipMemcpyHostToDevice));
  hipLaunchKernelGGL(k_mfma_check, dim3(1), dim3(64), 0, 0, da, db, dd);
  HIPCHK(hipGetLastError());
  HIPCHK(hipMemcpy(d, dd, 256 * 4, hipMemcpyDeviceToHost));
  return 0;
}

}  // extern "C"
