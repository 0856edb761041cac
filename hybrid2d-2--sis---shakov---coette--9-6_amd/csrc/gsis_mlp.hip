// gsis_mlp.hip -- hand-written gfx950 kernels of the learned HoT closure:
// forward, backward and Adam for an 8-128-128-128-128-5 SiLU network with BF16
// weights and activations and FP32 accumulation on the matrix cores.
//
// A batch is two kernels.  k_mlp_pass: a workgroup takes 64 samples through all
// layers and back, with activations and gradients in LDS (BF16) and
// pre-activations in registers (FP32), and leaves the operands of the weight
// gradients in memory.  k_mlp_grad: a wavefront per 32 x 32 block of a weight
// gradient and the bias sums, with the Adam step of those parameters.
// Every product is C = A B with both operands stored so that a lane's MFMA
// operand is contiguous along k:
//   forward   Z_l  = H_{l-1} W_l^T    A = H_{l-1} [sample][in],  B = W_l [out][in]
//   backward  dH_l = dZ_{l+1} W_{l+1} A = dZ_{l+1} [sample][out], B = W^T [in][out]
//             dW_l = dZ_l^T H_{l-1}   A = dZ_l^T [out][sample],  B = H^T [in][sample]
// One wavefront computes 32 x 32 blocks of C with v_mfma_f32_32x32x8_bf16 (A:
// lane l holds row l%32, k = 4(l/32)..+3; B likewise for column l%32; C: lane l
// holds column l%32 and rows 8(r/4) + 4(l/32) + r%4 of its 16 accumulators r).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "gsis_mlp.h"

namespace gsis {

void set_last_error(const std::string &msg);

namespace {
int mfail(int code, const std::string &msg) {
  set_last_error(msg);
  return code;
}
}  // namespace

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

int mlp_woff(int l) {
  int o = 0;
  for (int k = 0; k < l; k++) o += mlp_rows(k) * mlp_cols(k) + mlp_rows(k);
  return o;
}
int mlp_boff(int l) { return mlp_woff(l) + mlp_rows(l) * mlp_cols(l); }
int mlp_nparams() { return mlp_woff(kMlpLayers); }

// FP32 -> BF16, round to nearest even
__host__ __device__ inline unsigned short to_bf16(float f) {
  unsigned u;
  memcpy(&u, &f, 4);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}

__device__ inline float silu(float z) { return z / (1.0f + __expf(-z)); }
__device__ inline float silu_grad(float z) {
  const float s = 1.0f / (1.0f + __expf(-z));
  return s * (1.0f + z * (1.0f - s));
}

// What a pass reads of a network
struct MlpNet {
  const float *p, *scale;
  const unsigned short *w[kMlpLayers], *wt[kMlpLayers];
};
// offsets of W_l and b_l in the parameter vector
struct MlpOff {
  int w[kMlpLayers], b[kMlpLayers];
  __host__ __device__ constexpr MlpOff() : w(), b() {
    int o = 0;
    for (int l = 0; l < kMlpLayers; l++) {
      w[l] = o;
      b[l] = o + mlp_rows(l) * mlp_cols(l);
      o = b[l] + mlp_rows(l);
    }
  }
};
constexpr MlpOff kOffs{};

// LDS rows: 8-byte aligned, and 32 lanes reading 8 bytes of 32 rows hit each bank once
constexpr int kLdF = kMlpW + 4;     // [sample][feature]
constexpr int kLdX = kMlpInPad + 4;  // [sample][input]
constexpr int kMlpThreads = 512;    // 8 wavefronts: one 32 x 32 block of a 64 x 128 layer each
constexpr int kHid = kMlpLayers - 1;

// What a batch leaves for the weight gradients.  in_t[l] (the inputs of layer l)
// and dz_t[l] in operand order: feature f of sample s at
// (s/16 F + f) 16 + 8 h + 4 j + e with s%16 = 8 j + 4 h + e, so the lanes of a
// wavefront (feature f, half h) read the operands of two products with one
// 16-byte load each, 1 KiB in a row.
struct MlpTape {
  unsigned short *in_t[kMlpLayers], *dz_t[kMlpLayers];
  float *dz[kHid], *dy;
  double *lpart;
};
typedef short bf16x8 __attribute__((ext_vector_type(8)));

struct MlpShared {
  unsigned short f[kMlpRows * kLdF];  // H of the last layer, or dZ
  unsigned short x[kMlpRows * kLdX];  // inputs
  double red[2];
};

// A barrier for what is in LDS: loads and stores of global memory stay under way
// (__syncthreads would wait for them, about 1 us at each of 11 barriers).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// this lane's operands of the K/8 products over B's row
template <int K>
struct Operands {
  bf16x4 v[K / 8];
  __device__ explicit Operands(const unsigned short *b) {
#pragma unroll
    for (int k = 0; k < K / 8; k++) v[k] = *reinterpret_cast<const bf16x4 *>(b + 8 * k);
  }
};
// C (32 x 32) = sum over k < K of A's row and B's row of this lane
template <int K>
__device__ __forceinline__ f32x16 mm(const unsigned short *a, const Operands<K> &b) {
  f32x16 acc = {0};
#pragma unroll
  for (int k = 0; k < K / 8; k++)
    acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(*reinterpret_cast<const bf16x4 *>(a + 8 * k), b.v[k], acc, 0, 0, 0);
  return acc;
}

// Samples 64 blockIdx.x .. +63 of n (through idx if given) forward, and with
// TRAIN back, for the gradient of the mean squared error of the n x 5
// standardised outputs.  Samples past n have zero inputs and no error.
//
// What bounds it: 64 workgroups (a batch of 4096) leave the chip mostly idle;
// a workgroup is a chain of 9 products, each 4 to 16 dependent matrix
// instructions and an exchange through LDS.  The weights of a product are
// loaded one product ahead.  Before, each product and each element-wise step
// was a launch of its own over matrices in memory.
template <bool TRAIN>
__global__ void __launch_bounds__(kMlpThreads) k_mlp_pass(MlpNet net, const float *x, const int *idx, int n, float *y,
                                                          const float *target, MlpTape tape) {
  __shared__ __align__(16) MlpShared sh;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 31, h = lane >> 5, kq = 4 * h;
  const int nb = wave & 3, rb = wave >> 2;  // this wavefront's feature block and sample block
  const int row0 = blockIdx.x * kMlpRows, n0 = 32 * nb, m0 = 32 * rb, col = n0 + r;
  auto qrow = [&](int q) { return (q >> 2) * 8 + 4 * h + (q & 3); };  // row of accumulator q within a block
  const Operands<kMlpInPad> b0(net.w[0] + col * kMlpInPad + kq);
  // the standardised inputs, zero past the 8 columns and past n
  for (int e = tid; e < kMlpRows * kMlpInPad; e += kMlpThreads) {
    const int row = e / kMlpInPad, f = e % kMlpInPad;
    float v = 0.0f;
    if (row0 + row < n && f < kMlpIn) {
      const size_t s = idx ? idx[row0 + row] : row0 + row;
      v = (x[s * kMlpIn + f] - net.scale[f]) / net.scale[kMlpIn + f];
    }
    const unsigned short b = to_bf16(v);
    sh.x[row * kLdX + f] = b;
    if constexpr (TRAIN) {
      const int s = row & 15;
      tape.in_t[0][((size_t)((row0 + row) / 16) * kMlpInPad + f) * 16 + 8 * ((s >> 2) & 1) + 4 * (s >> 3) + (s & 3)] = b;
    }
  }
  // this lane's 16 samples of a column: [sample][feature] to LDS, operand order to memory (F features)
  auto put = [&](const float *v, unsigned short *t, int F) {
#pragma unroll
    for (int q = 0; q < 16; q += 8) {
      bf16x8 b;
      for (int e = 0; e < 8; e++) {
        const unsigned short u = to_bf16(v[q + e]);
        b[e] = (short)u;
        sh.f[(m0 + qrow(q + e)) * kLdF + col] = u;
      }
      if constexpr (TRAIN)
        if (col < F)
          *reinterpret_cast<bf16x8 *>(t + ((size_t)((row0 + m0) / 16 + q / 8) * F + col) * 16 + 8 * h) = b;
    }
  };
  float z[TRAIN ? kHid : 1][16];
  constexpr int L = kMlpLayers - 1;
  float bias[kHid];
#pragma unroll
  for (int l = 0; l < kHid; l++) bias[l] = net.p[kOffs.b[l] + col];
  const float ob = r < kMlpOut ? net.p[kOffs.b[L] + r] : 0.0f;
  const float om = r < kMlpOut ? net.scale[2 * kMlpIn + r] : 0.0f;
  const float os = r < kMlpOut ? net.scale[2 * kMlpIn + kMlpOut + r] : 1.0f;
  Operands<kMlpW> b(net.w[1] + col * kMlpW + kq);
  lds_barrier();
#pragma unroll
  for (int l = 0; l < kHid; l++) {
    const f32x16 c = l == 0 ? mm(sh.x + (m0 + r) * kLdX + kq, b0) : mm(sh.f + (m0 + r) * kLdF + kq, b);
    if (l > 0) b = Operands<kMlpW>(net.w[l + 1] + (l + 1 < L ? col : r) * kMlpW + kq);
    float v[16];
    for (int q = 0; q < 16; q++) {
      v[q] = c[q] + bias[l];
      if constexpr (TRAIN) z[l][q] = v[q];
      v[q] = silu(v[q]);
    }
    lds_barrier();  // the layer before is read
    put(v, TRAIN ? tape.in_t[l + 1] : nullptr, kMlpW);
    lds_barrier();
  }
  // the output layer: wavefronts 0 and 4 have the two blocks of samples
  f32x16 c = {0};
  if (nb == 0) c = mm(sh.f + (m0 + r) * kLdF + kq, b);
  if constexpr (!TRAIN) {
    if (nb == 0 && r < kMlpOut)
      for (int q = 0; q < 16; q++) {
        const int row = row0 + m0 + qrow(q);
        if (row < n) y[(size_t)row * kMlpOut + r] = (c[q] + ob) * os + om;
      }
    return;
  } else {
    const Operands<kMlpOutPad> b5(net.wt[L] + col * kMlpOutPad + kq);
    b = Operands<kMlpW>(net.wt[kHid - 1] + col * kMlpW + kq);
    // dY = 2 (Y - T) / (5 n), zero outside the n x 5 values
    double acc = 0.0;
    float dy[16];
    for (int q = 0; q < 16; q++) {
      dy[q] = 0.0f;
      const int row = row0 + m0 + qrow(q);
      if (nb == 0 && row < n && r < kMlpOut) {
        const size_t s = idx ? idx[row] : row;
        const float e = c[q] + ob - (target[s * kMlpOut + r] - om) / os;
        acc += (double)e * e;
        dy[q] = 2.0f * e / (float)(kMlpOut * n);
      }
    }
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    lds_barrier();  // H of the last hidden layer is read
    if (nb == 0) {
      put(dy, tape.dz_t[L], kMlpOutPad);
      if (lane == 0) sh.red[rb] = acc;
      if (r < 8)
        for (int q = 0; q < 16; q++) tape.dy[(size_t)(row0 + m0 + qrow(q)) * 8 + r] = dy[q];
    }
    lds_barrier();
    if (tid == 0) tape.lpart[blockIdx.x] = sh.red[0] + sh.red[1];
    f32x16 dh = mm(sh.f + (m0 + r) * kLdF + kq, b5);
#pragma unroll
    for (int l = kHid - 1; l >= 0; l--) {
      float g[16];  // dZ = dH SiLU'(Z), zero past n
      for (int q = 0; q < 16; q++) {
        const int row = row0 + m0 + qrow(q);
        g[q] = row < n ? dh[q] * silu_grad(z[l][q]) : 0.0f;
        tape.dz[l][(size_t)row * kMlpW + col] = g[q];
      }
      lds_barrier();  // dZ of the layer above is read
      put(g, tape.dz_t[l], kMlpW);
      lds_barrier();
      if (l > 0) {
        dh = mm(sh.f + (m0 + r) * kLdF + kq, b);
        if (l > 1) b = Operands<kMlpW>(net.wt[l - 1] + col * kMlpW + kq);
      }
    }
  }
}

// BF16 copies of W_l: W [rows_pad x cols_pad] and W^T [cols_pad x rows_pad],
// the padding zero
__global__ void k_mlp_pack(const float *w, int rows, int rows_pad, int cols, int cols_pad, unsigned short *wb,
                           unsigned short *wtb) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= rows_pad * cols_pad) return;
  const int r = t / cols_pad, c = t % cols_pad;
  const unsigned short b = r < rows && c < cols ? to_bf16(w[(size_t)r * cols + c]) : (unsigned short)0;
  wb[t] = b;
  wtb[(size_t)c * rows_pad + r] = b;
}

// One parameter's gradient gt: stored, and with ADAM the step (c1, c2: bias
// corrections).
struct MlpAdam {
  float *p, *g, *m1, *m2;
  unsigned short *w[kMlpLayers], *wt[kMlpLayers];
  float lr, b1, b2, eps, c1, c2;
};
template <bool ADAM>
__device__ __forceinline__ float mlp_param(const MlpAdam &o, int t, float gt) {
  o.g[t] = gt;
  if constexpr (!ADAM) return 0.0f;
  const float a = fmaf(1.0f - o.b1, gt, o.b1 * o.m1[t]);
  const float b = fmaf(gt, (1.0f - o.b2) * gt, o.b2 * o.m2[t]);
  o.m1[t] = a;
  o.m2[t] = b;
  return o.p[t] -= o.lr * (a / o.c1) / (sqrtf(b / o.c2) + o.eps);
}

// The gradients of a batch of n samples, padded to Mp (a multiple of 64), and
// with ADAM the step of each parameter and the BF16 copies of the new weights.
// One wavefront per workgroup:
//  * kGradBlocks workgroups: a 32 x 32 block of a weight gradient, one chain of
//    Mp/8 matrix instructions in the order of the samples, operands kAhead
//    loads ahead.  The chain is what it costs (29 us for 4096 samples); a
//    split of the samples over wavefronts, with the parts added afterwards,
//    rounds in another order, and Adam carries such
//    differences into the parameters (2e-4 after 128 steps);
//  * kBiasBlocks: the column sums of dZ for four hidden units, in the order of
//    256 interleaved partial sums;
//  * the last: the output bias (8 interleaved partial sums) and the loss.
constexpr int kGradBlocks = 4 + 3 * 16 + 4;  // output layer, hidden layers, first layer
constexpr int kBiasBlocks = kHid * kMlpW / 4;
constexpr int kAhead = 24;
template <bool ADAM>
__global__ void __launch_bounds__(64) k_mlp_grad(MlpTape tape, int n, int Mp, double *loss, MlpAdam o) {
  const int lane = threadIdx.x;
  int blk = blockIdx.x;
  if (blk < kGradBlocks) {
    int l, ob, ib;  // layer, block of outputs, block of inputs
    if (blk < 4) { l = kMlpLayers - 1; ob = 0; ib = blk; }
    else if (blk < 52) { l = 1 + (blk - 4) / 16; ob = (blk - 4) % 16 / 4; ib = (blk - 4) % 4; }
    else { l = 0; ob = blk - 52; ib = 0; }
    const int r = lane & 31, h = lane >> 5;
    const int Fa = mlp_rows_pad(l), Fb = mlp_cols_pad(l), groups = Mp / 16;
    const unsigned short *dz = tape.dz_t[0], *in = tape.in_t[0];
#pragma unroll
    for (int k = 1; k < kMlpLayers; k++)
      if (l == k) { dz = tape.dz_t[k]; in = tape.in_t[k]; }
    const bf16x8 *a = reinterpret_cast<const bf16x8 *>(dz) + (ob * 32 + r) * 2 + h;
    const bf16x8 *b = reinterpret_cast<const bf16x8 *>(in) + (ib * 32 + r) * 2 + h;
    const int sa = Fa * 2, sb = Fb * 2;  // per group of 16 samples
    bf16x8 av[kAhead], bv[kAhead];
#pragma unroll
    for (int k = 0; k < kAhead; k++) {
      const int q = min(k, groups - 1);
      av[k] = a[(size_t)q * sa];
      bv[k] = b[(size_t)q * sb];
    }
    f32x16 acc = {0};
    for (int q0 = 0; q0 < groups; q0 += kAhead) {
#pragma unroll
      for (int k = 0; k < kAhead; k++) {
        if (q0 + k < groups) {
          const bf16x8 x = av[k], y = bv[k];
          acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(bf16x4{x[0], x[1], x[2], x[3]}, bf16x4{y[0], y[1], y[2], y[3]},
                                                         acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(bf16x4{x[4], x[5], x[6], x[7]}, bf16x4{y[4], y[5], y[6], y[7]},
                                                         acc, 0, 0, 0);
        }
        const int q = min(q0 + k + kAhead, groups - 1);
        av[k] = a[(size_t)q * sa];
        bv[k] = b[(size_t)q * sb];
      }
    }
    const int col = ib * 32 + r, cols = mlp_cols(l), rows = mlp_rows(l);
    if (col >= cols) return;
    int off = kOffs.w[0];
    unsigned short *w = o.w[0], *wt = o.wt[0];
#pragma unroll
    for (int k = 1; k < kMlpLayers; k++)
      if (l == k) { off = kOffs.w[k]; w = o.w[k]; wt = o.wt[k]; }
#pragma unroll
    for (int q = 0; q < 16; q++) {
      const int row = ob * 32 + (q >> 2) * 8 + 4 * h + (q & 3);
      if (row >= rows) continue;
      const float v = mlp_param<ADAM>(o, off + row * cols + col, acc[q]);
      if constexpr (ADAM) {
        const unsigned short u = to_bf16(v);
        w[row * Fb + col] = u;
        wt[col * Fa + row] = u;
      }
    }
    return;
  }
  blk -= kGradBlocks;
  if (blk < kBiasBlocks) {
    const int l = blk / (kMlpW / 4), c0 = blk % (kMlpW / 4) * 4;
    const float *dz = tape.dz[0];
    int off = kOffs.b[0];
#pragma unroll
    for (int k = 1; k < kHid; k++)
      if (l == k) { dz = tape.dz[k]; off = kOffs.b[k]; }
    float s[4][4] = {};  // partial sum lane + 64 m of column c0 + e
    for (int r0 = 0; r0 < Mp; r0 += 256)
#pragma unroll
      for (int m = 0; m < 4; m++) {
        const int row = r0 + 64 * m + lane;
        if (row >= Mp) continue;
        const float4 v = *reinterpret_cast<const float4 *>(dz + (size_t)row * kMlpW + c0);
        s[m][0] += v.x; s[m][1] += v.y; s[m][2] += v.z; s[m][3] += v.w;
      }
    for (int e = 0; e < 4; e++) {
      float v = (s[0][e] + s[2][e]) + (s[1][e] + s[3][e]);
      for (int k = 32; k > 0; k >>= 1) v += __shfl_down(v, k, 64);
      if (lane == 0) (void)mlp_param<ADAM>(o, off + c0 + e, v);
    }
    return;
  }
  // partial sum j of output c: samples j, j + 8, ...
  const int j = lane >> 3, c = lane & 7;
  float s = 0.0f;
#pragma unroll 16
  for (int row = j; row < Mp; row += 8) s += tape.dy[(size_t)row * 8 + c];
  for (int k = 32; k > 0; k >>= 1)
    if (k >= 8) s += __shfl_down(s, k, 64);
  if (lane < kMlpOut) (void)mlp_param<ADAM>(o, kOffs.b[kMlpLayers - 1] + lane, s);
  if (lane == 63) {
    double e = 0.0;
    for (int k = 0; k < Mp / kMlpRows; k++) e += tape.lpart[k];
    e = e / (double)(kMlpOut * n);
    loss[0] = e;
    loss[1] += e;
  }
}

namespace {

unsigned nblk(size_t n, int b = 256) { return (unsigned)((n + b - 1) / b); }

template <typename P>
int malloc_d(MlpDev &d, P **p, size_t bytes) {
  void *q = nullptr;
  if (hipMalloc(&q, std::max(bytes, (size_t)8)) != hipSuccess) return mfail(GSIS_EHIP, "mlp: hipMalloc failed");
  // cleared on the network's own stream, before whatever uses it there
  if (hipMemsetAsync(q, 0, std::max(bytes, (size_t)8), d.s) != hipSuccess)
    return mfail(GSIS_EHIP, "mlp: hipMemset failed");
  d.allocs.push_back(q);
  *p = reinterpret_cast<P *>(q);
  return 0;
}

void pack(MlpDev &d) {
  for (int l = 0; l < kMlpLayers; l++) {
    const int rp = mlp_rows_pad(l), cp = mlp_cols_pad(l);
    hipLaunchKernelGGL(k_mlp_pack, dim3(nblk((size_t)rp * cp)), dim3(256), 0, d.s, d.p + mlp_woff(l), mlp_rows(l), rp,
                       mlp_cols(l), cp, d.w[l], d.wt[l]);
  }
}

MlpNet net_of(const MlpDev &d) {
  MlpNet m{d.p, d.dscale, {}, {}};
  for (int l = 0; l < kMlpLayers; l++) {
    m.w[l] = d.w[l];
    m.wt[l] = d.wt[l];
  }
  return m;
}

MlpTape tape_of(const MlpDev &d) {
  MlpTape t{{}, {}, {}, d.dy, d.lpart};
  for (int l = 0; l < kMlpLayers; l++) {
    t.in_t[l] = d.in_t[l];
    t.dz_t[l] = d.dz_t[l];
    if (l < kHid) t.dz[l] = d.dz[l];
  }
  return t;
}

// the gradient and loss of the n samples x, t (through idx if given) into d.g
// and d.loss, and with ADAM the step with the constants of o
template <bool ADAM>
void batch_step(MlpDev &d, const float *x, const float *t, const int *idx, int n, MlpAdam o) {
  const int wgs = (n + kMlpRows - 1) / kMlpRows;
  o.p = d.p;
  o.g = d.g;
  o.m1 = d.m1;
  o.m2 = d.m2;
  for (int l = 0; l < kMlpLayers; l++) {
    o.w[l] = d.w[l];
    o.wt[l] = d.wt[l];
  }
  const MlpTape tape = tape_of(d);
  hipLaunchKernelGGL(k_mlp_pass<true>, dim3(wgs), dim3(kMlpThreads), 0, d.s, net_of(d), x, idx, n, (float *)nullptr, t,
                     tape);
  hipLaunchKernelGGL(k_mlp_grad<ADAM>, dim3(kGradBlocks + kBiasBlocks + 1), dim3(64), 0, d.s, tape, n, wgs * kMlpRows,
                     d.loss, o);
}

int ensure_cap(MlpDev &d, size_t n) {
  if (n <= d.cap) return 0;
  for (void *q : {(void *)d.xin, (void *)d.yin, (void *)d.idx}) {
    if (q) {
      (void)hipFree(q);
      d.allocs.erase(std::remove(d.allocs.begin(), d.allocs.end(), q), d.allocs.end());
    }
  }
  int rc;
  if ((rc = malloc_d(d, &d.xin, n * kMlpIn * 4)) || (rc = malloc_d(d, &d.yin, n * kMlpOut * 4)) ||
      (rc = malloc_d(d, &d.idx, n * 4)))
    return rc;
  d.cap = n;
  return 0;
}

int sync(MlpDev &d) {
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(d.s);
  if (e != hipSuccess) return mfail(GSIS_EHIP, std::string("mlp: ") + hipGetErrorString(e));
  return 0;
}

}  // namespace

// Standardised forward pass of n device-resident raw inputs (x: n x 8) into
// y (n x 5, raw units), on the network's stream.  Used by the closure in the
// synthetic solve.
int mlp_forward_dev(MlpDev &d, const float *x, int n, float *y, hipStream_t s) {
  if (n > 0)
    hipLaunchKernelGGL(k_mlp_pass<false>, dim3((n + kMlpRows - 1) / kMlpRows), dim3(kMlpThreads), 0, s, net_of(d), x,
                       (const int *)nullptr, n, y, (const float *)nullptr, MlpTape{});
  return 0;
}

}  // namespace gsis

using namespace gsis;

extern "C" {

int gsis_mlp_nparams(void) { return mlp_nparams(); }

int gsis_mlp_destroy(gsis_mlp *m) {
  if (!m) return 0;
  if (m->d.s) (void)hipStreamSynchronize(m->d.s);
  for (void *q : m->d.allocs) (void)hipFree(q);
  if (m->d.s) (void)hipStreamDestroy(m->d.s);
  delete m;
  return 0;
}

int gsis_mlp_create(gsis_mlp **out) {
  if (!out) return mfail(GSIS_EARG, "out is NULL");
  *out = nullptr;
  gsis_mlp *m = new gsis_mlp();
  MlpDev &d = m->d;
  auto bail = [&](int rc) {
    gsis_mlp_destroy(m);
    return rc;
  };
  if (hipStreamCreateWithFlags(&d.s, hipStreamNonBlocking) != hipSuccess)
    return bail(mfail(GSIS_EHIP, "mlp: hipStreamCreate failed"));
  const size_t np = mlp_nparams();
  int rc;
  if ((rc = malloc_d(d, &d.p, np * 4)) || (rc = malloc_d(d, &d.g, np * 4)) || (rc = malloc_d(d, &d.m1, np * 4)) ||
      (rc = malloc_d(d, &d.m2, np * 4)) || (rc = malloc_d(d, &d.dscale, sizeof(d.scale))))
    return bail(rc);
  for (int l = 0; l < kMlpLayers; l++) {
    const size_t e = (size_t)mlp_rows_pad(l) * mlp_cols_pad(l);
    if ((rc = malloc_d(d, &d.w[l], e * 2)) || (rc = malloc_d(d, &d.wt[l], e * 2))) return bail(rc);
  }
  const size_t B = kMlpBatchMax;
  if ((rc = malloc_d(d, &d.dy, B * 8 * 4)) || (rc = malloc_d(d, &d.lpart, B / kMlpRows * 8)) ||
      (rc = malloc_d(d, &d.loss, 16)))
    return bail(rc);
  for (int l = 0; l < kMlpLayers; l++) {
    if ((rc = malloc_d(d, &d.in_t[l], B * mlp_cols_pad(l) * 2)) || (rc = malloc_d(d, &d.dz_t[l], B * mlp_rows_pad(l) * 2)))
      return bail(rc);
    if (l < kMlpLayers - 1 && (rc = malloc_d(d, &d.dz[l], B * kMlpW * 4))) return bail(rc);
  }
  for (int k = 0; k < kMlpIn; k++) d.scale[kMlpIn + k] = 1.0f;
  for (int k = 0; k < kMlpOut; k++) d.scale[2 * kMlpIn + kMlpOut + k] = 1.0f;
  // on the network's stream, behind the clear of the same memory
  if (hipMemcpyAsync(d.dscale, d.scale, sizeof(d.scale), hipMemcpyHostToDevice, d.s) != hipSuccess)
    return bail(mfail(GSIS_EHIP, "mlp: scaling upload failed"));
  pack(d);
  if ((rc = sync(d))) return bail(rc);
  *out = m;
  return 0;
}

int gsis_mlp_set_params(gsis_mlp *m, const float *params) {
  if (!m || !params) return mfail(GSIS_EARG, "NULL argument");
  MlpDev &d = m->d;
  if (hipMemcpyAsync(d.p, params, (size_t)mlp_nparams() * 4, hipMemcpyHostToDevice, d.s) != hipSuccess)
    return mfail(GSIS_EHIP, "mlp: parameter upload failed");
  (void)hipMemsetAsync(d.m1, 0, (size_t)mlp_nparams() * 4, d.s);
  (void)hipMemsetAsync(d.m2, 0, (size_t)mlp_nparams() * 4, d.s);
  d.step = 0;
  pack(d);
  return sync(d);
}

int gsis_mlp_get_params(gsis_mlp *m, float *params) {
  if (!m || !params) return mfail(GSIS_EARG, "NULL argument");
  MlpDev &d = m->d;
  if (hipMemcpyAsync(params, d.p, (size_t)mlp_nparams() * 4, hipMemcpyDeviceToHost, d.s) != hipSuccess)
    return mfail(GSIS_EHIP, "mlp: parameter download failed");
  return sync(d);
}

int gsis_mlp_set_scaling(gsis_mlp *m, const float *scaling) {
  if (!m || !scaling) return mfail(GSIS_EARG, "NULL argument");
  MlpDev &d = m->d;
  for (int k = 0; k < 2 * kMlpIn + 2 * kMlpOut; k++) {
    const bool is_std = (k >= kMlpIn && k < 2 * kMlpIn) || k >= 2 * kMlpIn + kMlpOut;
    if (is_std && !(scaling[k] > 0.0f)) return mfail(GSIS_EARG, "mlp: standard deviations must be positive");
    d.scale[k] = scaling[k];
  }
  if (hipMemcpyAsync(d.dscale, d.scale, sizeof(d.scale), hipMemcpyHostToDevice, d.s) != hipSuccess)
    return mfail(GSIS_EHIP, "mlp: scaling upload failed");
  return sync(d);
}

int gsis_mlp_forward(gsis_mlp *m, const float *x, int32_t n, float *y) {
  if (!m || !x || !y || n < 0) return mfail(GSIS_EARG, "bad argument");
  if (n == 0) return 0;
  MlpDev &d = m->d;
  int rc = ensure_cap(d, (size_t)n);
  if (rc) return rc;
  if (hipMemcpyAsync(d.xin, x, (size_t)n * kMlpIn * 4, hipMemcpyHostToDevice, d.s) != hipSuccess)
    return mfail(GSIS_EHIP, "mlp: input upload failed");
  mlp_forward_dev(d, d.xin, n, d.yin, d.s);
  if (hipMemcpyAsync(y, d.yin, (size_t)n * kMlpOut * 4, hipMemcpyDeviceToHost, d.s) != hipSuccess)
    return mfail(GSIS_EHIP, "mlp: output download failed");
  return sync(d);
}

int gsis_mlp_loss_grad(gsis_mlp *m, const float *x, const float *y, int32_t n, double *loss, float *grad) {
  if (!m || !x || !y || n < 1 || n > kMlpBatchMax) return mfail(GSIS_EARG, "bad argument (1 <= n <= 8192)");
  MlpDev &d = m->d;
  int rc = ensure_cap(d, (size_t)n);
  if (rc) return rc;
  if (hipMemcpyAsync(d.xin, x, (size_t)n * kMlpIn * 4, hipMemcpyHostToDevice, d.s) != hipSuccess ||
      hipMemcpyAsync(d.yin, y, (size_t)n * kMlpOut * 4, hipMemcpyHostToDevice, d.s) != hipSuccess)
    return mfail(GSIS_EHIP, "mlp: sample upload failed");
  batch_step<false>(d, d.xin, d.yin, nullptr, n, MlpAdam{});
  if (loss && hipMemcpyAsync(loss, d.loss, 8, hipMemcpyDeviceToHost, d.s) != hipSuccess)
    return mfail(GSIS_EHIP, "mlp: loss download failed");
  if (grad && hipMemcpyAsync(grad, d.g, (size_t)mlp_nparams() * 4, hipMemcpyDeviceToHost, d.s) != hipSuccess)
    return mfail(GSIS_EHIP, "mlp: gradient download failed");
  return sync(d);
}

int gsis_mlp_train(gsis_mlp *m, const float *x, const float *y, int32_t n, int32_t epochs, int32_t batch, float lr,
                   uint64_t seed, double *loss_per_epoch) {
  if (!m || !x || !y || n < 1 || epochs < 0 || batch < 64 || batch > kMlpBatchMax || batch % 64)
    return mfail(GSIS_EARG, "bad argument (batch a multiple of 64 in 64..8192)");
  MlpDev &d = m->d;
  int rc = ensure_cap(d, (size_t)n);
  if (rc) return rc;
  if (hipMemcpyAsync(d.xin, x, (size_t)n * kMlpIn * 4, hipMemcpyHostToDevice, d.s) != hipSuccess ||
      hipMemcpyAsync(d.yin, y, (size_t)n * kMlpOut * 4, hipMemcpyHostToDevice, d.s) != hipSuccess)
    return mfail(GSIS_EHIP, "mlp: sample upload failed");
  std::vector<int> perm(n);
  for (int k = 0; k < n; k++) perm[k] = k;
  std::mt19937_64 rng(seed);
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  std::vector<double> lossb;
  for (int ep = 0; ep < epochs; ep++) {
    std::shuffle(perm.begin(), perm.end(), rng);
    if (hipMemcpyAsync(d.idx, perm.data(), (size_t)n * 4, hipMemcpyHostToDevice, d.s) != hipSuccess ||
        hipMemsetAsync(d.loss, 0, 16, d.s) != hipSuccess)
      return mfail(GSIS_EHIP, "mlp: index upload failed");
    const int nb = n / batch;  // full batches only
    for (int b = 0; b < std::max(nb, 1); b++) {
      const int cnt = nb > 0 ? batch : n;
      d.step += 1;
      const float c1 = 1.0f - std::pow(b1, (float)d.step), c2 = 1.0f - std::pow(b2, (float)d.step);
      MlpAdam o{};
      o.lr = lr; o.b1 = b1; o.b2 = b2; o.eps = eps; o.c1 = c1; o.c2 = c2;
      batch_step<true>(d, d.xin, d.yin, d.idx + (size_t)b * batch, cnt, o);
    }
    double l[2] = {0.0, 0.0};
    if (hipMemcpyAsync(l, d.loss, 16, hipMemcpyDeviceToHost, d.s) != hipSuccess ||
        hipStreamSynchronize(d.s) != hipSuccess)
      return mfail(GSIS_EHIP, "mlp: loss download failed");
    lossb.push_back(l[1] / std::max(nb, 1));
  }
  if ((rc = sync(d))) return rc;
  if (loss_per_epoch) std::copy(lossb.begin(), lossb.end(), loss_per_epoch);
  return 0;
}

}  // extern "C"
