// closure_kernels.h -- device code of the learned subgrid closure, included by
// tslb.hip inside its anonymous namespace.
//
// A per-node MLP maps 10 local inputs (strain rate S from the isotropic
// gradient of the velocity, grad(phi), phi) to an eddy viscosity nu_t and six
// interfacial-stress corrections dsigma; the collision then relaxes with
// omega = 1/(tau + 3 nu_t) and adds dsigma to the post-collision stress.  The
// reference has no such closure; the network shape and the input/output sets
// follow the target description of the path (10 -> 64 -> 64 -> 64 -> 7, GELU).
//
// Matrix cores.  Every layer is one chain of v_mfma_f32_16x16x32_bf16 in the
// transposed form Z^T = W^T X^T: the A operand is the weight block (16 output
// features x 32 inputs), the B operand 32 inputs x 16 nodes, the accumulator
// 16 features x 16 nodes.  Lane l = 16 g + c holds, per MFMA,
//   A[c][8g + i], B[8g + i][c] (i < 8)  and  D[4g + i][c] (i < 4).
// The D registers of a layer become the B operand of the next one without a
// shuffle: the 32-wide K step ks of the next layer takes output blocks 2ks and
// 2ks+1, so its k = 8g + i stands for feature
//   perm(ks, g, i) = 16 (2 ks + i/4) + 4 g + i%4,
// and the weights are packed on the device in that order (k_mlp_pack).  The
// bias of layer 1 rides on a constant-1 input (k = 10); the other biases
// initialise the accumulators.
//
// Training.  k_mlp_grad runs forward, backward (the backward products
// delta_{l-1} = W_l delta_l use a second, transposed pack) and the weight
// gradients (dW = delta H^T, K = samples) of 64 samples in one block, all
// operands in LDS; k_mlp_update sums the blocks' FP32 gradients, updates the
// FP32 master weights by Adam and repacks them.  Batches of up to kColsMax
// samples keep their activations and deltas instead, and k_mlp_wgrad forms dW
// from them in slices of 512 samples.  The loss is summed in FP64.
#pragma once

constexpr int kMlpNF = 10, kMlpNH = 64, kMlpNO = 7;
// offsets in the natural parameter vector (in x out row-major per layer)
constexpr int kOffW1 = 0, kOffB1 = 640, kOffW2 = 704, kOffB2 = 4800, kOffW3 = 4864, kOffB3 = 8960,
              kOffW4 = 9024, kOffB4 = 9472, kOffIn = 9479, kOffOut = 9489, kMlpNParam = 9496;
constexpr int kFwdBlocks = 22, kBwdBlocks = 20;
constexpr float kGeluC = 0.7978845608028654f, kGeluA = 0.044715f;
// per-sample auxiliary record: rho_bar, tau_xx, tau_yy, tau_zz, tau_xy, tau_xz, tau_yz
constexpr int kAux = 7;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__host__ __device__ constexpr int mlp_perm(int ks, int g, int i) {
  return 16 * (2 * ks + (i >> 2)) + 4 * g + (i & 3);
}
// z sigmoid(2u) = z / (1 + 2^(-2 u log2 e)), u = c (z + a z^3): one v_exp_f32
// and one v_rcp_f32
__device__ __forceinline__ float gelu_f(float z) {
  constexpr float c0 = -2.f * kGeluC * 1.4426950408889634f, c1 = c0 * kGeluA;
  const float e = __builtin_amdgcn_exp2f(z * fmaf(c1, z * z, c0));
  return z * __builtin_amdgcn_rcpf(1.f + e);
}
__device__ __forceinline__ float gelu_grad_f(float z) {
  const float u = kGeluC * fmaf(kGeluA * z * z, z, z);
  const float s = 1.f / (1.f + __expf(-2.f * u));
  return fmaf(z * s * (1.f - s) * 2.f * kGeluC, fmaf(3.f * kGeluA, z * z, 1.f), s);
}
__device__ __forceinline__ float softplus_f(float x) {
  return x > 20.f ? x : log1pf(__expf(x));
}

// natural parameters -> packed BF16 operand blocks (forward: 22 blocks, then
// backward: 20 blocks), 64 lanes x 8 values each
__global__ __launch_bounds__(256) void k_mlp_pack(const float *__restrict__ th, bf16x8 *__restrict__ fwd,
                                                  bf16x8 *__restrict__ bwd) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= (kFwdBlocks + kBwdBlocks) * 64) return;
  const int b = t / 64, l = t % 64, g = l >> 4, c = l & 15;
  bf16x8 v;
  for (int i = 0; i < 8; i++) {
    float x = 0.f;
    if (b < kFwdBlocks) {
      if (b < 4) {  // layer 1: A[16 mb + c][k], k = 8 g + i; k = 10 is the bias
        const int m = 16 * b + c, k = 8 * g + i;
        x = k < kMlpNF ? th[kOffW1 + k * kMlpNH + m] : (k == kMlpNF ? th[kOffB1 + m] : 0.f);
      } else if (b < 20) {  // layers 2, 3: A[16 mb + c][perm(ks, g, i)]
        const int r = (b - 4) & 7, mb = r >> 1, ks = r & 1;
        const int off = b < 12 ? kOffW2 : kOffW3;
        x = th[off + mlp_perm(ks, g, i) * kMlpNH + 16 * mb + c];
      } else {  // layer 4: 7 outputs of 16 rows
        const int ks = b - 20;
        x = c < kMlpNO ? th[kOffW4 + mlp_perm(ks, g, i) * kMlpNO + c] : 0.f;
      }
    } else {
      const int bb = b - kFwdBlocks;
      if (bb < 4) {  // W4 (64 x 7): A[m = input 16 mb + c][k = output 8 g + i]
        const int m = 16 * bb + c, k = 8 * g + i;
        x = k < kMlpNO ? th[kOffW4 + m * kMlpNO + k] : 0.f;
      } else {  // W3 then W2: A[m = input 16 mb + c][k = output perm(ks, g, i)]
        const int r = (bb - 4) & 7, mb = r >> 1, ks = r & 1;
        const int off = bb < 12 ? kOffW3 : kOffW2;
        x = th[off + (16 * mb + c) * kMlpNH + mlp_perm(ks, g, i)];
      }
    }
    v[i] = (__bf16)x;
  }
  if (b < kFwdBlocks) fwd[b * 64 + l] = v;
  else bwd[(b - kFwdBlocks) * 64 + l] = v;
}

// B operand of layer 1 (lane group g: scaled inputs 8g..8g+7, the constant 1 at
// k = 10), from FP32 inputs (SoA, read ahead of their use) ...
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
struct MlpPlain {
  struct Raw {
    float v[8];
  };
  const float *f;
  long long fstride;
  float sc[8];
  int g;
  __device__ __forceinline__ MlpPlain(const float *feat, long long fs, long long, const float *th, int g_)
      : f(feat + 8LL * g_ * fs), fstride(fs), g(g_) {
#pragma unroll
    for (int i = 0; i < 8; i++) sc[i] = 8 * g + i < kMlpNF ? th[kOffIn + 8 * g + i] : 0.f;
  }
  __device__ __forceinline__ void load(Raw &r, long long node) const {
#pragma unroll
    for (int i = 0; i < 8; i++) r.v[i] = 8 * g + i < kMlpNF ? f[i * fstride + node] : 0.f;
  }
  __device__ __forceinline__ bf16x8 operand(const Raw &r) const {
    bf16x8 B;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int k = 8 * g + i;
      B[i] = (__bf16)(k < kMlpNF ? r.v[i] * sc[i] : (k == kMlpNF ? 1.f : 0.f));
    }
    return B;
  }
};
// ... or from the operand as k_features writes it: eight values a node, then two
struct MlpPacked {
  typedef bf16x8 Raw;
  const bf16x8 *lo;
  const bf16x2 *hi;
  int g;
  __device__ __forceinline__ MlpPacked(const float *feat, long long, long long n, const float *, int g_)
      : lo((const bf16x8 *)feat), hi((const bf16x2 *)(feat + 4 * n)), g(g_) {}
  __device__ __forceinline__ void load(Raw &r, long long node) const {
#pragma unroll
    for (int i = 0; i < 8; i++) r[i] = (__bf16)0.f;
    if (g == 0) {
      r = lo[node];
    } else if (g == 1) {
      const bf16x2 v = hi[node];
      r[0] = v[0];
      r[1] = v[1];
      r[2] = (__bf16)1.f;
    }
  }
  __device__ __forceinline__ bf16x8 operand(const Raw &r) const { return r; }
};

// GELU of four accumulator blocks, packed as the two K steps of the next layer
__device__ __forceinline__ void mlp_act(const f32x4 (&z)[4], bf16x8 (&B)[2]) {
#pragma unroll
  for (int ks = 0; ks < 2; ks++)
#pragma unroll
    for (int i = 0; i < 8; i++) B[ks][i] = (__bf16)gelu_f(z[2 * ks + (i >> 2)][i & 3]);
}

// Inference: features of n nodes (In: MlpPlain, SoA 10 x fstride, or MlpPacked)
// -> closure fields (SoA, 7 x cstride): nu_t = s0 softplus(o0), dsigma_k =
// s_{k+1} o_{k+1}.
//
// The GELU bounds it: 192 a node, each two quarter-rate instructions and five
// others, 126 us at 128^3 for 256 CUs.  So the rest is kept small: a wave takes
// two 16-node tiles at a time, which share the reads of the weights (in LDS, one
// copy per block, as operands) and, the second tile's outputs taken from rows
// 8..14 of the last product, one output pass over all 64 lanes; the inputs come
// as finished operands.  One tile at a time, its inputs loaded and scaled by
// predicated FP32 reads, took 205 us; this takes 159 us (262144 stored samples, read as FP32: 34 -> 26 us).
template <typename In>
__global__ __launch_bounds__(256, 4) void k_mlp_infer(const float *__restrict__ feat, long long fstride,
                                                      long long n, const bf16x8 *__restrict__ wf,
                                                      const float *__restrict__ th, float *__restrict__ clo,
                                                      long long cstride) {
  __shared__ bf16x8 wl[kFwdBlocks * 64];
  __shared__ alignas(16) float bl[2][kMlpNH];
  for (int i = threadIdx.x; i < kFwdBlocks * 64; i += 256) wl[i] = wf[i];
  if (threadIdx.x < 2 * kMlpNH)
    bl[threadIdx.x / kMlpNH][threadIdx.x % kMlpNH] =
        th[(threadIdx.x < kMlpNH ? kOffB2 : kOffB3) + threadIdx.x % kMlpNH];
  __syncthreads();
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const bf16x8 *A = wl + lane;       // block b at A[b * 64]
  const bf16x8 *Ah = wl + (lane ^ 8);  // its rows 8..15 and 0..7 exchanged
  const In in(feat, fstride, n, th, g);
  // lane groups 0, 1 write outputs 0..3, 4..6 of the first tile, 2, 3 of the second
  const int q0 = 4 * (g & 1);
  float so[4], bo[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    so[i] = q0 + i < kMlpNO ? th[kOffOut + q0 + i] : 0.f;
    bo[i] = q0 + i < kMlpNO ? th[kOffB4 + q0 + i] : 0.f;
  }
  const long long npair = (n + 31) / 32;
  const long long nw = (long long)gridDim.x * 4;
  long long t = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
  auto last = [&](long long node) { return node < n ? node : n - 1; };
  typename In::Raw nxt[2];
  if (t < npair) {
    in.load(nxt[0], last(t * 32 + c));
    in.load(nxt[1], last(t * 32 + 16 + c));
  }
  for (; t < npair; t += nw) {
    // keep the LDS reads inside the loop (hoisted, they would occupy the
    // registers the LDS copy is meant to free)
    asm volatile("" ::: "memory");
    const bf16x8 B1[2] = {in.operand(nxt[0]), in.operand(nxt[1])};
    if (t + nw < npair) {  // the next pair's inputs load while this one computes
      in.load(nxt[0], last((t + nw) * 32 + c));
      in.load(nxt[1], last((t + nw) * 32 + 16 + c));
    }
    f32x4 z[2][4];
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int mb = 0; mb < 4; mb++) {
      const bf16x8 a = A[mb * 64];
      z[0][mb] = mfma16(a, B1[0], zero);
      z[1][mb] = mfma16(a, B1[1], zero);
    }
    bf16x8 B[2][2];
    mlp_act(z[0], B[0]);
    mlp_act(z[1], B[1]);
#pragma unroll
    for (int l = 0; l < 2; l++) {
#pragma unroll
      for (int mb = 0; mb < 4; mb++) {
        const f32x4 b = *(const f32x4 *)&bl[l][16 * mb + 4 * g];
        const bf16x8 a0 = A[(4 + 8 * l + 2 * mb) * 64], a1 = A[(5 + 8 * l + 2 * mb) * 64];
#pragma unroll
        for (int k = 0; k < 2; k++) z[k][mb] = mfma16(a1, B[k][1], mfma16(a0, B[k][0], b));
      }
      mlp_act(z[0], B[0]);
      mlp_act(z[1], B[1]);
    }
    const f32x4 b = {bo[0], bo[1], bo[2], bo[3]};
    const f32x4 o0 = mfma16(A[21 * 64], B[0][1], mfma16(A[20 * 64], B[0][0], b));
    const f32x4 o1 = mfma16(Ah[21 * 64], B[1][1], mfma16(Ah[20 * 64], B[1][0], b));
    const long long node = t * 32 + 16 * (g >> 1) + c;
    f32x4 o;
#pragma unroll
    for (int i = 0; i < 4; i++) o[i] = g < 2 ? o0[i] : o1[i];
    const float sp = softplus_f(o[0]);
    o[0] = q0 ? o[0] : sp;
    if (node < n) {
      float *d = clo + q0 * cstride + node;
#pragma unroll
      for (int i = 0; i < 3; i++) d[i * cstride] = so[i] * o[i];
      if (q0 == 0) d[3 * cstride] = so[3] * o[3];
    }
  }
}

// Training, first launch: loss and gradient of a batch, one row of partial
// sums per block.  Column j of the batch is sample idx[j], first + j (no
// index list), or drawn from (seed, step, j) by k_mlp_grad itself.
//
// A block of 16 waves takes 64 samples at a time, wave (mb, t) the 16 features
// of block mb for the 16 samples of tile t: four activations a lane and layer
// where one wave per tile had 16, so the chain of MFMA, GELU and exchange is
// short and four waves per SIMD hide it.  Activations and deltas stay in LDS
// in two forms: as the operand of the next layer's product (`ex`) and
// feature-major (`row`), from which the block forms dW = delta H^T on the matrix
// cores right away, K = its 64 samples, into accumulators it keeps over all its
// groups.  inv = 1/(t_scale^2 * batch).
//
// Latency bounds it: a batch of 16384 is one group per CU (256 groups), and
// takes 17 us, k_mlp_update 5 us.  One wave per tile, 13.6 MB of BF16
// activations written for a second kernel that added dW with atomics, took 29 +
// 15.5 us, and the indices, two fills, Adam and the packing a launch each, 15 us
// more.  The weights are in LDS as they do not fit the registers: spilled, they
// were waited for in every phase (25 us).
constexpr int kGradTile = 64, kGradThreads = 1024;
constexpr int kRowH0 = 0, kRowH1 = 16, kRowH2 = 80, kRowH3 = 144, kRowD1 = 208, kRowD2 = 272, kRowD3 = 336,
              kRowD4 = 400, kGradRows = 416;
// row pitch 72: the four lane groups of a store fall on different banks, and
// 16-byte reads stay aligned
constexpr int kGradPitch = kGradTile + 8;
static_assert(kAux <= kMlpNF && kMlpNF < 16, "wave w brings input w and record entry w");

struct GradIdx {
  const int *idx;  // explicit columns, or null
  long long first; // idx null, ns == 0: sample first + j
  long long ns;    // > 0: drawn from ns samples
  uint64_t inv;    // floor((2^64 - 1) / ns)
  uint32_t seed, step;
};
__device__ __forceinline__ int grad_sample(const GradIdx &gi, int j) {
  if (gi.idx) return gi.idx[j];
  if (!gi.ns) return (int)(gi.first + j);
  // splitmix64 of (seed, step, j)
  uint64_t x = (uint64_t)gi.seed * 0x9E3779B97F4A7C15ull + (uint64_t)gi.step * 0xD1B54A32D192ED03ull + (uint64_t)j;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  x ^= x >> 31;
  // x mod ns: the quotient by the reciprocal is at most two short
  const uint64_t n = (uint64_t)gi.ns;
  uint64_t r = x - __umul64hi(x, gi.inv) * n;
  r -= r >= n ? n : 0;
  r -= r >= n ? n : 0;
  return (int)r;
}

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

// COLS: the columns of activations and deltas go to `cols`, [group of 64
// samples][row][sample], in place of dW.
template <bool COLS>
__global__ __launch_bounds__(kGradThreads) void k_mlp_grad(const float *__restrict__ feat, long long fstride,
                                                           const float *__restrict__ aux, long long astride,
                                                           GradIdx gi, int nb, const bf16x8 *__restrict__ wf,
                                                           const bf16x8 *__restrict__ wb,
                                                           const float *__restrict__ th, float inv,
                                                           float *__restrict__ part, bf16x8 *__restrict__ cols,
                                                           double *__restrict__ lpart) {
  __shared__ alignas(16) __bf16 row[kGradRows][kGradPitch];
  __shared__ bf16x8 ex[2][4][2][64];            // operand of the next product: [buffer][tile][K step][lane]
  __shared__ float raw[kMlpNF + kAux][kGradTile];  // inputs and the auxiliary record
  __shared__ bf16x8 wl[(kFwdBlocks + kBwdBlocks) * 64];  // both packs
  __shared__ float cst[kMlpNParam - kOffB4];  // its bias, the input and output scales
  __shared__ double lw[4];
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
  // scalar: the matrix instructions ignore the execution mask, so a branch on
  // the wave around them has to be a jump
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int t = w & 3, mb = w >> 2;
  const int col = 16 * t + c;
  for (int i = tid; i < (kFwdBlocks + kBwdBlocks) * 64; i += kGradThreads)
    wl[i] = i < kFwdBlocks * 64 ? wf[i] : wb[i - kFwdBlocks * 64];
  const bf16x8 *W = wl + lane, *T = W + kFwdBlocks * 64;  // block k at [k * 64]
  const f32x4 b2 = *(const f32x4 *)(th + kOffB2 + 16 * mb + 4 * g);
  const f32x4 b3 = *(const f32x4 *)(th + kOffB3 + 16 * mb + 4 * g);
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  if (w == 15 && lane < kMlpNParam - kOffB4) cst[lane] = th[kOffB4 + lane];
  const float *sin = cst + (kOffIn - kOffB4), *sout = cst + (kOffOut - kOffB4);
  __syncthreads();
  f32x4 w2 = zero, w3 = zero, wx = zero, wy = zero;  // accumulators of dW
  bf16x8 ones;
#pragma unroll
  for (int i = 0; i < 8; i++) ones[i] = (__bf16)(c == 0 ? 1.f : 0.f);
  double lsum = 0.0;

  // four features of a sample: exchanged as its operand, kept feature-major
  auto put = [&](int buf, int row0, const f32x4 &v) {
    const bf16x4 h = __builtin_convertvector(v, bf16x4);
#pragma unroll
    for (int i = 0; i < 4; i++) row[row0 + 16 * mb + 4 * g + i][col] = h[i];
    if (buf >= 0) ((bf16x4 *)&ex[buf][t][mb >> 1][lane])[mb & 1] = h;
  };
  // dW block of 16 output features (rows d0..) by 16 input features (rows h0..;
  // negative: the bias)
  auto contract = [&](f32x4 &acc, int d0, int h0) {
#pragma unroll
    for (int k = 0; k < kGradTile; k += 32) {
      const bf16x8 a = *(const bf16x8 *)&row[d0 + c][k + 8 * g];
      const bf16x8 b = h0 < 0 ? ones : *(const bf16x8 *)&row[(h0 < 0 ? 0 : h0) + c][k + 8 * g];
      acc = mfma16(a, b, acc);
    }
  };

  for (int j0 = blockIdx.x * kGradTile; j0 < nb; j0 += gridDim.x * kGradTile) {
    // ---- inputs: wave w brings input w (rows 10..15 of H0: the constant 1,
    // zeros) and record entry w, lane = sample
    const int j = j0 + lane;
    const bool in = j < nb;
    float v = 0.f, a = 0.f;
    if (in && w < kMlpNF) {
      const long long s = grad_sample(gi, j);
      v = feat[w * fstride + s];
      if (w < kAux) a = aux[w * astride + s];
    }
    if (w < kMlpNF) raw[w][lane] = v;
    if (w < kAux) raw[kMlpNF + w][lane] = a;
    row[kRowH0 + w][lane] = (__bf16)(w < kMlpNF ? (in ? v * sin[w] : 0.f) : (w == kMlpNF ? 1.f : 0.f));
    __syncthreads();
    // ---- forward
    bf16x8 B;
#pragma unroll
    for (int i = 0; i < 8; i++) B[i] = g < 2 ? row[kRowH0 + 8 * (g & 1) + i][col] : (__bf16)0.f;
    const f32x4 z1 = mfma16(W[mb * 64], B, zero);
    // GELU; its derivative stays for the backward pass
    auto act = [&](const f32x4 &z, f32x4 &dg) {
      f32x4 h;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        h[i] = gelu_f(z[i]);
        dg[i] = gelu_grad_f(z[i]);
      }
      return h;
    };
    // the two weight blocks of a product are read ahead of the barrier before it
    f32x4 g1, g2, g3;
    bf16x8 A0 = W[(4 + 2 * mb) * 64], A1 = W[(5 + 2 * mb) * 64];
    put(0, kRowH1, act(z1, g1));
    __syncthreads();
    f32x4 z2 = mfma16(A0, ex[0][t][0][lane], b2);
    z2 = mfma16(A1, ex[0][t][1][lane], z2);
    A0 = W[(12 + 2 * mb) * 64], A1 = W[(13 + 2 * mb) * 64];
    put(1, kRowH2, act(z2, g2));
    __syncthreads();
    f32x4 z3 = mfma16(A0, ex[1][t][0][lane], b3);
    z3 = mfma16(A1, ex[1][t][1][lane], z3);
    A0 = W[20 * 64], A1 = W[21 * 64];
    put(0, kRowH3, act(z3, g3));
    __syncthreads();
    // ---- loss and output deltas: one wave per tile (lane group 0 holds a
    // sample's outputs 0..3, group 1 outputs 4..6)
    if (mb == 0) {
      f32x4 o;
#pragma unroll
      for (int i = 0; i < 4; i++) o[i] = 4 * g + i < kMlpNO ? cst[4 * (g & 1) + i] : 0.f;
      o = mfma16(A0, ex[0][t][0][lane], o);
      o = mfma16(A1, ex[0][t][1][lane], o);
      const float o4 = __shfl(o[0], c + 16), o5 = __shfl(o[1], c + 16), o6 = __shfl(o[2], c + 16);
      bf16x8 Bd;
#pragma unroll
      for (int i = 0; i < 8; i++) Bd[i] = (__bf16)0.f;
      if (g == 0) {
        float dlt[7] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (j0 + col < nb) {
          const float ov[7] = {o[0], o[1], o[2], o[3], o4, o5, o6};
          const float s0 = sout[0];
          const float nu = s0 * softplus_f(ov[0]);
          const float rho = raw[kMlpNF][col];
          float dnu = 0.f, l = 0.f;
#pragma unroll
          for (int k = 0; k < 6; k++) {
            const float S = raw[k][col];
            const float T = raw[kMlpNF + 1 + k][col];
            const float sk = sout[1 + k];
            const float M = fmaf(-2.f * rho * nu, S, sk * ov[1 + k]);
            const float r = M - T;
            const float wk = k < 3 ? 1.f : 2.f;
            l += wk * r * r;
            const float dM = 2.f * wk * r * inv;
            dnu += dM * (-2.f * rho * S);
            dlt[1 + k] = dM * sk;
          }
          dlt[0] = dnu * s0 / (1.f + __expf(-ov[0]));
          lsum += (double)l * (double)inv;
        }
#pragma unroll
        for (int i = 0; i < 7; i++) Bd[i] = (__bf16)dlt[i];
#pragma unroll
        for (int i = 0; i < 8; i++) {
          row[kRowD4 + i][col] = Bd[i];
          row[kRowD4 + 8 + i][col] = (__bf16)0.f;
        }
      }
      ex[1][t][0][lane] = Bd;
    }
    A0 = T[mb * 64];
    __syncthreads();
    // ---- backward: delta_3 = (W4 delta_4) * gelu'(z3), ...
    put(0, kRowD3, mfma16(A0, ex[1][t][0][lane], zero) * g3);
    A0 = T[(4 + 2 * mb) * 64], A1 = T[(5 + 2 * mb) * 64];
    __syncthreads();
    f32x4 acc = mfma16(A0, ex[0][t][0][lane], zero);
    acc = mfma16(A1, ex[0][t][1][lane], acc);
    A0 = T[(12 + 2 * mb) * 64], A1 = T[(13 + 2 * mb) * 64];
    put(1, kRowD2, acc * g2);
    __syncthreads();
    acc = mfma16(A0, ex[1][t][0][lane], zero);
    acc = mfma16(A1, ex[1][t][1][lane], acc);
    put(-1, kRowD1, acc * g1);
    __syncthreads();
    if constexpr (COLS) {
      bf16x8 *o = cols + (size_t)(j0 / kGradTile) * kGradRows * (kGradTile / 8);
      for (int i = tid; i < kGradRows * (kGradTile / 8); i += kGradThreads)
        o[i] = *(const bf16x8 *)&row[i / (kGradTile / 8)][i % (kGradTile / 8) * 8];
    } else {
      // ---- dW: the 16 blocks each of layers 2 and 3, a block per wave; the four
      // of layers 1 (its bias is input row 10) and 4 and the biases of layers 2
      // and 3 on waves t = 0..3; the bias of layer 4 on one wave more
      contract(w2, kRowD2 + 16 * mb, kRowH1 + 16 * t);
      contract(w3, kRowD3 + 16 * mb, kRowH2 + 16 * t);
      contract(wx, t == 1 ? kRowD4 : (t == 0 ? kRowD1 : (t == 2 ? kRowD2 : kRowD3)) + 16 * mb,
               t == 0 ? kRowH0 : (t == 1 ? kRowH3 + 16 * mb : -1));
      if (w == 0) contract(wy, kRowD4, -1);
    }
    __syncthreads();  // the next group overwrites the rows
  }

  if constexpr (!COLS) {
    // ---- partial sums in the natural parameter order: lane (g, c) of a block has
    // outputs 16 m + 4g + i of input 16 n + c
    float *o = part + (size_t)blockIdx.x * kMlpNParam;
    const int m0 = 16 * mb + 4 * g;
    *(f32x4 *)(o + kOffW2 + (16 * t + c) * kMlpNH + m0) = w2;
    *(f32x4 *)(o + kOffW3 + (16 * t + c) * kMlpNH + m0) = w3;
    if (t == 0) {
      if (c < kMlpNF) *(f32x4 *)(o + kOffW1 + c * kMlpNH + m0) = wx;
      else if (c == kMlpNF) *(f32x4 *)(o + kOffB1 + m0) = wx;
    } else if (t == 1) {
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (4 * g + i < kMlpNO) o[kOffW4 + (16 * mb + c) * kMlpNO + 4 * g + i] = wx[i];
    } else if (c == 0) {
      *(f32x4 *)(o + (t == 2 ? kOffB2 : kOffB3) + m0) = wx;
    }
    if (w == 0 && c == 0) {
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (4 * g + i < kMlpNO) o[kOffB4 + 4 * g + i] = wy[i];
    }
  }
  // FP64 loss: one sum per tile column, then per block
  for (int off = 32; off > 0; off >>= 1) lsum += __shfl_down(lsum, off);
  if (mb == 0 && lane == 0) lw[t] = lsum;
  __syncthreads();
  if (tid == 0) lpart[blockIdx.x] = (lw[0] + lw[1]) + (lw[2] + lw[3]);
}

// position of a weight in the packed operand blocks (the inverse of
// k_mlp_pack): a forward and, but for layer 1 and the biases, a backward entry
__device__ __forceinline__ void mlp_repack(int i, float x, __bf16 *__restrict__ fwd, __bf16 *__restrict__ bwd) {
  const __bf16 h = (__bf16)x;
  // element (row 16 mb + c, k) of a 64-wide product: block 2 mb + ks, in the order perm
  auto hidden = [](int r, int k) {
    const int q = k & 31;
    return ((2 * (r >> 4) + (k >> 5)) * 64 + 16 * ((q & 15) >> 2) + (r & 15)) * 8 + 4 * (q >> 4) + (q & 3);
  };
  if (i < kOffW2) {  // W1 (10 x 64) and, as input 10, b1
    const int k = i / kMlpNH, m = i % kMlpNH;
    fwd[((m >> 4) * 64 + 16 * (k >> 3) + (m & 15)) * 8 + (k & 7)] = h;
  } else if (i < kOffB2) {
    const int k = (i - kOffW2) / kMlpNH, m = (i - kOffW2) % kMlpNH;
    fwd[4 * 512 + hidden(m, k)] = h;
    bwd[12 * 512 + hidden(k, m)] = h;
  } else if (i >= kOffW3 && i < kOffB3) {
    const int k = (i - kOffW3) / kMlpNH, m = (i - kOffW3) % kMlpNH;
    fwd[12 * 512 + hidden(m, k)] = h;
    bwd[4 * 512 + hidden(k, m)] = h;
  } else if (i >= kOffW4 && i < kOffB4) {
    const int k = (i - kOffW4) / kMlpNO, q = (i - kOffW4) % kMlpNO;
    fwd[20 * 512 + hidden(q, k)] = h;
    bwd[((k >> 4) * 64 + (k & 15)) * 8 + q] = h;
  }
}

// Adam: the 1-based step t, one parameter i with its gradient g and its state,
// and its packed operands
struct AdamStep {
  float *th, *m1, *m2;
  __bf16 *fwd, *bwd;
  float lr, b1, b2, eps, t;
  // 1 - b2^t cancels: the power's last bit is up to 6e-5 / t of it and scales
  // every step, so the power is the device's, and is formed while the gradient
  // is read
  struct Corr {
    float c1, c2;
  };
  __device__ __forceinline__ Corr corrections() const { return {1.f - powf(b1, t), 1.f - powf(b2, t)}; }
  __device__ __forceinline__ void operator()(const Corr &k, int i, float g, float x, float a, float v) const {
    a = fmaf(b1, a, (1.f - b1) * g);
    v = fmaf(b2, v, (1.f - b2) * g * g);
    m1[i] = a;
    m2[i] = v;
    const float mh = a / k.c1, vh = v / k.c2;
    x -= lr * mh / (sqrtf(vh) + eps);
    th[i] = x;
    mlp_repack(i, x, fwd, bwd);
  }
};

// Training, second launch: the sums of `rows` partial gradients, in a fixed
// order, and of the partial losses.  ADAM: one Adam step on the weights and
// biases (the scales stay); else the sums are added to grad and *loss.
//
// A block takes 64 parameters, its 16 waves every 16th row each: 256 rows are
// 9.7 MB read by 149 blocks.
template <bool ADAM>
__global__ __launch_bounds__(1024) void k_mlp_update(const float *__restrict__ part, const double *__restrict__ lpart,
                                                     int rows, float *__restrict__ grad, double *__restrict__ loss,
                                                     AdamStep adam) {
  __shared__ float s[16][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int i = blockIdx.x * 64 + lane;
  AdamStep::Corr corr;
  if constexpr (ADAM) corr = adam.corrections();
  float a = 0.f;
  if (i < kOffIn) {
#pragma unroll 8
    for (int r = w; r < rows; r += 16) a += part[(size_t)r * kMlpNParam + i];
  }
  s[w][lane] = a;
  __syncthreads();
  if (blockIdx.x == 0 && w == 1) {
    double l = 0.0;
    for (int r = lane; r < rows; r += 64) l += lpart[r];
    for (int off = 32; off > 0; off >>= 1) l += __shfl_down(l, off);
    if (lane == 0) *loss = ADAM ? l : *loss + l;
  }
  if (w || i >= kOffIn) return;
  float gsum = 0.f;
#pragma unroll
  for (int k = 0; k < 16; k++) gsum += s[k][lane];
  if constexpr (ADAM) {
    adam(corr, i, gsum, adam.th[i], adam.m1[i], adam.m2[i]);
  } else {
    grad[i] += gsum;
  }
}

// Training, second launch after k_mlp_grad<true>: one block per dW block of 16
// output features by 16 input features (or by the bias), one wave per slice
// of 512 samples, each one chain of matrix instructions, added in a fixed order:
// a partial slice first, then the others.
//
// The rounding of these sums decides what comes out of a training: one other
// bit of a gradient is 1e-5 in the weights and 3e-3 in the outputs 100 steps
// on.  Slices of 512 added with atomics gave the same sums, bit for bit with
// one or two slices and in many runs with up to five (a partial one arrived
// first: 2088 samples, 22 steps: outputs 7e-9 from a run of theirs, theirs 1e-8
// from one another, k_mlp_update's 7e-7, in the median).  From nine on
// k_mlp_update's sums, in groups of 64, lie as close to a run of theirs as two of
// theirs to one another (4227 samples, 41 steps: 2e-5, theirs 3e-4).  So the line
// is eight slices.  Latency bounds it: one read of the columns, all of a slice in
// flight, 16 dependent MFMAs and Adam.  A step of 1024 samples takes 16.7 us, of
// 2048 19.1, of 4096 23.7 (k_mlp_update's way 14.7, 15.1 and 16.2; with atomics
// 31, 32 and 35).
constexpr int kSlice = 512, kWgradJobs = 4 + 20 + 20 + 5, kWgradWaves = 8;
struct WgradJob {
  int layer;  // 1..4
  int mb;     // output-feature block (rows of delta)
  int nb;     // input-feature block (rows of H), -1: bias
};
__device__ __forceinline__ WgradJob wgrad_job(int j) {
  if (j < 4) return {1, j, 0};  // 16 input rows: 10 features, the bias row, zeros
  j -= 4;
  if (j < 20) return {2, j / 5, j % 5 == 4 ? -1 : j % 5};
  j -= 20;
  if (j < 20) return {3, j / 5, j % 5 == 4 ? -1 : j % 5};
  j -= 20;
  return {4, 0, j == 4 ? -1 : j};
}
// parameter of output feature jo and input feature ki (of the bias: column 0), or -1
__device__ __forceinline__ int wgrad_param(const WgradJob &jb, int jo, int ki) {
  switch (jb.layer) {
    case 1:
      return ki < kMlpNF ? kOffW1 + ki * kMlpNH + jo : (ki == kMlpNF ? kOffB1 + jo : -1);
    case 2:
      return jb.nb >= 0 ? kOffW2 + ki * kMlpNH + jo : (ki == 0 ? kOffB2 + jo : -1);
    case 3:
      return jb.nb >= 0 ? kOffW3 + ki * kMlpNH + jo : (ki == 0 ? kOffB3 + jo : -1);
    default:
      if (jo >= kMlpNO) return -1;
      return jb.nb >= 0 ? kOffW4 + ki * kMlpNO + jo : (ki == 0 ? kOffB4 + jo : -1);
  }
}
template <bool ADAM>
__global__ __launch_bounds__(64 * kWgradWaves) void k_mlp_wgrad(const bf16x8 *__restrict__ cols, int nb,
                                                                const double *__restrict__ lpart, int rows,
                                                                float *__restrict__ grad, double *__restrict__ loss,
                                                                AdamStep adam) {
  __shared__ f32x4 s[kWgradWaves][64];
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (blockIdx.x == kWgradJobs) {
    if (w) return;
    double l = 0.0;
    for (int r = lane; r < rows; r += 64) l += lpart[r];
    for (int off = 32; off > 0; off >>= 1) l += __shfl_down(l, off);
    if (lane == 0) *loss = ADAM ? l : *loss + l;
    return;
  }
  const WgradJob jb = wgrad_job(blockIdx.x);
  AdamStep::Corr corr;
  if constexpr (ADAM) corr = adam.corrections();
  int par[4];
  float x[4], a1[4], a2[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    par[i] = wgrad_param(jb, 16 * jb.mb + 4 * g + i, 16 * (jb.nb < 0 ? 0 : jb.nb) + c);
    if (ADAM && w == 0 && par[i] >= 0) {
      x[i] = adam.th[par[i]];
      a1[i] = adam.m1[par[i]];
      a2[i] = adam.m2[par[i]];
    }
  }
  constexpr int kCh = kGradTile / 8, kGroups = kSlice / kGradTile;  // 16-byte chunks of a row, groups of a slice
  const int d0 = (jb.layer == 1 ? kRowD1 : (jb.layer == 2 ? kRowD2 : (jb.layer == 3 ? kRowD3 : kRowD4))) + 16 * jb.mb;
  const int h0 = (jb.layer == 1 ? kRowH0 : (jb.layer == 2 ? kRowH1 : (jb.layer == 3 ? kRowH2 : kRowH3))) + 16 * jb.nb;
  const int groups = (nb + kGradTile - 1) / kGradTile;
  bf16x8 none, ones;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    none[i] = (__bf16)0.f;
    ones[i] = (__bf16)(c == 0 ? 1.f : 0.f);
  }
  bf16x8 a[2 * kGroups], b[2 * kGroups];
#pragma unroll
  for (int k = 0; k < 2 * kGroups; k++) {
    // groups beyond the batch: zeros
    a[k] = none;
    b[k] = ones;
    const int gr = w * kGroups + k / 2;
    if (gr < groups) {
      const bf16x8 *p = cols + (size_t)gr * kGradRows * kCh + 4 * (k & 1) + g;
      a[k] = p[(d0 + c) * kCh];
      if (jb.nb >= 0) b[k] = p[(h0 + c) * kCh];
    }
  }
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < 2 * kGroups; k++) acc = mfma16(a[k], b[k], acc);
  s[w][lane] = acc;
  __syncthreads();
  if (w) return;
  const int whole = nb / kSlice;
  f32x4 sum = {0.f, 0.f, 0.f, 0.f};
  if (nb % kSlice) sum += s[whole][lane];
  for (int k = 0; k < whole; k++) sum += s[k][lane];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    if (par[i] < 0) continue;
    if constexpr (ADAM) adam(corr, par[i], sum[i], x[i], a1[i], a2[i]);
    else grad[par[i]] += sum[i];
  }
}

// Field views for the filter and input kernels: the lattice state (storage
// type S, per-field scale) or a plain FP32 SoA buffer.  `col` locates a column
// (x, y), `get` reads field q of its node in plane z.
template <typename S>
struct StateView {
  const S *base;
  struct Col {
    uint64_t off;  // in the moment layout
    uint32_t xy;   // in the plain phi field
  };
  __device__ __forceinline__ Col col(int x, int y, const Params &p) const {
    return Col{node_off<(int)sizeof(S)>(p, x, y), (uint32_t)(x + p.nx * y)};
  }
  __device__ __forceinline__ float get(int q, const Col &c, int z, const Params &p) const {
    if (q == TSLB_PHI) return ldv(base, (uint64_t)p.phi0 + (uint64_t)((long long)p.nx * p.ny * z) + c.xy, p, q);
    return ldv(base, plane_off(p, z) + c.off + (uint64_t)(q * p.qs), p, q);
  }
};
struct PlainView {
  const float *base;
  long long fs;
  struct Col {
    uint32_t xy;
  };
  __device__ __forceinline__ Col col(int x, int y, const Params &p) const { return Col{(uint32_t)(x + p.nx * y)}; }
  __device__ __forceinline__ float get(int q, const Col &c, int z, const Params &p) const {
    return base[q * fs + (long long)p.nx * p.ny * z + c.xy];
  }
};

// Box filter of a fine lattice by r^3 blocks: coarse rho_bar - 1, Favre
// velocity, phi_bar (SoA, 5 x nc) and the aux record rho_bar, tau[6]
// (SoA, 7 x astride, written at column offset aoff).  tau = <rho (u-u~)(u-u~)>.
template <typename S>
__global__ __launch_bounds__(256) void k_box_filter(StateView<S> f, Params p, int r, float *__restrict__ coarse,
                                                    long long nc, float *__restrict__ aux, long long astride,
                                                    long long aoff) {
  const int ncx = p.nx / r, ncy = p.ny / r, ncz = p.nz / r;
  const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
  if (t >= nc) return;
  const int I = (int)(t % ncx), J = (int)((t / ncx) % ncy), K = (int)(t / ((long long)ncx * ncy));
  (void)ncz;
  double sr = 0, su = 0, sv = 0, sw = 0, sp = 0;
  for (int k = 0; k < r; k++)
    for (int j = 0; j < r; j++)
      for (int i = 0; i < r; i++) {
        const auto c = f.col(I * r + i, J * r + j, p);
        const int z = K * r + k;
        const float rho = 1.f + f.get(TSLB_RHO, c, z, p);
        sr += rho;
        su += (double)rho * f.get(TSLB_U, c, z, p);
        sv += (double)rho * f.get(TSLB_V, c, z, p);
        sw += (double)rho * f.get(TSLB_W, c, z, p);
        if (p.ncomp == 2) sp += f.get(TSLB_PHI, c, z, p);
      }
  const double inv = 1.0 / ((double)r * r * r);
  const double rb = sr * inv, ut = su / sr, vt = sv / sr, wt = sw / sr;
  double txx = 0, tyy = 0, tzz = 0, txy = 0, txz = 0, tyz = 0;
  for (int k = 0; k < r; k++)
    for (int j = 0; j < r; j++)
      for (int i = 0; i < r; i++) {
        const auto c = f.col(I * r + i, J * r + j, p);
        const int z = K * r + k;
        const double rho = 1.0 + f.get(TSLB_RHO, c, z, p);
        const double du = f.get(TSLB_U, c, z, p) - ut, dv = f.get(TSLB_V, c, z, p) - vt,
                     dw = f.get(TSLB_W, c, z, p) - wt;
        txx += rho * du * du;
        tyy += rho * dv * dv;
        tzz += rho * dw * dw;
        txy += rho * du * dv;
        txz += rho * du * dw;
        tyz += rho * dv * dw;
      }
  coarse[t] = (float)(rb - 1.0);
  coarse[nc + t] = (float)ut;
  coarse[2 * nc + t] = (float)vt;
  coarse[3 * nc + t] = (float)wt;
  coarse[4 * nc + t] = (float)(sp * inv);
  const long long a = aoff + t;
  aux[a] = (float)rb;
  aux[astride + a] = (float)(txx * inv);
  aux[2 * astride + a] = (float)(tyy * inv);
  aux[3 * astride + a] = (float)(tzz * inv);
  aux[4 * astride + a] = (float)(txy * inv);
  aux[5 * astride + a] = (float)(txz * inv);
  aux[6 * astride + a] = (float)(tyz * inv);
}

// Closure inputs of every node of a grid (nx, ny, nz, periodic flags of p):
// S from the isotropic gradient (3 sum_l w_l c_l f(x + c_l), the stencil of
// grad_axis) of (u, v, w), grad(phi), phi; the nearest
// interior node across a wall.  Velocity at fields fu..fu+2 and phi at field
// fphi of a source (without PHI: phi = 0).  Out takes them as FP32 (SoA 10 x
// stride) or as the scaled BF16 operand of the first layer.
struct FeatPlain {
  float *o;
  long long stride;
  __device__ __forceinline__ void put(long long node, const float (&v)[kMlpNF]) const {
#pragma unroll
    for (int k = 0; k < kMlpNF; k++) o[k * stride + node] = v[k];
  }
};
struct FeatPacked {
  bf16x8 *lo;
  bf16x2 *hi;
  const float *th;
  __device__ __forceinline__ void put(long long node, const float (&v)[kMlpNF]) const {
    bf16x8 a;
#pragma unroll
    for (int k = 0; k < 8; k++) a[k] = (__bf16)(v[k] * th[kOffIn + k]);
    lo[node] = a;
    hi[node] = bf16x2{(__bf16)(v[8] * th[kOffIn + 8]), (__bf16)(v[9] * th[kOffIn + 9])};
  }
};
//
// A 64x4 block marches a z-chunk.  It keeps four planes of its 66x6 footprint
// in an LDS ring (25 KiB; the plane two ahead loads into registers meanwhile)
// and forms the 12 sums of a node from 104 LDS reads, in the order of the
// directions, those with a zero coefficient too: a NaN or an infinity of any
// neighbour shows in all components (2 us of the 33).  One thread per node
// reading its 26 neighbours from memory took 79 us at 128^3 for its addresses
// and L1 reads; this one takes 33 us (84 MB written and 34 MB read: 24 us at the
// rate of a copy).
constexpr int FTX = 64, FTY = 4, FSW = FTX + 2, FSH = FTY + 2, FNSLOT = FSW * FSH, FNT = FTX * FTY;
static_assert(FNSLOT <= 2 * FNT, "at most two footprint slots per thread");
template <typename Src, bool PHI, typename Out>
__global__ __launch_bounds__(FNT) void k_features(Src f, Params p, int fu, int fphi, Out out, int zc) {
  constexpr int NQ = PHI ? 4 : 3;
  __shared__ float ring[4][NQ][FNSLOT];
  const int tid = threadIdx.x, tx = tid % FTX, ty = tid / FTX;
  const int tilx = (p.nx + FTX - 1) / FTX, tily = (p.ny + FTY - 1) / FTY;
  int b = xcd_tile(blockIdx.x, gridDim.x);
  const int x0 = b % tilx * FTX;
  b /= tilx;
  const int y0 = b % tily * FTY, z0 = b / tily * zc, z1 = min(z0 + zc, p.nz);
  const int x = x0 + tx, y = y0 + ty;
  const bool active = x < p.nx && y < p.ny, two = tid + FNT < FNSLOT;
  auto column = [&](int sl) {
    return f.col(clampw(x0 + sl % FSW - 1, p.nx, p.px), clampw(y0 + sl / FSW - 1, p.ny, p.py), p);
  };
  const auto c0 = column(tid), c1 = column(two ? tid + FNT : tid);
  float n0[NQ], n1[NQ];
  auto issue = [&](int z) {
    const int gz = clampw(z, p.nz, p.pz);
#pragma unroll
    for (int q = 0; q < NQ; q++) {
      const int fq = q < 3 ? fu + q : fphi;
      n0[q] = f.get(fq, c0, gz, p);
      if (two) n1[q] = f.get(fq, c1, gz, p);
    }
  };
  auto commit = [&](int z) {
    float(*d)[FNSLOT] = ring[(z - z0 + 4) & 3];
#pragma unroll
    for (int q = 0; q < NQ; q++) {
      d[q][tid] = n0[q];
      if (two) d[q][tid + FNT] = n1[q];
    }
  };
  issue(z0 - 1);
  commit(z0 - 1);
  issue(z0);
  commit(z0);
  issue(z0 + 1);
  // the slot of plane z + 1 held plane z - 3, last read before the previous
  // barrier
  for (int z = z0; z < z1; z++) {
    commit(z + 1);
    if (z + 2 <= z1) issue(z + 2);
    __syncthreads();
    if (!active) continue;
    const int own = (ty + 1) * FSW + tx + 1;
    float g[NQ][3];
#pragma unroll
    for (int q = 0; q < NQ; q++) g[q][0] = g[q][1] = g[q][2] = 0.f;
#pragma unroll
    for (int l = 1; l < 27; l++) {
      const float *s = ring[(z + kCZ[l] - z0 + 4) & 3][0] + own + kCY[l] * FSW + kCX[l];
      const float w3 = 3.f * wgt(l);
#pragma unroll
      for (int q = 0; q < NQ; q++) {
        const float v = s[q * FNSLOT];
        g[q][0] = fmaf(w3 * (float)kCX[l], v, g[q][0]);
        g[q][1] = fmaf(w3 * (float)kCY[l], v, g[q][1]);
        g[q][2] = fmaf(w3 * (float)kCZ[l], v, g[q][2]);
      }
    }
    const float v[kMlpNF] = {g[0][0],
                             g[1][1],
                             g[2][2],
                             0.5f * (g[0][1] + g[1][0]),
                             0.5f * (g[0][2] + g[2][0]),
                             0.5f * (g[1][2] + g[2][1]),
                             PHI ? g[NQ - 1][0] : 0.f,
                             PHI ? g[NQ - 1][1] : 0.f,
                             PHI ? g[NQ - 1][2] : 0.f,
                             PHI ? ring[(z - z0 + 4) & 3][NQ - 1][own] : 0.f};
    out.put((long long)p.nx * p.ny * z + (x + p.nx * y), v);
  }
}
