// lceq_mlp.hip -- learned proposal for the adjoint-Higgs update (no
// counterpart in the reference; the plain update it competes with is the
// Metropolis step of f/ahiggs1.f).
//
// Per site x of the parity being updated, with F = the hopping force of
// f/a_force.f (fixed while this parity is updated), a small network
//   10 inputs -> 64 SiLU -> 64 SiLU -> 6 outputs
// gives the mean mu and log-scale s of a Gaussian proposal in the frame
// (e1, e2, e3) with e1 = F/|F|.  The inputs are the local a (3) and the
// hopping sum (3) in that frame, |F|, beta_A, beta_2 and beta_4; the frame
// removes the global SO(3) orientation, on which the action does not depend.
// a' is drawn from N(mu(a), exp(s(a))) and accepted with the FP64 Metropolis-
// Hastings probability
//   min(1, exp(S(a) - S(a')) q(a | a') / q(a' | a)),
// S the site action of f/ahiggs1.f:64-92, so the chain is exact whatever the
// network computes; the reverse density needs a second evaluation at a'.
// Inference runs on bf16 MFMA (v_mfma_f32_16x16x32_bf16, fp32 accumulation),
// one 64-site batch per wave.  Training (maximum likelihood of the moves of
// several Metropolis steps at fixed F) is hand-written FP32 with Adam.
#include <math.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <cmath>
#include <numeric>
#include <vector>

#include "../../include/lceq.h"
#include "lceq_internal.hpp"
#include "lceq_sites.hpp"

using namespace lceq;

#include "lceq_mlp.hpp"

using namespace lceq::mlp;

namespace {

constexpr int TB = 256;

template <int ST>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_higgs_mlp(MlpArgs p) {
  __shared__ MlpLds lds[4];
  mlp_higgs_site<ST>(p, xcd_block(p.nb), lds[threadIdx.x >> 6]);
}

// The inference network on given raw inputs (rows of NIN), for tests
__global__ __launch_bounds__(256) void k_mlp_eval(const MlpPack* __restrict__ P,
                                                  const float* __restrict__ x, float* __restrict__ y,
                                                  int n) {
  __shared__ MlpLds lds[4];
  int i = blockIdx.x * TB + threadIdx.x;
  int il = i < n ? i : n - 1;
  float xin[NIN], o[NOUT];
  MlpRegs W;
  mlp_load(P, W);
  mlp_stage_bias(P, lds[threadIdx.x >> 6]);
#pragma unroll
  for (int k = 0; k < NIN; ++k) xin[k] = x[(size_t)il * NIN + k];
  mlp_eval<4>(P, W, xin, o, lds[threadIdx.x >> 6]);
  if (i < n)
#pragma unroll
    for (int j = 0; j < NOUT; ++j) y[(size_t)i * NOUT + j] = o[j];
}

// ---------------------------------------------------------- training data

// Record of site s (every stride-th site of parity eo): the raw features of
// the current a at the current F, and (second kernel, after the heatbath
// steps) the new a in the same frame.
__global__ __launch_bounds__(256) void k_mlp_record(Geom g, const double* __restrict__ U,
                                                    const double* __restrict__ A, int eo, int stride,
                                                    int nrec, double ba, double b2, double b4,
                                                    float* __restrict__ out, int target) {
  int r = blockIdx.x * TB + threadIdx.x;
  if (r >= nrec) return;
  unsigned s = (unsigned)r * (unsigned)stride;
  Coord c = site_coord(g, eo, (int)s);
  vec3 F = hop_force(U, A, g, eo, s, c);
  Frame fr = make_frame(F.x);
  vec3 av = ld_higgs(A, g, eo, s);
  double y[3];
  to_frame(fr, av.x, y);
  float* rec = out + (size_t)r * NREC;
  if (target) {
    rec[NIN] = (float)y[0];
    rec[NIN + 1] = (float)y[1];
    rec[NIN + 2] = (float)y[2];
  } else {
    float x[NIN];
    raw_features(y, fr.fn, ba, b2, b4, x);
    for (int k = 0; k < NIN; ++k) rec[k] = x[k];
  }
}

// --------------------------------------------------------------- training

constexpr int TR_SAMPLES = 32;  // samples per block: one partial gradient and loss each
constexpr int TR_TB = 512;

// Rows of a block's samples are padded to 36 floats, rows of W2 to 68: the 16
// rows x 4 columns of an MFMA operand then fall on 64 banks.  x and dout are
// padded to whole K steps of 4: row NIN of x is ones (its products with a
// layer's deltas are the bias gradients), the others zero.
constexpr int XROWS = 12, DROWS = 8;
struct alignas(16) TrainLds {
  float x[XROWS][36], y[3][36];
  float h1[NH][36], d1[NH][36], h2[NH][36], d2[NH][36];
  float o[NOUT][36], dout[DROWS][36];
  float w1[NIN][NH], w2[NH][68], w3[NH][NOUT];
  float b1[NH], b2[NH], b3[8];
  float loss[36];
};
static_assert(sizeof(TrainLds) <= 64 * 1024, "static LDS of one block");

__device__ __forceinline__ float dsilu(float z) {
  float sg = 1.0f / (1.0f + expf(-z));
  return sg * (1.0f + z * (1.0f - sg));
}

// Record b of a mini-batch of the epoch's permutation i -> (mult i + offs)
// mod n: (base + mult b) mod n, base that of the batch's first record; mult
// and base below n < 2^32, b < 2^31.  The quotient mult b / n, below 2^31, is
// within one of its estimate in double precision.
struct TrainBatch {
  uint64_t mult, base, n;
  double rn;  // 1 / n
};
__device__ __forceinline__ size_t train_record(const TrainBatch& t, int b) {
  uint64_t a = t.mult * (uint64_t)b;
  int64_t n = (int64_t)t.n, r = (int64_t)(a - (uint64_t)((double)a * t.rn) * t.n);
  r += r < 0 ? n : 0;
  r -= r >= n ? n : 0;
  r += (int64_t)t.base;
  return (size_t)(r >= n ? r - n : r);
}

// D = C + A B with fp32 operands and accumulation: lane l holds A[l % 16][l /
// 16] (16 x 4), B[l / 16][l % 16] (4 x 16) and D's column l % 16, rows 4 (l /
// 16) .. + 3.  The four products enter one after the other, each by a fused
// multiply-add (checked on the device bit for bit), so a chain of them is the
// sum in index order.
__device__ __forceinline__ floatx4 mfma4(float a, float b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Gradient of the mean negative log-likelihood of one block of samples with
// respect to all parameters; one partial gradient and one partial loss per
// block.  A step of 4096 records is 128 blocks and 0.13 GFLOP: what bounds it
// is one block's latency.  The weights and records are loaded at once into
// LDS, and every product of the forward and backward pass and of the
// gradients runs on fp32 MFMA tiles of 16 x 16 (eight waves: 4 unit tiles x 2
// sample tiles), which take one LDS word per operand and lane where register
// tiles on the vector unit waited for LDS reads.  Per 4096 records: 194 us
// with one lane per sample and the weights read from global memory, 13.9 us
// with 2 x 4 register tiles from LDS, 10.1 us as below; the sums run in the
// same order in all three.
__global__ __launch_bounds__(TR_TB) void k_mlp_grad(const float* __restrict__ w,
                                                    const float* __restrict__ norm,
                                                    const float* __restrict__ data, TrainBatch tb,
                                                    int batch, float* __restrict__ gpart,
                                                    float* __restrict__ lpart) {
  __shared__ TrainLds T;
  const int tid = threadIdx.x, first = blockIdx.x * TR_SAMPLES;
  // records (32 x 13 values) and weights: every load issued before the first
  // is stored, so the block waits for memory once
  {
    constexpr int W4 = NH * NH / 4 / TR_TB;  // 16-byte pieces of W2 per thread
    static_assert(TR_SAMPLES * NREC <= TR_TB && NH * NOUT <= TR_TB && NIN * NH <= 2 * TR_TB, "");
    const floatx4* w2 = reinterpret_cast<const floatx4*>(w + OFF_W2);
    floatx4 c[W4];
    float c1[2], c3, cb = 0.0f;
    int i = min(tid, TR_SAMPLES * NREC - 1), t = i / NREC, k = i - t * NREC;
    float v = data[train_record(tb, first + t) * NREC + k];
    float mean = norm[min(k, NIN - 1)], inv = norm[NIN + min(k, NIN - 1)];
#pragma unroll
    for (int u = 0; u < W4; ++u) c[u] = w2[tid + u * TR_TB];
#pragma unroll
    for (int u = 0; u < 2; ++u) c1[u] = w[OFF_W1 + min(tid + u * TR_TB, NIN * NH - 1)];
    c3 = w[OFF_W3 + min(tid, NH * NOUT - 1)];
    if (tid < NH)
      cb = w[OFF_B1 + tid];
    else if (tid < 2 * NH)
      cb = w[OFF_B2 + tid - NH];
    else if (tid < 2 * NH + NOUT)
      cb = w[OFF_B3 + tid - 2 * NH];
    __builtin_amdgcn_sched_barrier(0);
    if (tid < TR_SAMPLES) {
      T.x[NIN][tid] = 1.0f;
      T.x[NIN + 1][tid] = 0.0f;
      T.dout[NOUT][tid] = T.dout[NOUT + 1][tid] = 0.0f;
    }
    if (k < NIN)
      T.x[k][t] = (v - mean) * inv;
    else
      T.y[k - NIN][t] = v;
#pragma unroll
    for (int u = 0; u < W4; ++u) {
      int j = 4 * (tid + u * TR_TB);
      *reinterpret_cast<floatx4*>(&T.w2[j / NH][j % NH]) = c[u];
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
      if (tid + u * TR_TB < NIN * NH) (&T.w1[0][0])[tid + u * TR_TB] = c1[u];
    if (tid < NH * NOUT) (&T.w3[0][0])[tid] = c3;
    if (tid < NH)
      T.b1[tid] = cb;
    else if (tid < 2 * NH)
      T.b2[tid - NH] = cb;
    else if (tid < 2 * NH + NOUT)
      T.b3[tid - 2 * NH] = cb;
  }
  __syncthreads();

  // wave: unit tile ut, sample tile st; lane: operand row or column c, K
  // element kq of a step; its results are sample sc, units ur .. ur + 3
  const int lane = tid & 63, wv = tid >> 6, c = lane & 15, kq = lane >> 4;
  const int ut = 16 * (wv & 3), st = 16 * (wv >> 2), sc = st + c, ur = ut + 4 * kq;
  // forward; d1, d2 hold silu'(z) until the backward pass scales them
  {
    floatx4 z = *reinterpret_cast<const floatx4*>(&T.b1[ur]);
#pragma unroll
    for (int k = 0; k < XROWS; k += 4) {
      float a = k + kq < NIN ? T.w1[min(k + kq, NIN - 1)][ut + c] : 0.0f;
      z = mfma4(a, T.x[k + kq][sc], z);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      T.h1[ur + i][sc] = silu(z[i]);
      T.d1[ur + i][sc] = dsilu(z[i]);
    }
  }
  __syncthreads();
  {
    floatx4 z = *reinterpret_cast<const floatx4*>(&T.b2[ur]);
#pragma unroll
    for (int k = 0; k < NH; k += 4) z = mfma4(T.w2[k + kq][ut + c], T.h1[k + kq][sc], z);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      T.h2[ur + i][sc] = silu(z[i]);
      T.d2[ur + i][sc] = dsilu(z[i]);
    }
  }
  __syncthreads();
  if ((wv & 3) == 0) {  // one wave per sample tile; rows NOUT and up are not used
    const int j = min(c, NOUT - 1);
    floatx4 z;
#pragma unroll
    for (int i = 0; i < 4; ++i) z[i] = T.b3[min(4 * kq + i, NOUT - 1)];
#pragma unroll
    for (int k = 0; k < NH; k += 4) z = mfma4(T.w3[k + kq][j], T.h2[k + kq][sc], z);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (4 * kq + i < NOUT) T.o[4 * kq + i][sc] = z[i];
  }
  __syncthreads();
  // loss sum_i [s_i + (y_i - mu_i)^2 exp(-2 s_i) / 2] and its gradient
  if (tid < TR_SAMPLES) {
    float scale = 1.0f / (float)batch, loss = 0.0f;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      float os = T.o[3 + i][tid], sv = fminf(fmaxf(os, S_MIN), S_MAX);
      float inv = expf(-sv), r = (T.y[i][tid] - T.o[i][tid]) * inv;
      loss += sv + 0.5f * r * r;
      T.dout[i][tid] = -r * inv * scale;
      bool clamped = os < S_MIN || os > S_MAX;
      T.dout[3 + i][tid] = clamped ? 0.0f : (1.0f - r * r) * scale;
    }
    T.loss[tid] = loss;
  }
  __syncthreads();
  // backward through the hidden layers
  {
    floatx4 z = {};
#pragma unroll
    for (int j = 0; j < DROWS; j += 4) {
      float a = j + kq < NOUT ? T.w3[ut + c][min(j + kq, NOUT - 1)] : 0.0f;
      z = mfma4(a, T.dout[j + kq][sc], z);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) T.d2[ur + i][sc] *= z[i];
  }
  __syncthreads();
  {
    floatx4 z = {};
#pragma unroll
    for (int j = 0; j < NH; j += 4) z = mfma4(T.w2[ut + c][j + kq], T.d2[j + kq][sc], z);
#pragma unroll
    for (int i = 0; i < 4; ++i) T.d1[ur + i][sc] *= z[i];
  }
  __syncthreads();
  // parameter gradients, sums over the block's samples: rows ut .. + 15 of W2
  // by two column tiles, and one tile each of W1 with the biases of layer 1
  // (waves 0-3), of layer 2's biases (the same waves), of W3 (waves 4-7) and,
  // wave 4, of layer 3's biases and the loss
  float* gp = gpart + (size_t)blockIdx.x * NPARAM;
  const float* xr = T.x[min(c, XROWS - 1)];
  const bool low = wv < 4;
  const float* dr = T.dout[min(c, DROWS - 1)];
  const float* lr = c == NOUT ? T.loss : dr;
  floatx4 g2[2] = {}, ga = {}, gb = {};
#pragma unroll
  for (int s = 0; s < TR_SAMPLES; s += 4) {
    float h = T.h1[ut + c][s + kq];
#pragma unroll
    for (int u = 0; u < 2; ++u) g2[u] = mfma4(h, T.d2[2 * st + 16 * u + c][s + kq], g2[u]);
    if (low) {
      float x = xr[s + kq];
      ga = mfma4(x, T.d1[ut + c][s + kq], ga);
      gb = mfma4(x, T.d2[ut + c][s + kq], gb);
    } else {
      ga = mfma4(T.h2[ut + c][s + kq], dr[s + kq], ga);
      gb = mfma4(xr[s + kq], lr[s + kq], gb);
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int u = 0; u < 2; ++u) gp[OFF_W2 + (ur + i) * NH + 2 * st + 16 * u + c] = g2[u][i];
    const int row = 4 * kq + i;
    if (low) {
      if (row < NIN) gp[OFF_W1 + row * NH + ut + c] = ga[i];
      if (row == NIN) {
        gp[OFF_B1 + ut + c] = ga[i];
        gp[OFF_B2 + ut + c] = gb[i];
      }
    } else {
      if (c < NOUT) gp[OFF_W3 + (ur + i) * NOUT + c] = ga[i];
      if (wv == 4 && row == NIN) {
        if (c < NOUT) gp[OFF_B3 + c] = gb[i];
        if (c == NOUT) lpart[blockIdx.x] = gb[i];
      }
    }
  }
}

// Sum the block gradients in order and take one Adam step, 64 parameters per
// block.  Latency again (2.7 MB for 128 blocks, written by other compute
// units): eight waves bring 128 partials of each parameter to LDS at once, and
// the first wave adds them in order.  31.6 us with one thread per parameter
// and a load waited for at a time, 8.3 us with 64 loads in flight per thread,
// 3.6 us as below.
constexpr int ADAM_P = 64, ADAM_TB = 512, ADAM_FLIGHT = 128;
__global__ __launch_bounds__(ADAM_TB) void k_mlp_adam(float* __restrict__ params,
                                                      float* __restrict__ m, float* __restrict__ v,
                                                      const float* __restrict__ gpart, int nblk,
                                                      float lr, float c1, float c2) {
  __shared__ float part[ADAM_FLIGHT][ADAM_P];
  constexpr int WAVES = ADAM_TB / 64, EACH = ADAM_FLIGHT / WAVES;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int i = blockIdx.x * ADAM_P + lane, il = min(i, NPARAM - 1);
  float mo = 0.0f, vo = 0.0f, po = 0.0f, g = 0.0f;
  if (wv == 0) {
    mo = m[il];
    vo = v[il];
    po = params[il];
  }
  for (int b0 = 0; b0 < nblk; b0 += ADAM_FLIGHT) {
    float y[EACH];
#pragma unroll
    for (int u = 0; u < EACH; ++u)
      y[u] = gpart[(size_t)min(b0 + wv * EACH + u, nblk - 1) * NPARAM + il];
    if (b0) __syncthreads();  // the previous partials are added
#pragma unroll
    for (int u = 0; u < EACH; ++u) part[wv * EACH + u][lane] = y[u];
    __syncthreads();
    if (wv == 0) {
      const int k = min(ADAM_FLIGHT, nblk - b0);
#pragma unroll 16
      for (int u = 0; u < k; ++u) g += part[u][lane];
    }
  }
  if (wv != 0 || i >= NPARAM) return;
  float mi = 0.9f * mo + 0.1f * g, vi = 0.999f * vo + 0.001f * g * g;
  m[i] = mi;
  v[i] = vi;
  params[i] = po - lr * (mi / c1) / (sqrtf(vi / c2) + 1e-8f);
}

// Sums and sums of squares of the NIN inputs over the records, in double: one
// row of 2 NIN partial sums per block
constexpr int NORM_BLOCKS = 1024;
__global__ __launch_bounds__(256) void k_mlp_norm(const float* __restrict__ data, int64_t nrec,
                                                  double* __restrict__ part) {
  __shared__ double red[4][2 * NIN];
  double s[2 * NIN] = {};
  for (int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x; r < nrec; r += (int64_t)gridDim.x * 256)
#pragma unroll
    for (int k = 0; k < NIN; ++k) {
      double x = data[(size_t)r * NREC + k];
      s[k] += x;
      s[NIN + k] += x * x;
    }
#pragma unroll
  for (int k = 0; k < 2 * NIN; ++k) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s[k] += __shfl_xor(s[k], off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][k] = s[k];
  }
  __syncthreads();
  if (threadIdx.x < 2 * NIN) {
    int k = threadIdx.x;
    part[(size_t)blockIdx.x * 2 * NIN + k] = ((red[0][k] + red[1][k]) + red[2][k]) + red[3][k];
  }
}

uint64_t splitmix(uint64_t& x) {
  uint64_t z = (x += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

unsigned short host_bf16(float f) {  // round to nearest even
  uint32_t u;
  memcpy(&u, &f, 4);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}

}  // namespace

struct lceq_mlp {
  int device;
  hipStream_t stream;
  std::vector<float> host;  // NSTATE: params, feature mean, inverse scale
  float *params, *adam_m, *adam_v, *norm, *gpart, *lpart;
  int64_t gpart_blocks, lpart_cap;  // lpart: [steps of one download][blocks]
  MlpPack* pack;
  int sites_per_wave;  // learned Higgs launch: 0 = by lattice size, 32 or 64
  float* data;  // NREC floats per record
  int64_t nrec, cap;
  int64_t adam_t;
};

#define mfail lceq::set_error
#define MHIP(call)                                                                        \
  do {                                                                                    \
    hipError_t e_ = (call);                                                               \
    if (e_ != hipSuccess) return mfail(LCEQ_ERR_HIP, "%s: %s", #call, hipGetErrorString(e_)); \
  } while (0)

static int mlp_upload(lceq_mlp* M) {
  MHIP(hipMemcpyAsync(M->params, M->host.data(), NPARAM * sizeof(float), hipMemcpyHostToDevice,
                      M->stream));
  MHIP(hipMemcpyAsync(M->norm, M->host.data() + NPARAM, 2 * NIN * sizeof(float),
                      hipMemcpyHostToDevice, M->stream));
  // inference pack
  MlpPack h;
  memset(&h, 0, sizeof(h));
  const float* w = M->host.data();
  // A operand of lane l: row (output unit) 16 nt + l % 16, K elements
  // 8 (l / 16) + j, natural for the inputs, hidden_of_k for hidden layers
  auto frag = [&](bf16x8& f, int K, int N, int off, int kb, int nt, int l, bool hidden) {
    unsigned short e[8];
    for (int j = 0; j < 8; ++j) {
      int g = l / 16, n = 16 * nt + l % 16;
      int k = hidden ? hidden_of_k(kb, g, j) : 32 * kb + 8 * g + j;
      e[j] = (k < K && n < N) ? host_bf16(w[off + k * N + n]) : (unsigned short)0;
    }
    memcpy(&f, e, 16);
  };
  for (int l = 0; l < 64; ++l) {
    for (int nt = 0; nt < 4; ++nt) {
      frag(h.w1[nt][l], NIN, NH, OFF_W1, 0, nt, l, false);
      frag(h.w2[nt][0][l], NH, NH, OFF_W2, 0, nt, l, true);
      frag(h.w2[nt][1][l], NH, NH, OFF_W2, 1, nt, l, true);
    }
    frag(h.w3[0][l], NH, NOUT, OFF_W3, 0, 0, l, true);
    frag(h.w3[1][l], NH, NOUT, OFF_W3, 1, 0, l, true);
  }
  for (int j = 0; j < NH; ++j) {
    h.b1[j] = w[OFF_B1 + j];
    h.b2[j] = w[OFF_B2 + j];
  }
  for (int j = 0; j < NOUT; ++j) h.b3[j] = w[OFF_B3 + j];
  for (int k = 0; k < NIN; ++k) {
    h.xmean[k] = w[NPARAM + k];
    h.xinv[k] = w[NPARAM + NIN + k];
  }
  MHIP(hipMemcpyAsync(M->pack, &h, sizeof(h), hipMemcpyHostToDevice, M->stream));
  MHIP(hipStreamSynchronize(M->stream));
  return LCEQ_OK;
}

extern "C" int lceq_mlp_create(uint64_t seed, lceq_mlp** out) {
  if (!out) return mfail(LCEQ_ERR_ARG, "null output");
  *out = nullptr;
  lceq_mlp* M = new lceq_mlp();
  M->host.assign(NSTATE, 0.0f);
  // Glorot-uniform weights, zero biases; a small last layer so that the
  // first proposals stay near the current configuration's scale
  uint64_t st = seed;
  auto uni = [&]() { return (double)(splitmix(st) >> 11) * 0x1.0p-53; };
  auto init = [&](int off, int fan_in, int fan_out, double gain) {
    double lim = gain * std::sqrt(6.0 / (fan_in + fan_out));
    for (int i = 0; i < fan_in * fan_out; ++i) M->host[off + i] = (float)((2.0 * uni() - 1.0) * lim);
  };
  init(OFF_W1, NIN, NH, 1.0);
  init(OFF_W2, NH, NH, 1.0);
  init(OFF_W3, NH, NOUT, 0.1);
  for (int k = 0; k < NIN; ++k) M->host[NPARAM + NIN + k] = 1.0f;  // identity normalisation
  int rc = LCEQ_OK;
  auto alloc = [&](void** p, size_t bytes) {
    if (rc) return;
    if (hipMalloc(p, bytes) != hipSuccess) rc = mfail(LCEQ_ERR_HIP, "hipMalloc(%zu) failed", bytes);
  };
  if (hipGetDevice(&M->device) != hipSuccess) rc = mfail(LCEQ_ERR_HIP, "no HIP device");
  if (!rc && hipStreamCreateWithFlags(&M->stream, hipStreamNonBlocking) != hipSuccess)
    rc = mfail(LCEQ_ERR_HIP, "hipStreamCreate failed");
  alloc((void**)&M->params, NPARAM * sizeof(float));
  alloc((void**)&M->adam_m, NPARAM * sizeof(float));
  alloc((void**)&M->adam_v, NPARAM * sizeof(float));
  alloc((void**)&M->norm, 2 * NIN * sizeof(float));
  alloc((void**)&M->pack, sizeof(MlpPack));
  if (rc) {
    lceq_mlp_destroy(M);
    return rc;
  }
  if ((rc = mlp_upload(M))) {
    lceq_mlp_destroy(M);
    return rc;
  }
  *out = M;
  return LCEQ_OK;
}

extern "C" int lceq_mlp_destroy(lceq_mlp* M) {
  if (!M) return LCEQ_OK;
  void* bufs[] = {M->params, M->adam_m, M->adam_v, M->norm, M->gpart, M->lpart, M->pack, M->data};
  for (void* b : bufs)
    if (b) (void)hipFree(b);
  if (M->stream) (void)hipStreamDestroy(M->stream);
  delete M;
  return LCEQ_OK;
}

extern "C" int lceq_mlp_get_state(lceq_mlp* M, float* state, int n) {
  if (!M || !state || n != NSTATE) return mfail(LCEQ_ERR_ARG, "state has %d floats", NSTATE);
  memcpy(state, M->host.data(), NSTATE * sizeof(float));
  return LCEQ_OK;
}

extern "C" int lceq_mlp_set_state(lceq_mlp* M, const float* state, int n) {
  if (!M || !state || n != NSTATE) return mfail(LCEQ_ERR_ARG, "state has %d floats", NSTATE);
  memcpy(M->host.data(), state, NSTATE * sizeof(float));
  M->adam_t = 0;
  MHIP(hipMemsetAsync(M->adam_m, 0, NPARAM * sizeof(float), M->stream));
  MHIP(hipMemsetAsync(M->adam_v, 0, NPARAM * sizeof(float), M->stream));
  return mlp_upload(M);
}

extern "C" int lceq_mlp_clear(lceq_mlp* M) {
  if (!M) return mfail(LCEQ_ERR_ARG, "null model");
  M->nrec = 0;
  return LCEQ_OK;
}

extern "C" int lceq_mlp_records(lceq_mlp* M, int64_t* n) {
  if (!M || !n) return mfail(LCEQ_ERR_ARG, "null argument");
  *n = M->nrec;
  return LCEQ_OK;
}

// Training pairs from the lattice's current configuration: for each parity,
// the features at the current F, then nsteps ahiggs1 Metropolis steps of
// that parity at the lattice's current step size (F does not change while
// one parity is updated), then the new a in the same frame; every stride-th
// site.  The Metropolis steps are kept (each is a valid update of the
// chain).  The Metropolis step rather than the ahiggs2 heatbath: the
// heatbath's Gaussian width beta_2 is negative in the broken phase.
const MlpPack* lceq::mlp::device_pack(const lceq_mlp* M) { return M->pack; }

float* lceq::mlp::reserve_records(lceq_mlp* M, int64_t n) {
  int64_t need = M->nrec + n;
  if (need > M->cap) {
    int64_t cap = std::max<int64_t>(need, 2 * M->cap);
    float* d = nullptr;
    hipError_t e = hipMalloc((void**)&d, (size_t)cap * NREC * sizeof(float));
    if (e != hipSuccess) {
      mfail(LCEQ_ERR_HIP, "hipMalloc(%lld records): %s", (long long)cap, hipGetErrorString(e));
      return nullptr;
    }
    if (M->data) {
      e = hipMemcpy(d, M->data, (size_t)M->nrec * NREC * sizeof(float), hipMemcpyDeviceToDevice);
      if (e == hipSuccess) e = hipFree(M->data);
      if (e != hipSuccess) {
        (void)hipFree(d);
        mfail(LCEQ_ERR_HIP, "moving the training records: %s", hipGetErrorString(e));
        return nullptr;
      }
    }
    M->data = d;
    M->cap = cap;
  }
  if (hipStreamSynchronize(M->stream) != hipSuccess) {
    mfail(LCEQ_ERR_HIP, "model stream sync failed");
    return nullptr;
  }
  return M->data + (size_t)M->nrec * NREC;
}

void lceq::mlp::commit_records(lceq_mlp* M, int64_t n) { M->nrec += n; }

void lceq::mlp::launch_record(hipStream_t stream, const Geom& g, const double* U, const double* A,
                              int eo, int stride, int nrec, double ba, double b2, double b4,
                              float* out, int target) {
  int nb = (nrec + TB - 1) / TB;
  hipLaunchKernelGGL(k_mlp_record, dim3(nb), dim3(TB), 0, stream, g, U, A, eo, stride, nrec, ba,
                     b2, b4, out, target);
}

// Training pairs from the lattice's current configuration: for each parity,
// the features at the current F, then nsteps ahiggs1 Metropolis steps of
// that parity at the lattice's current step size (F does not change while
// one parity is updated), then the new a in the same frame; every stride-th
// site.  The Metropolis steps are kept (each is a valid update of the
// chain).  The Metropolis step rather than the ahiggs2 heatbath: the
// heatbath's Gaussian width beta_2 is negative in the broken phase.
extern "C" int lceq_mlp_collect(lceq_lattice* L, lceq_mlp* M, int nsteps, int stride) {
  if (!L || !M) return mfail(LCEQ_ERR_ARG, "null argument");
  if (nsteps < 1 || stride < 1) return mfail(LCEQ_ERR_ARG, "nsteps and stride must be >= 1");
  if (L->rng_mode != LCEQ_RNG_PHILOX) return mfail(LCEQ_ERR_ARG, "collect needs Philox streams");
  int nrec = (L->g.n + stride - 1) / stride;
  float* base = reserve_records(M, 2 * (int64_t)nrec);
  if (!base) return LCEQ_ERR_HIP;
  for (int eo = 0; eo < 2; ++eo) {
    float* out = base + (size_t)eo * nrec * NREC;
    launch_record(L->stream, L->g, L->U, L->A, eo, stride, nrec, L->beta_a, L->beta_2, L->beta_4,
                  out, 0);
    for (int h = 0; h < nsteps; ++h) launch_higgs(L, 1, eo, 0, nullptr, next_pass(L), 0);
    launch_record(L->stream, L->g, L->U, L->A, eo, stride, nrec, L->beta_a, L->beta_2, L->beta_4,
                  out, 1);
  }
  int rc = check_launch();
  if (rc) return rc;
  MHIP(hipStreamSynchronize(L->stream));
  commit_records(M, 2 * (int64_t)nrec);
  return LCEQ_OK;
}

// Feature normalisation from the collected records (mean, 1/std; constant
// features get scale 1): the sums on the device, where the records are
static int mlp_fit_norm(lceq_mlp* M) {
  int nb = (int)std::min<int64_t>(NORM_BLOCKS, (M->nrec + 255) / 256);
  double* part = nullptr;
  std::vector<double> h((size_t)nb * 2 * NIN);
  MHIP(hipMalloc((void**)&part, h.size() * sizeof(double)));
  hipLaunchKernelGGL(k_mlp_norm, dim3(nb), dim3(256), 0, M->stream, M->data, M->nrec, part);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess)
    e = hipMemcpyAsync(h.data(), part, h.size() * sizeof(double), hipMemcpyDeviceToHost, M->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(M->stream);
  (void)hipFree(part);
  if (e != hipSuccess)
    return mfail(LCEQ_ERR_HIP, "summing the training records: %s", hipGetErrorString(e));
  for (int k = 0; k < NIN; ++k) {
    double s = 0.0, s2 = 0.0;
    for (int b = 0; b < nb; ++b) {
      s += h[(size_t)b * 2 * NIN + k];
      s2 += h[(size_t)b * 2 * NIN + NIN + k];
    }
    double mean = s / (double)M->nrec, var = s2 / (double)M->nrec - mean * mean;
    double sd = var > 1e-12 ? std::sqrt(var) : 0.0;
    M->host[NPARAM + k] = (float)mean;
    M->host[NPARAM + NIN + k] = sd > 1e-6 ? (float)(1.0 / sd) : 1.0f;
  }
  return LCEQ_OK;
}

// Adam on the collected records: `steps` mini-batches of `batch` records,
// each batch a stretch of a seeded affine permutation of the records.
// loss (optional, steps values) receives the mean negative log-likelihood
// per step (up to the constant 3/2 log 2 pi).  The steps are queued without
// waiting: the kernels form the record indices themselves, and the blocks'
// losses are downloaded LOSS_STEPS steps at a time.
constexpr int LOSS_STEPS = 512;

extern "C" int lceq_mlp_train(lceq_mlp* M, int steps, int batch, double lr, uint64_t seed,
                              int fit_norm, double* loss) {
  if (!M || steps < 0 || batch < TR_SAMPLES || batch % TR_SAMPLES)
    return mfail(LCEQ_ERR_ARG, "batch must be a positive multiple of %d", TR_SAMPLES);
  if (M->nrec < batch) return mfail(LCEQ_ERR_ARG, "only %lld records", (long long)M->nrec);
  if (M->nrec > (int64_t)UINT32_MAX)  // the permutation's products are 64-bit
    return mfail(LCEQ_ERR_ARG, "%lld records are more than 2^32 - 1", (long long)M->nrec);
  int rc;
  if (fit_norm) {
    if ((rc = mlp_fit_norm(M))) return rc;
    if ((rc = mlp_upload(M))) return rc;
  }
  const int nblk = batch / TR_SAMPLES;
  const int rows = loss ? std::max(1, std::min(steps, LOSS_STEPS)) : 1;
  if (nblk > M->gpart_blocks) {
    if (M->gpart) MHIP(hipFree(M->gpart));
    M->gpart = nullptr;
    M->gpart_blocks = 0;
    MHIP(hipMalloc((void**)&M->gpart, (size_t)nblk * NPARAM * sizeof(float)));
    M->gpart_blocks = nblk;
  }
  if ((int64_t)rows * nblk > M->lpart_cap) {
    if (M->lpart) MHIP(hipFree(M->lpart));
    M->lpart = nullptr;
    M->lpart_cap = 0;
    MHIP(hipMalloc((void**)&M->lpart, (size_t)rows * nblk * sizeof(float)));
    M->lpart_cap = (int64_t)rows * nblk;
  }
  if (M->adam_t == 0) {
    MHIP(hipMemsetAsync(M->adam_m, 0, NPARAM * sizeof(float), M->stream));
    MHIP(hipMemsetAsync(M->adam_v, 0, NPARAM * sizeof(float), M->stream));
  }
  const int64_t N = M->nrec;
  uint64_t st = seed;
  int64_t mult = 1, offs = 0, pos = N;
  std::vector<float> lp(loss ? (size_t)rows * nblk : 0);
  for (int it = 0; it < steps; ++it) {
    if (pos + batch > N) {  // new epoch: a fresh affine permutation i -> (mult i + offs) mod N
      do {
        mult = (int64_t)(splitmix(st) % (uint64_t)N) | 1;
      } while (std::gcd(mult, N) != 1);
      offs = (int64_t)(splitmix(st) % (uint64_t)N);
      pos = 0;
    }
    TrainBatch tb{(uint64_t)(mult % N), ((uint64_t)mult * (uint64_t)pos % (uint64_t)N + offs) % N,
                  (uint64_t)N, 1.0 / (double)N};
    pos += batch;
    const int row = it % rows;
    hipLaunchKernelGGL(k_mlp_grad, dim3(nblk), dim3(TR_TB), 0, M->stream, M->params, M->norm,
                       M->data, tb, batch, M->gpart, M->lpart + (size_t)row * nblk);
    ++M->adam_t;
    float c1 = 1.0f - std::pow(0.9f, (float)M->adam_t), c2 = 1.0f - std::pow(0.999f, (float)M->adam_t);
    hipLaunchKernelGGL(k_mlp_adam, dim3((NPARAM + ADAM_P - 1) / ADAM_P), dim3(ADAM_TB), 0,
                       M->stream, M->params, M->adam_m, M->adam_v, M->gpart, nblk, (float)lr, c1,
                       c2);
    if ((rc = check_launch())) return rc;
    if (loss && (row == rows - 1 || it == steps - 1)) {
      MHIP(hipMemcpyAsync(lp.data(), M->lpart, (size_t)(row + 1) * nblk * sizeof(float),
                          hipMemcpyDeviceToHost, M->stream));
      MHIP(hipStreamSynchronize(M->stream));
      for (int r = 0; r <= row; ++r) {
        double l = 0.0;
        for (int b = 0; b < nblk; ++b) l += lp[(size_t)r * nblk + b];
        loss[it - row + r] = l / batch;
      }
    }
  }
  MHIP(hipMemcpyAsync(M->host.data(), M->params, NPARAM * sizeof(float), hipMemcpyDeviceToHost,
                      M->stream));
  MHIP(hipStreamSynchronize(M->stream));
  return mlp_upload(M);
}

extern "C" int lceq_mlp_set_sites_per_wave(lceq_mlp* M, int sites) {
  if (!M) return mfail(LCEQ_ERR_ARG, "null argument");
  if (sites != 0 && sites != 32 && sites != 64)
    return mfail(LCEQ_ERR_ARG, "sites per wave must be 0 (by lattice size), 32 or 64, not %d",
                 sites);
  M->sites_per_wave = sites;
  return LCEQ_OK;
}

extern "C" int lceq_mlp_eval(lceq_mlp* M, const float* x, int n, float* y) {
  if (!M || n < 1 || !x || !y) return mfail(LCEQ_ERR_ARG, "bad arguments");
  float *dx = nullptr, *dy = nullptr;
  MHIP(hipMalloc((void**)&dx, (size_t)n * NIN * sizeof(float)));
  if (hipMalloc((void**)&dy, (size_t)n * NOUT * sizeof(float)) != hipSuccess) {
    (void)hipFree(dx);
    return mfail(LCEQ_ERR_HIP, "hipMalloc failed");
  }
  int rc = LCEQ_OK;
  if (hipMemcpyAsync(dx, x, (size_t)n * NIN * sizeof(float), hipMemcpyHostToDevice, M->stream) !=
      hipSuccess)
    rc = mfail(LCEQ_ERR_HIP, "copy failed");
  if (!rc) {
    hipLaunchKernelGGL(k_mlp_eval, dim3((n + TB - 1) / TB), dim3(TB), 0, M->stream, M->pack, dx, dy,
                       n);
    rc = check_launch();
  }
  if (!rc && (hipMemcpyAsync(y, dy, (size_t)n * NOUT * sizeof(float), hipMemcpyDeviceToHost,
                             M->stream) != hipSuccess ||
              hipStreamSynchronize(M->stream) != hipSuccess))
    rc = mfail(LCEQ_ERR_HIP, "copy failed");
  (void)hipFree(dx);
  (void)hipFree(dy);
  return rc;
}

// both parities with the learned proposal; partials (always measured) in the
// Higgs slots
// Sites per wave of the learned Higgs launch: 64 (four MFMA column tiles,
// the default) or 32 (two tiles, half the lanes idle in the per-site FP64
// work).  32 shortens one wave's network evaluations but not its FP64
// chain; at 48^3 (fewer waves than SIMDs) it measured 15.6 us per parity
// against 13.8 us for 64.  The fields do not depend on the choice.
static int mlp_sites_per_wave(const lceq_lattice*, const lceq_mlp* M) {
  return M->sites_per_wave ? M->sites_per_wave : 64;
}
static int mlp_blocks(const lceq_lattice* L, const lceq_mlp* M) {
  int per_block = (TB / 64) * mlp_sites_per_wave(L, M);
  return (L->g.n + per_block - 1) / per_block;
}

static int mlp_higgs_sweep(lceq_lattice* L, lceq_mlp* M) {
  if (L->rng_mode != LCEQ_RNG_PHILOX) return mfail(LCEQ_ERR_ARG, "the learned proposal draws Philox");
  MlpArgs a;
  a.g = L->g;
  a.U = L->U;
  a.A = L->A;
  a.beta_a = L->beta_a;
  a.beta_2 = L->beta_2;
  a.beta_4 = L->beta_4;
  a.key = Philox{(uint32_t)L->seed, (uint32_t)(L->seed >> 32)};
  a.pack = M->pack;
  a.pstride = L->pstride;
  int spw = mlp_sites_per_wave(L, M);
  a.nb = mlp_blocks(L, M);
  prof_begin(L, KC_HIGGS);
  for (int eo = 0; eo < 2; ++eo) {
    a.eo = eo;
    a.pass = next_pass(L);
    a.part = L->partials + (size_t)(6 + eo) * LCEQ_NQ * L->pstride;
    prof_count(L, KC_HIGGS);
    if (spw == 32)
      hipLaunchKernelGGL(k_higgs_mlp<2>, dim3(a.nb), dim3(TB), 0, L->stream, a);
    else
      hipLaunchKernelGGL(k_higgs_mlp<4>, dim3(a.nb), dim3(TB), 0, L->stream, a);
  }
  prof_end(L, KC_HIGGS);
  return check_launch();
}

extern "C" int lceq_higgs_mlp(lceq_lattice* L, lceq_mlp* M, double* accept) {
  if (!L || !M) return mfail(LCEQ_ERR_ARG, "null argument");
  int rc = mlp_higgs_sweep(L, M);
  if (rc) return rc;
  launch_finalize(L, 0, 0, 2, 1, nullptr, accept != nullptr, mlp_blocks(L, M));
  if (accept) {
    if ((rc = finish_obs(L))) return rc;
    *accept = L->pin[OBS_ACC_HIGGS];
  }
  return LCEQ_OK;
}

// nsweep sweeps of 1 KP + n_or overrelaxation link sweeps + the learned
// Higgs update; with measflag one history row per sweep (as lceq_sweep)
extern "C" int lceq_sweep_mlp(lceq_lattice* L, lceq_mlp* M, int nsweep, int n_or, int measflag) {
  if (!L || !M) return mfail(LCEQ_ERR_ARG, "null argument");
  if (nsweep < 0 || n_or < 0) return mfail(LCEQ_ERR_ARG, "nsweep, n_or must be >= 0");
  if (measflag && L->hist_rows + nsweep > L->hist_cap)
    return mfail(LCEQ_ERR_ARG, "history full (%d rows); call lceq_history", L->hist_cap);
  int rc;
  for (int it = 0; it < nsweep; ++it) {
    double* row = measflag ? L->hist + (size_t)(L->hist_rows++) * LCEQ_OBS_N : nullptr;
    int meas_kp = measflag && n_or == 0;
    if ((rc = link_sweep(L, 1, meas_kp, 1, meas_kp))) return rc;
    for (int k = 0; k < n_or; ++k) {
      int m = measflag && k == n_or - 1;
      if ((rc = link_sweep(L, 0, m, 1, m))) return rc;
    }
    if ((rc = mlp_higgs_sweep(L, M))) return rc;
    launch_finalize(L, measflag ? (n_or ? 2 : 1) : 0, measflag, 2, 1, row, false,
                    mlp_blocks(L, M));
  }
  return check_launch();
}
