// mlp.hip -- the surrogate network of the warm start: a small MLP trained
// and evaluated on the GPU with hand-written MFMA kernels.
//
// Layers: n_in inputs (zero-padded to 32) -> n_hidden layers of `width` GELU
// units -> n_out linear outputs.  Weights live as FP32 masters (Adam
// updates them) with BF16 copies the matrix kernels read, row-major and
// transposed; products accumulate in FP32 (v_mfma_f32_32x32x16_bf16).
// Activations feeding a product are stored in BF16, pre-activations in FP32.
// Batches are padded to a multiple of 32 rows; padded rows carry zero loss
// and zero gradient.
//
// Every operand of a product is stored with the contracted index contiguous,
// so that a lane's eight values of it are one 16-byte load and no product
// needs an LDS transpose: a product's results lie in registers as four
// consecutive rows of one column per lane, so writing the transposed copy the
// weight gradients contract over is an 8-byte store.  Element-wise work
// (bias, GELU, its derivative, the loss, the bias sums, Adam) is done on those
// registers, where a kernel of its own would be one more pass over memory and
// one more launch.  A training step is n_hidden + 1 forward, n_hidden
// backward and one weight-gradient launch; at batch 2048, width 256 and three
// hidden layers a step is bounded by the latency of those eight dependent
// launches (a product reads 2 MB from L2): twenty steps with the copies of
// inputs, targets and weights take 1.76 ms.  Separate kernels with scalar
// loads, a one-workgroup loss and serial column sums took 68.8 ms.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <string.h>

#include <vector>

#include "dfargo_internal.h"

#define IN_PAD 32 // the input layer's K, padded to a whole output tile of dW

#define MCHK(call)                                                                                       \
  do {                                                                                                   \
    hipError_t e_ = (call);                                                                              \
    if (e_ != hipSuccess)                                                                                \
      return dfargo_set_error(DFARGO_ERR_HIP, "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_),     \
                              __FILE__, __LINE__);                                                       \
  } while (0)

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef uint16_t bf16;

#define MLP_MAX_LAYERS 17
#define DW_WAVES 16 // wavefronts that share the contraction of a weight-gradient tile

__device__ __forceinline__ bf16 to_bf16(float f) { // round to nearest even
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (bf16)(u >> 16);
}

__device__ __forceinline__ float gelu(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_grad(float z) {
  const float cdf = 0.5f * (1.0f + erff(z * 0.70710678118654752f));
  const float pdf = 0.39894228040143268f * expf(-0.5f * z * z);
  return cdf + z * pdf;
}

// One wavefront's 32x32 tile sum_k A(m, k) B(n, k), both operands with k
// contiguous, over `steps` blocks of 16 values of k that lie `stride` values
// apart.  Operand layout of the 32x32x16 instruction: lane l holds
// A(l % 32, 8 (l / 32) + v) and B(l % 32, 8 (l / 32) + v), v < 8; its 16 results
// are C(tile_row(v, l), l % 32).  Eight steps' loads are issued before their
// products, so a tile waits for memory once per 128 values of k.
__device__ __forceinline__ int tile_row(int v, int lane) { return 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3); }
template <int U>
__device__ __forceinline__ void tile_steps(const bf16 *&a, const bf16 *&b, long stride, floatx16 &acc) {
  bf16x8 x[U], y[U];
#pragma unroll
  for (int u = 0; u < U; u++) {
    x[u] = *(const bf16x8 *)(a + u * stride);
    y[u] = *(const bf16x8 *)(b + u * stride);
  }
#pragma unroll
  for (int u = 0; u < U; u++) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[u], y[u], acc, 0, 0, 0);
  a += U * stride;
  b += U * stride;
}
__device__ __forceinline__ floatx16 tile_product(const bf16 *a, const bf16 *b, int steps, long stride) {
  floatx16 acc;
#pragma unroll
  for (int v = 0; v < 16; v++) acc[v] = 0.0f;
  int s = 0;
  for (; s + 8 <= steps; s += 8) tile_steps<8>(a, b, stride, acc);
  for (; s + 2 <= steps; s += 2) tile_steps<2>(a, b, stride, acc);
  if (s < steps) tile_steps<1>(a, b, stride, acc);
  return acc;
}

// the tile's 16 values of this lane in BF16: rows of out (leading dimension
// ldo) and columns of its transpose (leading dimension ldt)
__device__ __forceinline__ void store_both(const float (&x)[16], bf16 *out, long ldo, bf16 *outT, long ldt, int m0,
                                           int n, int lane) {
#pragma unroll
  for (int g = 0; g < 4; g++) {
    ushort4 q;
    bf16 *e = (bf16 *)&q;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      e[k] = to_bf16(x[4 * g + k]);
      out[(long)(m0 + tile_row(4 * g + k, lane)) * ldo + n] = e[k];
    }
    *(ushort4 *)(outT + (long)n * ldt + m0 + tile_row(4 * g, lane)) = q;
  }
}
// sum over the tile's 32 rows of each column, in FP32, into part[n]
__device__ __forceinline__ void column_sums(const float (&x)[16], float *part, int n, int lane) {
  float s = 0.0f;
#pragma unroll
  for (int v = 0; v < 16; v++) s += x[v];
  s += __shfl_xor(s, 32, 64);
  if (lane < 32) part[n] = s;
}

// Forward product of a layer, one wavefront per 32x32 tile of its outputs.
// HIDDEN: h = GELU(z) in BF16 (row-major and transposed), z kept for the
// backward pass.  OUTPUT: z only.  LOSS: the output layer under training --
// d = z - t gives the tile's sum of squares and dZ = scale d; padded rows
// give 0.
enum { FWD_HIDDEN, FWD_OUTPUT, FWD_LOSS };
template <int MODE>
__global__ void __launch_bounds__(64) k_forward(const bf16 *__restrict__ in, const bf16 *__restrict__ wT,
                                                const float *__restrict__ bias, int K, int N, int rows, float *z,
                                                bf16 *out, bf16 *outT, const float *__restrict__ t, int batch,
                                                float scale, float *col_part, float *loss_part) {
  const int lane = threadIdx.x, m0 = blockIdx.y * 32, n0 = blockIdx.x * 32, n = n0 + (lane & 31);
  const int k0 = 8 * (lane >> 5);
  const floatx16 acc =
      tile_product(in + (long)(m0 + (lane & 31)) * K + k0, wT + (long)n * K + k0, K / 16, 16);
  const float b = bias[n];
  float x[16];
  float loss = 0.0f;
#pragma unroll
  for (int v = 0; v < 16; v++) {
    const int row = m0 + tile_row(v, lane);
    const float zz = acc[v] + b;
    if (MODE != FWD_LOSS) z[(long)row * N + n] = zz;
    if (MODE == FWD_HIDDEN) x[v] = gelu(zz);
    if (MODE == FWD_LOSS) {
      const float d = row < batch ? zz - t[(long)row * N + n] : 0.0f;
      loss += d * d;
      x[v] = d * scale;
    }
  }
  if (MODE != FWD_OUTPUT) store_both(x, out, N, outT, rows, m0, n, lane);
  if (MODE == FWD_LOSS) {
    column_sums(x, col_part + (long)blockIdx.y * N, n, lane);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) loss += __shfl_xor(loss, off, 64);
    if (lane == 0) loss_part[blockIdx.y * gridDim.x + blockIdx.x] = loss;
  }
}

// dZ of the layer below, (dZ W^T) GELU'(z), with its column sums per 32 rows
__global__ void __launch_bounds__(64) k_backward(const bf16 *__restrict__ dz, const bf16 *__restrict__ w, int K, int N,
                                                 int rows, const float *__restrict__ z, bf16 *out, bf16 *outT,
                                                 float *col_part) {
  const int lane = threadIdx.x, m0 = blockIdx.y * 32, n0 = blockIdx.x * 32, n = n0 + (lane & 31);
  const int k0 = 8 * (lane >> 5);
  const floatx16 acc = tile_product(dz + (long)(m0 + (lane & 31)) * K + k0, w + (long)n * K + k0, K / 16, 16);
  float x[16];
#pragma unroll
  for (int v = 0; v < 16; v++) x[v] = acc[v] * gelu_grad(z[(long)(m0 + tile_row(v, lane)) * N + n]);
  store_both(x, out, N, outT, rows, m0, n, lane);
  column_sums(x, col_part + (long)blockIdx.y * N, n, lane);
}

// Weight and bias gradients of every layer, dW = in^T dZ contracted over the
// rows, db the sums of dZ's columns; with `train` Adam on the FP32 masters
// and the refreshed BF16 copies, else the gradients themselves.  One
// workgroup per 32x32 tile of a dW: a tile alone on a wavefront would walk
// all rows in sequence (128 steps at 2048 rows) with 200 wavefronts on 256
// CUs, so the tile's wavefronts take every DW_WAVES-th block of 16 rows and
// their partial tiles are summed through LDS in wavefront order.
struct LayerGrad {
  int k, n, tile0;                       // inputs x outputs, first tile
  const bf16 *inT, *dzT;                 // [k][rows], [n][rows]
  const float *col_part;                 // [rows / 32][n]
  float *w, *b, *gw, *gb, *mw, *vw, *mb, *vb;
  bf16 *wb, *wT;
};
struct GradArgs {
  int nl, rows, train;
  float lr, b1, b2, eps, c1, c2;
  LayerGrad l[MLP_MAX_LAYERS];
};
__device__ __forceinline__ float adam(const GradArgs &a, float *w, float *m, float *v, long i, float g) {
  const float mi = a.b1 * m[i] + (1.0f - a.b1) * g, vi = a.b2 * v[i] + (1.0f - a.b2) * g * g;
  m[i] = mi;
  v[i] = vi;
  const float wi = w[i] - a.lr * (mi / a.c1) / (sqrtf(vi / a.c2) + a.eps);
  w[i] = wi;
  return wi;
}
__global__ void __launch_bounds__(64 * DW_WAVES) k_weights(GradArgs a) {
  __shared__ float sh[DW_WAVES][1024];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int q = 0;
  while (q + 1 < a.nl && (int)blockIdx.x >= a.l[q + 1].tile0) q++;
  const LayerGrad &y = a.l[q];
  const int tile = blockIdx.x - y.tile0, tn = y.n / 32, m0 = (tile / tn) * 32, n0 = (tile % tn) * 32;
  const int steps = a.rows / 16, k0 = 16 * wave + 8 * (lane >> 5);
  const int mine = wave < steps ? (steps - wave + DW_WAVES - 1) / DW_WAVES : 0;
  const floatx16 acc = tile_product(y.inT + (long)(m0 + (lane & 31)) * a.rows + k0,
                                    y.dzT + (long)(n0 + (lane & 31)) * a.rows + k0, mine, 16 * DW_WAVES);
#pragma unroll
  for (int v = 0; v < 16; v++) sh[wave][v * 64 + lane] = acc[v];
  __syncthreads();
  float g = 0.0f;
#pragma unroll
  for (int w = 0; w < DW_WAVES; w++) g += sh[w][tid];
  const int m = m0 + tile_row(wave, lane), n = n0 + (lane & 31); // tid = 64 v + lane
  const long i = (long)m * y.n + n;
  if (a.train) {
    const bf16 r = to_bf16(adam(a, y.w, y.mw, y.vw, i, g));
    y.wb[i] = r;
    y.wT[(long)n * y.k + m] = r;
  } else {
    y.gw[i] = g;
  }
  if (m0 != 0) return; // the whole workgroup
  // the bias gradients of the tile's columns: 32 threads per column
  const int c = tid & 31, grp = tid >> 5;
  float s = 0.0f;
  for (int r = grp; r < a.rows / 32; r += 32) s += y.col_part[(long)r * y.n + n0 + c];
  __syncthreads();
  sh[0][tid] = s;
  __syncthreads();
  if (tid < 32) {
    float db = 0.0f;
    for (int k = 0; k < 32; k++) db += sh[0][k * 32 + tid];
    if (a.train) adam(a, y.b, y.mb, y.vb, n0 + tid, db);
    else y.gb[n0 + tid] = db;
  }
}

// the padded input rows: x (batch x n_in, FP32) into X (rows x IN_PAD, BF16)
// and its transpose
__global__ void k_input(const float *x, bf16 *X, bf16 *XT, int batch, int n_in, int rows) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows * IN_PAD) return;
  const int r = i / IN_PAD, c = i % IN_PAD;
  const bf16 v = (r < batch && c < n_in) ? to_bf16(x[r * n_in + c]) : (bf16)0;
  X[i] = v;
  XT[(long)c * rows + r] = v;
}
// the loss from the tiles' sums of squares, a fixed-order tree
__global__ void __launch_bounds__(256) k_loss(const float *part, int n, float count, float *loss) {
  __shared__ float sh[256];
  const int tid = threadIdx.x;
  float s = 0.0f;
  for (int i = tid; i < n; i += 256) s += part[i];
  sh[tid] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (tid < w) sh[tid] += sh[tid + w];
    __syncthreads();
  }
  if (tid == 0) *loss = sh[0] / count;
}
__global__ void k_weights_bf16(const float *w, bf16 *wb, bf16 *wT, int k, int n) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)k * n) return;
  const bf16 r = to_bf16(w[i]);
  wb[i] = r;
  wT[(i % n) * k + i / n] = r;
}

// ------------------------------------------------------------------------

struct Layer {
  int k, n;          // inputs (padded) x outputs
  float *w, *b;      // FP32 masters: w[k][n] (padded rows zero), b[n]
  bf16 *wb, *wT;     // BF16 copies of w: [k][n], [n][k]
  float *gw, *gb;    // gradients
  float *mw, *vw, *mb, *vb;
  float *z;          // pre-activation (rows x n)
  bf16 *h, *hT;      // activation, [rows][n] and [n][rows]
  bf16 *dz, *dzT;    // gradient of z, [rows][n] and [n][rows]
  float *col_part;   // column sums of dz per 32 rows
};

struct dfargo_mlp {
  int n_in, width, n_hidden, n_out, max_rows, dev;
  long step = 0;
  hipStream_t stream = nullptr;
  std::vector<Layer> L;
  bf16 *X = nullptr, *XT = nullptr;
  float *x_in = nullptr, *t_in = nullptr, *loss = nullptr, *loss_part = nullptr;
  std::vector<void *> allocs;
};

static int malloc_zero(dfargo_mlp *m, void **p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipSuccess) return dfargo_set_error(DFARGO_ERR_ALLOC, "hipMalloc(%zu): %s", bytes, hipGetErrorString(e));
  m->allocs.push_back(*p);
  MCHK(hipMemset(*p, 0, bytes));
  return DFARGO_OK;
}

static unsigned long long splitmix(unsigned long long *s) {
  unsigned long long z = (*s += 0x9E3779B97F4A7C15ULL);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
  return z ^ (z >> 31);
}

extern "C" int dfargo_mlp_destroy(dfargo_mlp *m) {
  if (!m) return DFARGO_OK;
  hipSetDevice(m->dev);
  if (m->stream) hipStreamSynchronize(m->stream);
  for (void *p : m->allocs) hipFree(p);
  if (m->stream) hipStreamDestroy(m->stream);
  delete m;
  return DFARGO_OK;
}

extern "C" size_t dfargo_mlp_param_count(const dfargo_mlp *m) {
  if (!m) return 0;
  size_t n = 0;
  for (size_t l = 0; l < m->L.size(); l++) {
    const int kin = l == 0 ? m->n_in : m->L[l].k;
    n += (size_t)kin * m->L[l].n + m->L[l].n;
  }
  return n;
}

extern "C" int dfargo_mlp_create(int n_in, int width, int n_hidden, int n_out, int max_batch, unsigned long seed,
                                 int device, dfargo_mlp **out) {
  if (!out) return dfargo_set_error(DFARGO_ERR_ARG, "null output");
  *out = nullptr;
  if (n_in < 1 || n_in > IN_PAD || width < 32 || width % 32 || n_out < 32 || n_out % 32 || n_hidden < 1 ||
      n_hidden > 16 || max_batch < 1 || max_batch > 65536)
    return dfargo_set_error(DFARGO_ERR_ARG, "need 1 <= n_in <= 32, width and n_out multiples of 32, "
                                            "1 <= n_hidden <= 16, 1 <= max_batch <= 65536");
  MCHK(hipSetDevice(device));
  dfargo_mlp *m = new dfargo_mlp();
  m->n_in = n_in;
  m->width = width;
  m->n_hidden = n_hidden;
  m->n_out = n_out;
  m->max_rows = (max_batch + 31) / 32 * 32;
  m->dev = device;
  int rc = DFARGO_OK;
  if (hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) != hipSuccess) {
    delete m;
    return dfargo_set_error(DFARGO_ERR_HIP, "hipStreamCreate failed");
  }
  const size_t R = m->max_rows;
  unsigned long long st = seed;
  for (int l = 0; l <= n_hidden && !rc; l++) {
    Layer y;
    memset(&y, 0, sizeof y);
    y.k = l == 0 ? IN_PAD : width;
    y.n = l == n_hidden ? n_out : width;
    const size_t nw = (size_t)y.k * y.n;
    if ((rc = malloc_zero(m, (void **)&y.w, 4 * nw)) || (rc = malloc_zero(m, (void **)&y.b, 4 * y.n)) ||
        (rc = malloc_zero(m, (void **)&y.wb, 2 * nw)) || (rc = malloc_zero(m, (void **)&y.wT, 2 * nw)) ||
        (rc = malloc_zero(m, (void **)&y.gw, 4 * nw)) || (rc = malloc_zero(m, (void **)&y.gb, 4 * y.n)) ||
        (rc = malloc_zero(m, (void **)&y.mw, 4 * nw)) || (rc = malloc_zero(m, (void **)&y.vw, 4 * nw)) ||
        (rc = malloc_zero(m, (void **)&y.mb, 4 * y.n)) || (rc = malloc_zero(m, (void **)&y.vb, 4 * y.n)) ||
        (rc = malloc_zero(m, (void **)&y.z, 4 * R * y.n)) || (rc = malloc_zero(m, (void **)&y.h, 2 * R * y.n)) ||
        (rc = malloc_zero(m, (void **)&y.hT, 2 * R * y.n)) || (rc = malloc_zero(m, (void **)&y.dz, 2 * R * y.n)) ||
        (rc = malloc_zero(m, (void **)&y.dzT, 2 * R * y.n)) ||
        (rc = malloc_zero(m, (void **)&y.col_part, 4 * R / 32 * y.n)))
      break;
    // Glorot-uniform weights over the real inputs, zero biases
    const int kin = l == 0 ? n_in : y.k;
    const double lim = sqrt(6.0 / (double)(kin + y.n));
    std::vector<float> w(nw, 0.0f);
    for (int i = 0; i < kin; i++)
      for (int j = 0; j < y.n; j++)
        w[(size_t)i * y.n + j] = (float)(lim * (2.0 * (double)(splitmix(&st) >> 11) / 9007199254740992.0 - 1.0));
    if (hipMemcpy(y.w, w.data(), 4 * nw, hipMemcpyHostToDevice) != hipSuccess) {
      rc = dfargo_set_error(DFARGO_ERR_HIP, "weight upload failed");
      break;
    }
    hipLaunchKernelGGL(k_weights_bf16, dim3((nw + 255) / 256), dim3(256), 0, m->stream, y.w, y.wb, y.wT, y.k, y.n);
    m->L.push_back(y);
  }
  if (!rc && !(rc = malloc_zero(m, (void **)&m->X, 2 * R * IN_PAD)) &&
      !(rc = malloc_zero(m, (void **)&m->XT, 2 * R * IN_PAD)) &&
      !(rc = malloc_zero(m, (void **)&m->loss_part, 4 * (R / 32) * (n_out / 32))) &&
      !(rc = malloc_zero(m, (void **)&m->x_in, 4 * R * n_in)) && !(rc = malloc_zero(m, (void **)&m->t_in, 4 * R * n_out)))
    rc = malloc_zero(m, (void **)&m->loss, 4);
  if (!rc && hipStreamSynchronize(m->stream) != hipSuccess)
    rc = dfargo_set_error(DFARGO_ERR_HIP, "initialisation failed");
  if (rc) {
    dfargo_mlp_destroy(m);
    return rc;
  }
  *out = m;
  return DFARGO_OK;
}

// forward pass over `rows` padded rows (m->X filled); with loss_batch > 0
// the output layer forms the loss's partial sums and its gradient against the
// targets of the first loss_batch rows instead of the outputs
static int forward(dfargo_mlp *m, int rows, int loss_batch) {
  const bf16 *in = m->X;
  for (size_t l = 0; l < m->L.size(); l++) {
    Layer &y = m->L[l];
    const dim3 g(y.n / 32, rows / 32), b(64);
    const float scale = 2.0f / (float)((loss_batch > 0 ? loss_batch : 1) * m->n_out);
    if (l + 1 < m->L.size())
      hipLaunchKernelGGL(k_forward<FWD_HIDDEN>, g, b, 0, m->stream, in, y.wT, y.b, y.k, y.n, rows, y.z, y.h, y.hT,
                         (const float *)nullptr, 0, 0.0f, (float *)nullptr, (float *)nullptr);
    else if (loss_batch > 0)
      hipLaunchKernelGGL(k_forward<FWD_LOSS>, g, b, 0, m->stream, in, y.wT, y.b, y.k, y.n, rows, (float *)nullptr,
                         y.dz, y.dzT, m->t_in, loss_batch, scale, y.col_part, m->loss_part);
    else
      hipLaunchKernelGGL(k_forward<FWD_OUTPUT>, g, b, 0, m->stream, in, y.wT, y.b, y.k, y.n, rows, y.z,
                         (bf16 *)nullptr, (bf16 *)nullptr, (const float *)nullptr, 0, 0.0f, (float *)nullptr,
                         (float *)nullptr);
    in = y.h;
  }
  MCHK(hipGetLastError());
  return DFARGO_OK;
}

// the loss the last forward pass with targets left, into m->loss
static int form_loss(dfargo_mlp *m, int batch, int rows) {
  hipLaunchKernelGGL(k_loss, dim3(1), dim3(256), 0, m->stream, m->loss_part, (rows / 32) * (m->n_out / 32),
                     (float)(batch * m->n_out), m->loss);
  MCHK(hipGetLastError());
  return DFARGO_OK;
}

static int load_inputs(dfargo_mlp *m, int batch, const float *x, int *rows) {
  if (batch < 1 || batch > m->max_rows) return dfargo_set_error(DFARGO_ERR_ARG, "batch %d outside [1, %d]", batch, m->max_rows);
  *rows = (batch + 31) / 32 * 32;
  MCHK(hipMemcpyAsync(m->x_in, x, 4 * (size_t)batch * m->n_in, hipMemcpyHostToDevice, m->stream));
  const int n = *rows * IN_PAD;
  hipLaunchKernelGGL(k_input, dim3((n + 255) / 256), dim3(256), 0, m->stream, m->x_in, m->X, m->XT, batch, m->n_in,
                     *rows);
  MCHK(hipGetLastError());
  return DFARGO_OK;
}

extern "C" int dfargo_mlp_forward(dfargo_mlp *m, int batch, const float *x, float *y) {
  if (!m || !x || !y) return dfargo_set_error(DFARGO_ERR_ARG, "null argument");
  MCHK(hipSetDevice(m->dev));
  int rows, rc;
  if ((rc = load_inputs(m, batch, x, &rows)) || (rc = forward(m, rows, 0))) return rc;
  MCHK(hipMemcpyAsync(y, m->L.back().z, 4 * (size_t)batch * m->n_out, hipMemcpyDeviceToHost, m->stream));
  MCHK(hipStreamSynchronize(m->stream));
  return DFARGO_OK;
}

// the backward pass after a forward pass with targets: dZ of every hidden
// layer, from the top, then all weight and bias gradients in one launch (each
// dZ reads the weights of the layer above it, so none changes before).  With
// lr > 0 an Adam step, else the gradients into gw, gb.
static int backward(dfargo_mlp *m, int rows, float lr) {
  for (int l = (int)m->L.size() - 1; l > 0; l--) {
    Layer &y = m->L[l], &p = m->L[l - 1];
    hipLaunchKernelGGL(k_backward, dim3(p.n / 32, rows / 32), dim3(64), 0, m->stream, y.dz, y.wb, y.n, p.n, rows, p.z,
                       p.dz, p.dzT, p.col_part);
  }
  GradArgs a;
  a.nl = (int)m->L.size();
  a.rows = rows;
  a.train = lr > 0.0f;
  a.lr = lr;
  a.b1 = 0.9f;
  a.b2 = 0.999f;
  a.eps = 1e-8f;
  a.c1 = 1.0f - powf(a.b1, (float)m->step);
  a.c2 = 1.0f - powf(a.b2, (float)m->step);
  int tiles = 0;
  for (int l = 0; l < a.nl; l++) {
    Layer &y = m->L[l];
    LayerGrad &g = a.l[l];
    g.k = y.k; g.n = y.n; g.tile0 = tiles;
    g.inT = l == 0 ? m->XT : m->L[l - 1].hT;
    g.dzT = y.dzT; g.col_part = y.col_part;
    g.w = y.w; g.b = y.b; g.gw = y.gw; g.gb = y.gb;
    g.mw = y.mw; g.vw = y.vw; g.mb = y.mb; g.vb = y.vb;
    g.wb = y.wb; g.wT = y.wT;
    tiles += (y.k / 32) * (y.n / 32);
  }
  hipLaunchKernelGGL(k_weights, dim3(tiles), dim3(64 * DW_WAVES), 0, m->stream, a);
  MCHK(hipGetLastError());
  return DFARGO_OK;
}

static int load_targets(dfargo_mlp *m, int batch, const float *t) {
  MCHK(hipMemcpyAsync(m->t_in, t, 4 * (size_t)batch * m->n_out, hipMemcpyHostToDevice, m->stream));
  return DFARGO_OK;
}

// the parameters (or their gradients) in the flat order W0, b0, W1, b1, ...
// with W_l as n_in(l) x n(l) row-major over the real inputs
static int copy_params(dfargo_mlp *m, float *host, int grads, int to_device) {
  size_t off = 0;
  for (size_t l = 0; l < m->L.size(); l++) {
    Layer &y = m->L[l];
    const int kin = l == 0 ? m->n_in : y.k;
    float *w = grads ? y.gw : y.w, *b = grads ? y.gb : y.b;
    const size_t nw = (size_t)kin * y.n;
    if (to_device) {
      MCHK(hipMemcpyAsync(w, host + off, 4 * nw, hipMemcpyHostToDevice, m->stream));
      MCHK(hipMemcpyAsync(b, host + off + nw, 4 * (size_t)y.n, hipMemcpyHostToDevice, m->stream));
      const size_t all = (size_t)y.k * y.n;
      hipLaunchKernelGGL(k_weights_bf16, dim3((all + 255) / 256), dim3(256), 0, m->stream, y.w, y.wb, y.wT, y.k,
                         y.n);
    } else {
      MCHK(hipMemcpyAsync(host + off, w, 4 * nw, hipMemcpyDeviceToHost, m->stream));
      MCHK(hipMemcpyAsync(host + off + nw, b, 4 * (size_t)y.n, hipMemcpyDeviceToHost, m->stream));
    }
    off += nw + y.n;
  }
  MCHK(hipStreamSynchronize(m->stream));
  return DFARGO_OK;
}

extern "C" int dfargo_mlp_get_params(dfargo_mlp *m, float *out) {
  if (!m || !out) return dfargo_set_error(DFARGO_ERR_ARG, "null argument");
  MCHK(hipSetDevice(m->dev));
  return copy_params(m, out, 0, 0);
}

extern "C" int dfargo_mlp_set_params(dfargo_mlp *m, const float *in) {
  if (!m || !in) return dfargo_set_error(DFARGO_ERR_ARG, "null argument");
  MCHK(hipSetDevice(m->dev));
  return copy_params(m, (float *)in, 0, 1);
}

extern "C" int dfargo_mlp_gradients(dfargo_mlp *m, int batch, const float *x, const float *t, float *loss,
                                    float *grads) {
  if (!m || !x || !t || !loss || !grads) return dfargo_set_error(DFARGO_ERR_ARG, "null argument");
  MCHK(hipSetDevice(m->dev));
  int rows, rc;
  if ((rc = load_inputs(m, batch, x, &rows)) || (rc = load_targets(m, batch, t)) || (rc = forward(m, rows, batch)) ||
      (rc = backward(m, rows, 0.0f)) || (rc = form_loss(m, batch, rows)))
    return rc;
  MCHK(hipMemcpyAsync(loss, m->loss, 4, hipMemcpyDeviceToHost, m->stream));
  return copy_params(m, grads, 1, 0);
}

extern "C" int dfargo_mlp_train(dfargo_mlp *m, int batch, const float *x, const float *t, int steps, float lr,
                                float *loss) {
  if (!m || !x || !t) return dfargo_set_error(DFARGO_ERR_ARG, "null argument");
  if (steps < 0 || !(lr > 0.0f)) return dfargo_set_error(DFARGO_ERR_ARG, "need steps >= 0 and lr > 0");
  MCHK(hipSetDevice(m->dev));
  int rows, rc;
  if ((rc = load_inputs(m, batch, x, &rows)) || (rc = load_targets(m, batch, t))) return rc;
  for (int s = 0; s < steps; s++) {
    m->step++;
    if ((rc = forward(m, rows, batch)) || (rc = backward(m, rows, lr))) return rc;
  }
  if (loss) {
    // the loss of the parameters after the last step
    if ((rc = forward(m, rows, batch)) || (rc = form_loss(m, batch, rows))) return rc;
    MCHK(hipMemcpyAsync(loss, m->loss, 4, hipMemcpyDeviceToHost, m->stream));
  }
  MCHK(hipStreamSynchronize(m->stream));
  return DFARGO_OK;
}
