// se2w_mlp.hip -- the seismogram surrogate: an MLP trained and evaluated with
// hand-written gfx950 kernels (include/se2w_mlp.h).
//
// Every product is one kernel shape, C[M][N] = sum_k A[M][k] B[N][k] with
// both operands BF16 in MFMA order (op_index), on v_mfma_f32_16x16x32_bf16 with FP32
// accumulation.  The three products of a layer (forward, input gradient,
// weight gradient) all take that shape because the forward and backward
// epilogues also write the transposes of the activations and of the
// pre-activation gradients, and the Adam update keeps a transposed BF16 copy
// of each weight matrix.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <memory>
#include <new>
#include <vector>

#include "se2w.h"
#include "se2w_mlp.h"

namespace se2w {
int set_error(int code, const char *msg);
}

namespace {

typedef __bf16 bf16;
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

int mfail(int code, const char *fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  return se2w::set_error(code, buf);
}

#define MCHK(call)                                                                             \
  do {                                                                                         \
    hipError_t e_ = (call);                                                                    \
    if (e_ != hipSuccess) return mfail(SE2W_ERR_HIP, "%s: %s", #call, hipGetErrorString(e_)); \
  } while (0)

__device__ __forceinline__ float gelu(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_grad(float z) {
  return 0.5f * (1.0f + erff(z * 0.70710678118654752f)) + z * 0.39894228040143268f * expf(-0.5f * z * z);
}

// BF16 operands are stored in MFMA order: the 16 x 32 block (r / 16, k / 32)
// of an operand with K columns is 1 KB, lane l's eight values at 16 l bytes
// (row l % 16, columns 8 (l / 16) .. +7 of the block).  An operand load of a
// wave is then one contiguous KB.  From row-major storage neighbouring lanes
// read 16 bytes of different rows, and the loads ran at 16 bytes per clock
// and CU: a 256 x 1024 x 4096 product took 32.4 us instead of 12.1.
__host__ __device__ constexpr long op_index(int r, int k, int K) {
  return ((long)(r / 16) * (K / 32) + k / 32) * 512 + (16 * (k % 32 / 8) + r % 16) * 8 + k % 8;
}

enum { EPI_GELU = 0, EPI_LINEAR = 1, EPI_DGELU = 2, EPI_LOSS = 3 };

struct GemmArgs {
  const bf16 *A;  // M x K operand
  const bf16 *B;  // N x K operand
  int M, N, K;
  const float *bias;   // [N]          (all but EPI_DGELU)
  float *Cf;           // [M][N]       FP32 result: pre-activation (EPI_GELU), output (EPI_LINEAR)
  bf16 *Cb;            // M x N operand: BF16 activation / gradient
  bf16 *Cbt;           // N x ldt operand: its transpose, ldt the batch
  const float *Zprev;  // [M][N]       pre-activation whose GELU' scales the product (EPI_DGELU)
  int ldt;
  // EPI_LOSS: the mean-squared error against rows idx[m] of T and its
  // gradient scale (C + bias - T) as Cb, Cbt; each workgroup's sum of squares
  // to part[its linear index]
  const float *T;
  const int *idx;
  float scale;
  double *part;
};

// A workgroup of WM x WN waves, each forming TM x TN MFMA tiles of 16 x 16
// over the whole of K.  The products here have few rows (a batch), so a
// launch fills the chip only with small tiles and its time is the latency of
// the operand loads: each wave reads its operands from global memory straight
// into registers in MFMA layout, U steps of 32 at a time with the next U
// steps already in flight; no barrier and no LDS round trip per step.  Every
// element is one chain of products in ascending k, so its bits do not depend
// on the tile shape.  The result goes through LDS once, so that the epilogue
// reads and writes 16 bytes per lane.
// MFMA 16x16x32 operand layout: lane l holds A[l % 16][8 (l / 16) .. +7] and
// B[8 (l / 16) .. +7][l % 16] (B is stored [n][k], so also row l % 16, eight
// consecutive k); the result D[4 (l / 16) + r][l % 16] is its r-th
// accumulator.
template <int EPI, int TM, int TN, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN) void gemm_nt(GemmArgs g) {
  constexpr int MT = 16 * TM * WM, NT = 16 * TN * WN, THREADS = 64 * WM * WN, U = 16 / (TM + TN);
  __shared__ __attribute__((aligned(16))) float ct[MT][NT + 4];
  __shared__ __attribute__((aligned(16))) bf16 th[MT][NT + 8], tr[NT][MT + 8];  // BF16 result and its transpose
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int m0 = blockIdx.y * MT, n0 = blockIdx.x * NT;
  const int wm = 16 * TM * (wave / WN), wn = 16 * TN * (wave % WN);
  floatx4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  const int ks = g.K / 32;
  const bf16 *ga = g.A + op_index(m0 + wm, 0, g.K) + 8 * lane;
  const bf16 *gb = g.B + op_index(n0 + wn, 0, g.K) + 8 * lane;
  bf16x8 a[2][U][TM], b[2][U][TN];
  // loads of the steps k .. k + U - 1 (past the end the last step is read
  // again, and not multiplied)
  auto load = [&](int slot, int k) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int o = min(k + u, ks - 1);
#pragma unroll
      for (int i = 0; i < TM; i++) a[slot][u][i] = *(const bf16x8 *)(ga + 512l * (i * ks + o));
#pragma unroll
      for (int j = 0; j < TN; j++) b[slot][u][j] = *(const bf16x8 *)(gb + 512l * (j * ks + o));
    }
  };
  auto multiply = [&](int slot, int k) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (k + u < ks) {  // uniform
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int j = 0; j < TN; j++)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[slot][u][i], b[slot][u][j], acc[i][j], 0, 0, 0);
      }
    }
  };
  load(0, 0);
  for (int k = 0; k < ks; k += 2 * U) {
    load(1, k + U);
    multiply(0, k);
    load(0, k + 2 * U);
    multiply(1, k + U);
  }
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) ct[wm + 16 * i + 4 * (lane >> 4) + r][wn + 16 * j + (lane & 15)] = acc[i][j][r];
  __syncthreads();
  [[maybe_unused]] double sq = 0.0;
  for (int q = tid; q < MT * NT / 4; q += THREADS) {
    const int lm = q / (NT / 4), ln = 4 * (q % (NT / 4));
    floatx4 c = *(const floatx4 *)&ct[lm][ln];
    const int n = n0 + ln;
    const long o = (long)(m0 + lm) * g.N + n;
    if constexpr (EPI != EPI_DGELU) c += *(const floatx4 *)(g.bias + n);
    if constexpr (EPI == EPI_GELU || EPI == EPI_LINEAR) *(floatx4 *)(g.Cf + o) = c;
    if constexpr (EPI != EPI_LINEAR) {
      bf16x4 h;
      if constexpr (EPI == EPI_LOSS) {
        const floatx4 d = c - *(const floatx4 *)(g.T + (long)g.idx[m0 + lm] * g.N + n);
#pragma unroll
        for (int r = 0; r < 4; r++) {
          sq += (double)d[r] * d[r];
          h[r] = (bf16)(g.scale * d[r]);
        }
      } else if constexpr (EPI == EPI_DGELU) {
        const floatx4 z = *(const floatx4 *)(g.Zprev + o);
#pragma unroll
        for (int r = 0; r < 4; r++) h[r] = (bf16)(c[r] * gelu_grad(z[r]));
      } else {
#pragma unroll
        for (int r = 0; r < 4; r++) h[r] = (bf16)gelu(c[r]);
      }
      *(bf16x4 *)&th[lm][ln] = h;
#pragma unroll
      for (int r = 0; r < 4; r++) tr[ln + r][lm] = h[r];
    }
  }
  if constexpr (EPI != EPI_LINEAR) {
    __syncthreads();
    for (int q = tid; q < MT * NT / 8; q += THREADS) {  // 16 rows of one 16-byte column piece at a time
      const int c = 8 * (q / 16 % (NT / 8)), r = 16 * (q / (2 * NT)) + q % 16;
      *(bf16x8 *)(g.Cb + op_index(m0 + r, n0 + c, g.N)) = *(const bf16x8 *)&th[r][c];
      const int ct8 = 8 * (q / 16 % (MT / 8)), rt = 16 * (q / (2 * MT)) + q % 16;
      *(bf16x8 *)(g.Cbt + op_index(n0 + rt, m0 + ct8, g.ldt)) = *(const bf16x8 *)&tr[rt][ct8];
    }
  }
  if constexpr (EPI == EPI_LOSS) {
    __shared__ double red[WM * WN];
#pragma unroll
    for (int w = 32; w > 0; w >>= 1) sq += __shfl_down(sq, w);
    if (lane == 0) red[wave] = sq;
    __syncthreads();
    if (tid == 0) {
      for (int w = 1; w < WM * WN; w++) sq += red[w];
      g.part[blockIdx.y * gridDim.x + blockIdx.x] = sq;
    }
  }
}

// Batch gather: rows idx[r] of the FP32 data become the BF16 input
// activations and their transpose (the targets are read in place by the loss).
__global__ void k_gather(const float *X, const int *idx, int B, int in_pad, bf16 *H0, bf16 *H0t) {
  const int r = blockIdx.x;
  const long src = idx[r];
  for (int k = threadIdx.x; k < in_pad; k += blockDim.x) {
    const bf16 h = (bf16)X[src * in_pad + k];
    H0[op_index(r, k, in_pad)] = h;
    H0t[op_index(k, r, B)] = h;
  }
}

// Rows of a forward batch, read in place from pinned host memory (a batch is
// some tens of KB; its upload by a copy command took longer than the network
// for one row): x[n][in] become the rows from row0 of the input operand, zero
// in the padding and in the rows past n.
__global__ void k_rows(const float *x, int n, int row0, int in, int in_pad, bf16 *H0) {
  const int r = blockIdx.x;
  for (int k = blockIdx.y * blockDim.x + threadIdx.x; k < in_pad; k += gridDim.y * blockDim.x)
    H0[op_index(row0 + r, k, in_pad)] = (bf16)(r < n && k < in ? x[(long)r * in + k] : 0.f);
}

// Download of n 16-byte pieces into pinned host memory: queued behind the
// product like any kernel, where a copy command waits for another engine.
__global__ __launch_bounds__(256) void k_to_host(const floatx4 *src, floatx4 *dst, long n) {
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long)gridDim.x * 256) dst[i] = src[i];
}

// *out = inv_count times the sum of part[0..n), one workgroup, fixed order.
__global__ __launch_bounds__(256) void k_sum_parts(const double *part, long n, double inv_count, double *out) {
  __shared__ double red[256];
  double s = 0.0;
  for (long i = threadIdx.x; i < n; i += 256) s += part[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = red[0] * inv_count;
}

struct AdamArgs {
  float lr, b1, b2, eps, bc1, bc2;  // bc = 1 - beta^t
  float wd;                         // decoupled weight decay (AdamW); 0 = Adam
};

// The fused multiply-adds are spelled out, so that every kernel that inlines
// the update rounds alike.
__device__ __forceinline__ float adam_update(float &w, float &m, float &v, float g, const AdamArgs &a) {
  m = fmaf(a.b1, m, (1.f - a.b1) * g);
  v = fmaf(a.b2, v, (1.f - a.b2) * g * g);
  w = fmaf(-a.lr, fmaf(a.wd, w, (m / a.bc1) / (sqrtf(v / a.bc2) + a.eps)), w);
  return w;
}

// Adam on a [rows][cols] weight matrix (rows, cols multiples of 32): FP32
// master weights, BF16 operand Wb (rows x cols) and its transpose Wtb.
// A 32 x 32 tile per workgroup of 32 x 8 threads; the transpose goes through LDS.
__global__ __launch_bounds__(256) void k_adam_w(float *W, float *m, float *v, const float *g, int rows, int cols,
                                                AdamArgs a, bf16 *Wb, bf16 *Wtb) {
  __shared__ bf16 tile[32][33];
  const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int k = ty; k < 32; k += 8) {
    const long o = (long)(r0 + k) * cols + c0 + tx;
    float w = W[o], mm = m[o], vv = v[o];
    adam_update(w, mm, vv, g[o], a);
    W[o] = w;
    m[o] = mm;
    v[o] = vv;
    const bf16 h = (bf16)w;
    Wb[op_index(r0 + k, c0 + tx, cols)] = h;
    tile[k][tx] = h;
  }
  __syncthreads();
  for (int k = ty; k < 32; k += 8) Wtb[op_index(c0 + k, r0 + tx, rows)] = tile[tx][k];
}

__global__ void k_adam_b(float *b, float *m, float *v, const float *g, int n, AdamArgs a) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float w = b[i], mm = m[i], vv = v[i];
  adam_update(w, mm, vv, g[i], a);
  b[i] = w;
  m[i] = mm;
  v[i] = vv;
}

// One layer of the grouped weight kernel.
struct WgradLayer {
  const bf16 *dZt;  // out x B operand: gradient of the pre-activation, transposed
  const bf16 *Ht;   // in_pad x B operand: the layer's input, transposed
  int out, in_pad;
  int tile0;        // its first workgroup; it has (out / 64) (in_pad / 64) tiles, then ceil(out / 256) bias blocks
  float *W, *mW, *vW, *gW, *b, *mb, *vb, *gb;
  bf16 *Wb, *Wtb;
};

// Weight and bias gradients of every layer in one launch, and with ADAM the
// update in place of storing them: gW = dZt Ht^T (K = the batch) never goes
// to memory.  The update moves 28 bytes per weight (W, m, v read and written,
// both BF16 copies written), which bounds the kernel: a workgroup takes a
// 64 x 64 tile of W, whose product needs only 2 x 64 rows of the batch.  The
// four waves form a 32 x 32 quarter each from registers (as gemm_nt, one
// chain per element in ascending k), and the tile goes through LDS so that
// the update streams whole lines.  The bias blocks sum a row of dZt per
// thread in ascending order, with eight 16-byte loads in flight.
template <bool ADAM>
__global__ __launch_bounds__(256) void k_wgrad(const WgradLayer *layers, int nl, int B, AdamArgs a) {
  __shared__ __attribute__((aligned(16))) float gt[64][68];
  __shared__ __attribute__((aligned(16))) bf16 th[64][72], tr[64][72];
  const int tid = threadIdx.x;
  int l = nl - 1;
  while (l > 0 && (int)blockIdx.x < layers[l].tile0) l--;
  const WgradLayer L = layers[l];
  const int t = blockIdx.x - L.tile0, tx = L.in_pad / 64, nt = tx * (L.out / 64);
  if (t >= nt) {  // bias block
    const int o = (t - nt) * 256 + tid;
    if (o >= L.out) return;
    const bf16 *row = L.dZt + op_index(o, 0, B);  // eight values every 128, 512 per 32 columns
    float s = 0.f;
    for (int k = 0; k < B; k += 64) {
      bf16x8 x[8];
#pragma unroll
      for (int q = 0; q < 8; q++) x[q] = *(const bf16x8 *)(row + 16l * k + 128 * q);
#pragma unroll
      for (int q = 0; q < 8; q++)
#pragma unroll
        for (int r = 0; r < 8; r++) s += (float)x[q][r];
    }
    if constexpr (ADAM) {
      float w = L.b[o], mm = L.mb[o], vv = L.vb[o];
      adam_update(w, mm, vv, s, a);
      L.b[o] = w;
      L.mb[o] = mm;
      L.vb[o] = vv;
    } else {
      L.gb[o] = s;
    }
    return;
  }
  const int m0 = 64 * (t / tx), n0 = 64 * (t % tx);
  const int wave = tid >> 6, lane = tid & 63, wm = 32 * (wave >> 1), wn = 32 * (wave & 1);
  // this thread's part of the update: rows er + 16 q, four columns from ec
  const int er = tid >> 4, ec = 4 * (tid & 15);
  floatx4 w4[4], m4[4], v4[4];
  if constexpr (ADAM) {  // issued first: their latency overlaps the product
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const long o = (long)(m0 + er + 16 * q) * L.in_pad + n0 + ec;
      w4[q] = *(const floatx4 *)(L.W + o);
      m4[q] = *(const floatx4 *)(L.mW + o);
      v4[q] = *(const floatx4 *)(L.vW + o);
    }
  }
  floatx4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  const bf16 *ga = L.dZt + op_index(m0 + wm, 0, B) + 8 * lane;
  const bf16 *gb = L.Ht + op_index(n0 + wn, 0, B) + 8 * lane;
  for (int k = 0; k < B; k += 64) {  // B is a multiple of 64
    bf16x8 x[2][2], y[2][2];
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int i = 0; i < 2; i++) {
        x[u][i] = *(const bf16x8 *)(ga + 16l * (i * B + k + 32 * u));
        y[u][i] = *(const bf16x8 *)(gb + 16l * (i * B + k + 32 * u));
      }
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[u][i], y[u][j], acc[i][j], 0, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) gt[wm + 16 * i + 4 * (lane >> 4) + r][wn + 16 * j + (lane & 15)] = acc[i][j][r];
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int lm = er + 16 * q;
    const long o = (long)(m0 + lm) * L.in_pad + n0 + ec;
    const floatx4 g = *(const floatx4 *)&gt[lm][ec];
    if constexpr (ADAM) {
      bf16x4 h;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        float w = w4[q][r], mm = m4[q][r], vv = v4[q][r];
        adam_update(w, mm, vv, g[r], a);
        w4[q][r] = w;
        m4[q][r] = mm;
        v4[q][r] = vv;
        h[r] = (bf16)w;
        tr[ec + r][lm] = h[r];
      }
      *(bf16x4 *)&th[lm][ec] = h;
      *(floatx4 *)(L.W + o) = w4[q];
      *(floatx4 *)(L.mW + o) = m4[q];
      *(floatx4 *)(L.vW + o) = v4[q];
    } else {
      *(floatx4 *)(L.gW + o) = g;
    }
  }
  if constexpr (ADAM) {
    __syncthreads();
    for (int q = tid; q < 64 * 8; q += 256) {
      const int c = 8 * (q / 16 % 8), r = 16 * (q / 128) + q % 16;
      *(bf16x8 *)(L.Wb + op_index(m0 + r, n0 + c, L.in_pad)) = *(const bf16x8 *)&th[r][c];
      *(bf16x8 *)(L.Wtb + op_index(n0 + r, m0 + c, L.out)) = *(const bf16x8 *)&tr[r][c];
    }
  }
}

// BF16 copies of the FP32 master weights (after set_params / init).
__global__ void k_to_bf16(const float *W, int rows, int cols, bf16 *Wb, bf16 *Wtb) {
  const long n = (long)rows * cols;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const int r = (int)(i / cols), c = (int)(i - (long)r * cols);
    const bf16 h = (bf16)W[i];
    Wb[op_index(r, c, cols)] = h;
    Wtb[op_index(c, r, rows)] = h;
  }
}

int round_up(int x, int m) { return (x + m - 1) / m * m; }

}  // namespace

struct MlpLayer {
  int in = 0, in_pad = 0, out = 0;
  float *W = nullptr, *b = nullptr, *gW = nullptr, *gb = nullptr, *mW = nullptr, *vW = nullptr, *mb = nullptr,
        *vb = nullptr;
  bf16 *Wb = nullptr, *Wtb = nullptr;        // out x in_pad operand and its transpose
  float *Z = nullptr;                        // pre-activation [B][out] (hidden layers)
  bf16 *H = nullptr, *Ht = nullptr;          // activation, B x out operand and its transpose (hidden layers)
  bf16 *dZ = nullptr, *dZt = nullptr;        // d loss / d pre-activation, likewise
};

// Output chunks that se2w_mlp_forward keeps in flight.
constexpr int kAhead = 4;

struct se2w_mlp {
  int device = 0, nl = 0, B = 0, in = 0, in_pad = 0, out = 0;
  std::vector<MlpLayer> L;
  bf16 *H0 = nullptr, *H0t = nullptr;
  float *Y = nullptr;
  float *Xs = nullptr, *Ts = nullptr;  // staging of one host batch
  int *idx = nullptr;                  // batch row indices
  WgradLayer *wgrad = nullptr;         // [nl] the grouped weight kernel's layers
  int wgrad_blocks = 0;
  float *X = nullptr, *T = nullptr;    // training data
  int ndata = 0;
  // per-workgroup squared errors of the batches of an epoch, nparts each
  double *part = nullptr;
  int nparts = 0, part_batches = 0;
  // se2w_mlp_forward's pinned buffers: kAhead + 1 pieces of input rows and
  // kAhead chunks of output rows, with the events of each
  float *x_host = nullptr, *y_host = nullptr;
  hipEvent_t x_read[kAhead + 1] = {}, y_up[kAhead] = {}, f0[kAhead + 1] = {}, f1[kAhead + 1] = {};
  double *loss = nullptr;  // loss of one batch (se2w_mlp_gradient)
  // two permutations (this epoch's and the next one's), device and pinned
  int *perm_dev = nullptr, *perm_host = nullptr;
  size_t perm_cap = 0;  // entries of one
  hipEvent_t perm_up[2] = {nullptr, nullptr};
  hipStream_t stream = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  long t = 0;  // Adam steps taken
  float weight_decay = 0.f;
  int cosine = 0;  // cosine learning-rate decay over each se2w_mlp_train call
  double train_ms = 0.0, fwd_ms = 0.0;
  std::vector<void *> allocs;
};

namespace {

template <typename T>
int malloc_zero(se2w_mlp *m, T **p, size_t n) {
  *p = nullptr;
  void *q = nullptr;
  if (hipMalloc(&q, sizeof(T) * std::max<size_t>(n, 1)) != hipSuccess)
    return mfail(SE2W_ERR_MEM, "hipMalloc of %zu bytes failed", sizeof(T) * n);
  m->allocs.push_back(q);
  MCHK(hipMemsetAsync(q, 0, sizeof(T) * std::max<size_t>(n, 1), m->stream));
  *p = (T *)q;
  return SE2W_OK;
}

// Tile rule: 64 x 64 when that gives every CU a workgroup (256 of them), else
// 32 x 32 when that does, else 16 x 16 with one wave per workgroup: a smaller
// tile re-reads the operands more often, a larger one leaves CUs idle.
constexpr int kCUs = 256;
int tile_of(int M, int N) {
  const long tiles16 = (long)(M / 16) * (N / 16);
  return M % 64 == 0 && tiles16 >= 16 * kCUs ? 64 : M % 32 == 0 && tiles16 >= 4 * kCUs ? 32 : 16;
}
template <int EPI>
int gemm(se2w_mlp *m, const GemmArgs &g) {
  if (g.M % 16 || g.N % 64 || g.K % 64)
    return mfail(SE2W_ERR_ARG, "product shape %d x %d x %d not tileable", g.M, g.N, g.K);
  const int tile = tile_of(g.M, g.N);
  if (tile == 64)
    hipLaunchKernelGGL((gemm_nt<EPI, 2, 2, 2, 2>), dim3(g.N / 64, g.M / 64), dim3(256), 0, m->stream, g);
  else if (tile == 32)
    hipLaunchKernelGGL((gemm_nt<EPI, 1, 1, 2, 2>), dim3(g.N / 32, g.M / 32), dim3(256), 0, m->stream, g);
  else
    hipLaunchKernelGGL((gemm_nt<EPI, 1, 1, 1, 1>), dim3(g.N / 16, g.M / 16), dim3(64), 0, m->stream, g);
  return SE2W_OK;
}

// Targets and outputs of a batch's loss.
struct LossArgs {
  const float *T;   // [rows][out]
  const int *idx;   // [B] the batch's rows
  double *part;     // [nparts]
};

// Forward pass of the first `rows` rows in H0.  The outputs go to Y or, with a
// loss (rows = the batch), their error's gradient to the last layer's dZ, dZt
// and the squared errors to part; the outputs themselves are then not stored.
int forward(se2w_mlp *m, int rows, const LossArgs *loss, float *Y) {
  for (int l = 0; l < m->nl; l++) {
    MlpLayer &Ly = m->L[l];
    GemmArgs g = {};
    g.A = l == 0 ? m->H0 : m->L[l - 1].H;
    g.B = Ly.Wb;
    g.M = rows;
    g.N = Ly.out;
    g.K = Ly.in_pad;
    g.bias = Ly.b;
    g.ldt = m->B;
    int ierr;
    if (l < m->nl - 1) {
      g.Cf = Ly.Z;
      g.Cb = Ly.H;
      g.Cbt = Ly.Ht;
      ierr = gemm<EPI_GELU>(m, g);
    } else if (loss) {
      g.Cb = Ly.dZ;
      g.Cbt = Ly.dZt;
      g.T = loss->T;
      g.idx = loss->idx;
      g.part = loss->part;
      g.scale = 2.0f / ((float)m->B * (float)m->out);
      ierr = gemm<EPI_LOSS>(m, g);
    } else {
      g.Cf = Y;
      ierr = gemm<EPI_LINEAR>(m, g);
    }
    if (ierr) return ierr;
  }
  MCHK(hipGetLastError());
  return SE2W_OK;
}

// The gradient of every hidden pre-activation from the last layer's.
int backward(se2w_mlp *m) {
  for (int l = m->nl - 1; l > 0; l--) {
    MlpLayer &Ly = m->L[l];
    MlpLayer &Lp = m->L[l - 1];
    GemmArgs h = {};
    h.A = Ly.dZ;
    h.B = Ly.Wtb;
    h.M = m->B;
    h.N = Ly.in_pad;
    h.K = Ly.out;
    h.Zprev = Lp.Z;
    h.Cb = Lp.dZ;
    h.Cbt = Lp.dZt;
    h.ldt = m->B;
    if (int ierr = gemm<EPI_DGELU>(m, h)) return ierr;
  }
  MCHK(hipGetLastError());
  return SE2W_OK;
}

// The Adam step number t + 1 at learning rate lr.
AdamArgs next_adam(se2w_mlp *m, float lr) {
  m->t++;
  AdamArgs a;
  a.lr = lr;
  a.b1 = 0.9f;
  a.b2 = 0.999f;
  a.eps = 1e-8f;
  a.wd = m->weight_decay;
  a.bc1 = (float)(1.0 - std::pow(0.9, (double)m->t));
  a.bc2 = (float)(1.0 - std::pow(0.999, (double)m->t));
  return a;
}

// All parameter gradients of the batch into gW, gb.
int weight_gradients(se2w_mlp *m) {
  hipLaunchKernelGGL(k_wgrad<false>, dim3(m->wgrad_blocks), dim3(256), 0, m->stream, (const WgradLayer *)m->wgrad,
                     m->nl, m->B, AdamArgs{});
  MCHK(hipGetLastError());
  return SE2W_OK;
}

// The same gradients, applied as one Adam step.
int weight_update(se2w_mlp *m, float lr) {
  hipLaunchKernelGGL(k_wgrad<true>, dim3(m->wgrad_blocks), dim3(256), 0, m->stream, (const WgradLayer *)m->wgrad,
                     m->nl, m->B, next_adam(m, lr));
  MCHK(hipGetLastError());
  return SE2W_OK;
}

// One Adam step from the stored gradients gW, gb.
int adam(se2w_mlp *m, float lr) {
  const AdamArgs a = next_adam(m, lr);
  for (MlpLayer &Ly : m->L) {
    hipLaunchKernelGGL(k_adam_w, dim3(Ly.in_pad / 32, Ly.out / 32), dim3(256), 0, m->stream, Ly.W, Ly.mW, Ly.vW,
                       (const float *)Ly.gW, Ly.out, Ly.in_pad, a, Ly.Wb, Ly.Wtb);
    hipLaunchKernelGGL(k_adam_b, dim3((Ly.out + 255) / 256), dim3(256), 0, m->stream, Ly.b, Ly.mb, Ly.vb,
                       (const float *)Ly.gb, Ly.out, a);
  }
  MCHK(hipGetLastError());
  return SE2W_OK;
}

// Uploads n <= B host rows into the staging buffers (zero rows after n) and
// gathers them as the current batch.
int stage_batch(se2w_mlp *m, int n, const float *x, const float *t) {
  std::vector<float> xp((size_t)m->B * m->in_pad, 0.f);
  for (int r = 0; r < n; r++) memcpy(&xp[(size_t)r * m->in_pad], x + (size_t)r * m->in, sizeof(float) * m->in);
  MCHK(hipMemcpyAsync(m->Xs, xp.data(), sizeof(float) * xp.size(), hipMemcpyHostToDevice, m->stream));
  if (t) MCHK(hipMemcpyAsync(m->Ts, t, sizeof(float) * (size_t)n * m->out, hipMemcpyHostToDevice, m->stream));
  std::vector<int> id(m->B);
  for (int r = 0; r < m->B; r++) id[r] = r;
  MCHK(hipMemcpyAsync(m->idx, id.data(), sizeof(int) * m->B, hipMemcpyHostToDevice, m->stream));
  hipLaunchKernelGGL(k_gather, dim3(m->B), dim3(128), 0, m->stream, (const float *)m->Xs, (const int *)m->idx, m->B,
                     m->in_pad, m->H0, m->H0t);
  MCHK(hipStreamSynchronize(m->stream));  // the host vectors above go out of scope
  return SE2W_OK;
}

// Squared-error sums of `batches` batches.  A buffer that cannot grow stays:
// the loss of a gradient is written to it.
int ensure_parts(se2w_mlp *m, int batches) {
  if (batches <= m->part_batches) return SE2W_OK;
  double *part = nullptr;
  if (hipMalloc(&part, sizeof(double) * (size_t)batches * m->nparts) != hipSuccess)
    return mfail(SE2W_ERR_MEM, "hipMalloc failed");
  if (m->part) hipFree(m->part);
  m->part = part;
  m->part_batches = batches;
  return SE2W_OK;
}

// Output rows of one downloaded chunk: about 1 MB, so that the copy out of a
// chunk hides behind the next chunks' downloads, and at least the 16 rows that
// a product writes at once.
int chunk_rows(const se2w_mlp *m) { return std::min(m->B, std::max(16, (1 << 18) / m->out)); }

// Input rows of one pinned piece: a batch up to about 1 MB, so that what a
// network pins does not grow with its batch (pinning 5 x 134 MB took 250 ms).
int piece_rows(const se2w_mlp *m) { return std::min(m->B, std::max(1, (1 << 18) / m->in)); }

int forward_buffers(se2w_mlp *m) {
  for (hipEvent_t &e : m->y_up)
    if (!e) MCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  for (hipEvent_t &e : m->x_read)
    if (!e) MCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  for (int s = 0; s <= kAhead; s++) {
    if (!m->f0[s]) MCHK(hipEventCreate(&m->f0[s]));
    if (!m->f1[s]) MCHK(hipEventCreate(&m->f1[s]));
  }
  // Filled once: the host's first touch of a pinned page costs a fault each,
  // which the first forward would pay.
  const size_t nx = (size_t)(kAhead + 1) * piece_rows(m) * m->in, ny = (size_t)kAhead * chunk_rows(m) * m->out;
  if (!m->x_host) {
    MCHK(hipHostMalloc((void **)&m->x_host, sizeof(float) * nx, hipHostMallocDefault));
    memset(m->x_host, 0, sizeof(float) * nx);
  }
  if (!m->y_host) {
    MCHK(hipHostMalloc((void **)&m->y_host, sizeof(float) * ny, hipHostMallocDefault));
    memset(m->y_host, 0, sizeof(float) * ny);
  }
  return SE2W_OK;
}

// Both permutation buffers, n entries each.
int ensure_perm(se2w_mlp *m, size_t n) {
  for (hipEvent_t &e : m->perm_up)
    if (!e) MCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  if (n <= m->perm_cap) return SE2W_OK;
  if (m->perm_dev) hipFree(m->perm_dev);
  if (m->perm_host) hipHostFree(m->perm_host);
  m->perm_dev = m->perm_host = nullptr;
  m->perm_cap = 0;
  MCHK(hipMalloc(&m->perm_dev, 2 * sizeof(int) * n));
  MCHK(hipHostMalloc((void **)&m->perm_host, 2 * sizeof(int) * n, hipHostMallocDefault));
  m->perm_cap = n;
  return SE2W_OK;
}

uint64_t splitmix64(uint64_t &s) {
  uint64_t z = (s += 0x9E3779B97F4A7C15ull);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

double uniform01(uint64_t &s) { return (double)(splitmix64(s) >> 11) * (1.0 / 9007199254740992.0); }

int refresh_bf16(se2w_mlp *m) {
  for (MlpLayer &Ly : m->L)
    hipLaunchKernelGGL(k_to_bf16, dim3(256), dim3(256), 0, m->stream, (const float *)Ly.W, Ly.out, Ly.in_pad, Ly.Wb,
                       Ly.Wtb);
  MCHK(hipGetLastError());
  MCHK(hipStreamSynchronize(m->stream));
  return SE2W_OK;
}

}  // namespace

extern "C" {

int se2w_mlp_create(int32_t nlayers, const int32_t *widths, int32_t batch, uint64_t seed, int32_t device,
                    se2w_mlp **out) {
  if (!out || !widths || nlayers < 1 || batch < 64 || batch % 64) return mfail(SE2W_ERR_ARG, "bad network arguments");
  *out = nullptr;
  if (widths[0] < 1) return mfail(SE2W_ERR_ARG, "input width must be >= 1");
  for (int l = 1; l <= nlayers; l++)
    if (widths[l] < 64 || widths[l] % 64) return mfail(SE2W_ERR_ARG, "width %d (layer %d) must be a multiple of 64", widths[l], l);
  MCHK(hipSetDevice(device));
  se2w_mlp *m = new se2w_mlp;
  m->device = device;
  m->nl = nlayers;
  m->B = batch;
  m->in = widths[0];
  m->in_pad = round_up(widths[0], 64);
  m->out = widths[nlayers];
  int ierr = SE2W_OK;
  if (hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) != hipSuccess || hipEventCreate(&m->e0) != hipSuccess ||
      hipEventCreate(&m->e1) != hipSuccess) {
    se2w_mlp_destroy(m);
    return mfail(SE2W_ERR_HIP, "stream/event creation failed");
  }
  m->L.resize(nlayers);
  uint64_t rng = seed;
  for (int l = 0; l < nlayers && !ierr; l++) {
    MlpLayer &Ly = m->L[l];
    Ly.in = widths[l];
    Ly.in_pad = l == 0 ? m->in_pad : widths[l];
    Ly.out = widths[l + 1];
    const size_t nw = (size_t)Ly.out * Ly.in_pad;
    if ((ierr = malloc_zero(m, &Ly.W, nw)) || (ierr = malloc_zero(m, &Ly.b, Ly.out)) ||
        (ierr = malloc_zero(m, &Ly.gW, nw)) || (ierr = malloc_zero(m, &Ly.gb, Ly.out)) ||
        (ierr = malloc_zero(m, &Ly.mW, nw)) || (ierr = malloc_zero(m, &Ly.vW, nw)) ||
        (ierr = malloc_zero(m, &Ly.mb, Ly.out)) || (ierr = malloc_zero(m, &Ly.vb, Ly.out)) ||
        (ierr = malloc_zero(m, &Ly.Wb, nw)) || (ierr = malloc_zero(m, &Ly.Wtb, nw)) ||
        (ierr = malloc_zero(m, &Ly.dZ, (size_t)batch * Ly.out)) || (ierr = malloc_zero(m, &Ly.dZt, (size_t)batch * Ly.out)))
      break;
    if (l < nlayers - 1 &&
        ((ierr = malloc_zero(m, &Ly.Z, (size_t)batch * Ly.out)) || (ierr = malloc_zero(m, &Ly.H, (size_t)batch * Ly.out)) ||
         (ierr = malloc_zero(m, &Ly.Ht, (size_t)batch * Ly.out))))
      break;
    // U(-1/sqrt(fan_in), 1/sqrt(fan_in)) for weights and biases
    const double bound = 1.0 / std::sqrt((double)Ly.in);
    std::vector<float> w(nw, 0.f), b(Ly.out);
    for (int o = 0; o < Ly.out; o++)
      for (int i = 0; i < Ly.in; i++) w[(size_t)o * Ly.in_pad + i] = (float)((2.0 * uniform01(rng) - 1.0) * bound);
    for (int o = 0; o < Ly.out; o++) b[o] = (float)((2.0 * uniform01(rng) - 1.0) * bound);
    if (hipMemcpyAsync(Ly.W, w.data(), sizeof(float) * nw, hipMemcpyHostToDevice, m->stream) != hipSuccess ||
        hipMemcpyAsync(Ly.b, b.data(), sizeof(float) * Ly.out, hipMemcpyHostToDevice, m->stream) != hipSuccess ||
        hipStreamSynchronize(m->stream) != hipSuccess)
      ierr = mfail(SE2W_ERR_HIP, "weight upload failed");
  }
  m->nparts = (batch / tile_of(batch, m->out)) * (m->out / tile_of(batch, m->out));
  if (!ierr && ((ierr = malloc_zero(m, &m->H0, (size_t)batch * m->in_pad)) ||
                (ierr = malloc_zero(m, &m->H0t, (size_t)batch * m->in_pad)) ||
                (ierr = malloc_zero(m, &m->Y, (size_t)batch * m->out)) ||
                (ierr = malloc_zero(m, &m->Xs, (size_t)batch * m->in_pad)) ||
                (ierr = malloc_zero(m, &m->Ts, (size_t)batch * m->out)) || (ierr = malloc_zero(m, &m->idx, batch)) ||
                (ierr = malloc_zero(m, &m->loss, 1)) || (ierr = ensure_parts(m, 1))))
    ;
  if (!ierr && !(ierr = malloc_zero(m, &m->wgrad, nlayers))) {
    std::vector<WgradLayer> wl(nlayers);
    for (int l = 0; l < nlayers; l++) {
      const MlpLayer &Ly = m->L[l];
      wl[l] = WgradLayer{Ly.dZt, l == 0 ? m->H0t : m->L[l - 1].Ht, Ly.out, Ly.in_pad, m->wgrad_blocks,
                         Ly.W,   Ly.mW, Ly.vW, Ly.gW, Ly.b, Ly.mb, Ly.vb, Ly.gb, Ly.Wb, Ly.Wtb};
      m->wgrad_blocks += (Ly.out / 64) * (Ly.in_pad / 64) + (Ly.out + 255) / 256;
    }
    if (hipMemcpyAsync(m->wgrad, wl.data(), sizeof(WgradLayer) * nlayers, hipMemcpyHostToDevice, m->stream) != hipSuccess ||
        hipStreamSynchronize(m->stream) != hipSuccess)
      ierr = mfail(SE2W_ERR_HIP, "layer table upload failed");
  }
  if (!ierr) ierr = forward_buffers(m);
  if (!ierr) ierr = refresh_bf16(m);
  if (ierr) {
    se2w_mlp_destroy(m);
    return ierr;
  }
  *out = m;
  return SE2W_OK;
}

int se2w_mlp_param_count(se2w_mlp *m, int64_t *count) {
  if (!m || !count) return mfail(SE2W_ERR_ARG, "null argument");
  int64_t n = 0;
  for (const MlpLayer &Ly : m->L) n += (int64_t)Ly.out * Ly.in + Ly.out;
  *count = n;
  return SE2W_OK;
}

// Copy of a matrix between packed host rows of `in` values and device rows of
// `pad`.  Padded rows go through a host copy of a few MB at a time: a 2D copy
// of pageable memory moves row by row (48 ms for 1024 rows).  Packed copies
// are only queued on the stream.
static int copy_rows(se2w_mlp *m, float *host, float *dev, int rows, int in, int pad, bool to_host) {
  const hipMemcpyKind kind = to_host ? hipMemcpyDeviceToHost : hipMemcpyHostToDevice;
  if (in == pad) {
    MCHK(hipMemcpyAsync(to_host ? host : dev, to_host ? dev : host, sizeof(float) * (size_t)rows * in, kind, m->stream));
    return SE2W_OK;
  }
  const int block = std::min(rows, std::max(1, (1 << 20) / pad));
  std::unique_ptr<float[]> buf(new (std::nothrow) float[(size_t)block * pad]());  // the padding is zero
  if (!buf) return mfail(SE2W_ERR_MEM, "out of host memory");
  for (int r0 = 0; r0 < rows; r0 += block) {
    const int n = std::min(block, rows - r0);
    float *d = dev + (size_t)r0 * pad, *h = host + (size_t)r0 * in;
    if (!to_host)
      for (int r = 0; r < n; r++) memcpy(&buf[(size_t)r * pad], h + (size_t)r * in, sizeof(float) * in);
    MCHK(hipMemcpyAsync(to_host ? buf.get() : d, to_host ? d : buf.get(), sizeof(float) * (size_t)n * pad, kind, m->stream));
    MCHK(hipStreamSynchronize(m->stream));
    if (to_host)
      for (int r = 0; r < n; r++) memcpy(h + (size_t)r * in, &buf[(size_t)r * pad], sizeof(float) * in);
  }
  return SE2W_OK;
}

// Copy between the packed host layout and the device weights, whose rows are
// padded only where the input width is not a multiple of 64 (the first layer).
static int params_copy(se2w_mlp *m, float *host, bool to_host, const std::vector<float *> &dev_w,
                       const std::vector<float *> &dev_b) {
  size_t off = 0;
  for (int l = 0; l < m->nl; l++) {
    const MlpLayer &Ly = m->L[l];
    if (int ierr = copy_rows(m, host + off, dev_w[l], Ly.out, Ly.in, Ly.in_pad, to_host)) return ierr;
    off += (size_t)Ly.out * Ly.in;
    if (int ierr = copy_rows(m, host + off, dev_b[l], 1, Ly.out, Ly.out, to_host)) return ierr;
    off += Ly.out;
  }
  MCHK(hipStreamSynchronize(m->stream));
  return SE2W_OK;
}

int se2w_mlp_get_params(se2w_mlp *m, float *params) {
  if (!m || !params) return mfail(SE2W_ERR_ARG, "null argument");
  MCHK(hipSetDevice(m->device));
  std::vector<float *> w, b;
  for (MlpLayer &Ly : m->L) { w.push_back(Ly.W); b.push_back(Ly.b); }
  return params_copy(m, params, true, w, b);
}

int se2w_mlp_set_params(se2w_mlp *m, const float *params) {
  if (!m || !params) return mfail(SE2W_ERR_ARG, "null argument");
  MCHK(hipSetDevice(m->device));
  std::vector<float *> w, b;
  for (MlpLayer &Ly : m->L) {
    w.push_back(Ly.W);
    b.push_back(Ly.b);
    MCHK(hipMemsetAsync(Ly.mW, 0, sizeof(float) * (size_t)Ly.out * Ly.in_pad, m->stream));
    MCHK(hipMemsetAsync(Ly.vW, 0, sizeof(float) * (size_t)Ly.out * Ly.in_pad, m->stream));
    MCHK(hipMemsetAsync(Ly.mb, 0, sizeof(float) * Ly.out, m->stream));
    MCHK(hipMemsetAsync(Ly.vb, 0, sizeof(float) * Ly.out, m->stream));
  }
  m->t = 0;
  if (int ierr = params_copy(m, (float *)params, false, w, b)) return ierr;
  return refresh_bf16(m);
}

int se2w_mlp_forward(se2w_mlp *m, int32_t n, const float *x, float *y) {
  if (!m || n < 0 || (n > 0 && (!x || !y))) return mfail(SE2W_ERR_ARG, "bad forward arguments");
  MCHK(hipSetDevice(m->device));
  m->fwd_ms = 0.0;
  if (n == 0) return SE2W_OK;
  // a call that ended on an error may have left work that uses the buffers
  MCHK(hipStreamSynchronize(m->stream));
  // Batches in order on the stream, each followed by the download of its
  // chunks; chunk c is handed over once chunk c - kAhead has been copied out,
  // so a batch's products and the next chunks' downloads run while the host
  // copies the earlier ones out.
  const int cr = chunk_rows(m), per = (m->B + cr - 1) / cr;  // chunks of a whole batch
  const int nchunks = n / m->B * per + (n % m->B + cr - 1) / cr;
  const int xr = piece_rows(m);
  const bool split = xr < m->B;  // batches of several input pieces
  // workgroups of a row: a piece of long rows has few of them (256 rows of
  // 16384: 0.55 ms, with one workgroup a row 2.9)
  const int row_blocks = std::min(64, (m->in_pad + 1023) / 1024);
  long piece = 0;
  auto enqueue = [&](int c) -> int {
    const int b = c / per, s = b % (kAhead + 1), r0 = b * m->B, k = std::min(m->B, n - r0);
    const int c0 = (c % per) * cr, rows = std::min(cr, k - c0);
    float *slot = m->y_host + (size_t)(c % kAhead) * cr * m->out;
    // few rows are written to the pinned chunk by the last product itself
    const bool direct = k <= 16;
    if (c % per == 0) {
      const int M = k <= 16 ? 16 : k <= 32 ? 32 : round_up(k, 64);
      for (int p0 = 0; p0 < k; p0 += xr, piece++) {
        const int slot_x = piece % (kAhead + 1), rows_x = std::min(xr, k - p0);
        const bool last = p0 + xr >= k;
        // Whole batches: the chunks of the batch that had the slot are copied out.
        if (split && piece > kAhead) MCHK(hipEventSynchronize(m->x_read[slot_x]));
        float *xh = m->x_host + (size_t)slot_x * xr * m->in;
        memcpy(xh, x + (size_t)(r0 + p0) * m->in, sizeof(float) * (size_t)rows_x * m->in);
        if (last) MCHK(hipEventRecord(m->f0[s], m->stream));
        hipLaunchKernelGGL(k_rows, dim3(last ? M - p0 : rows_x, row_blocks), dim3(128), 0, m->stream, (const float *)xh, rows_x, p0,
                           m->in, m->in_pad, m->H0);
        if (split) MCHK(hipEventRecord(m->x_read[slot_x], m->stream));
      }
      if (int ierr = forward(m, M, nullptr, direct ? slot : m->Y)) return ierr;
      MCHK(hipEventRecord(m->f1[s], m->stream));
    }
    if (!direct)
      hipLaunchKernelGGL(k_to_host, dim3(128), dim3(256), 0, m->stream, (const floatx4 *)(m->Y + (size_t)c0 * m->out),
                         (floatx4 *)slot, (long)rows * m->out / 4);
    MCHK(hipEventRecord(m->y_up[c % kAhead], m->stream));
    return SE2W_OK;
  };
  for (int c = 0; c < std::min(kAhead, nchunks); c++)
    if (int ierr = enqueue(c)) return ierr;
  for (int c = 0; c < nchunks; c++) {
    const int b = c / per, s = b % (kAhead + 1), r0 = b * m->B, k = std::min(m->B, n - r0);
    const int c0 = (c % per) * cr, rows = std::min(cr, k - c0);
    MCHK(hipEventSynchronize(m->y_up[c % kAhead]));
    memcpy(y + (size_t)(r0 + c0) * m->out, m->y_host + (size_t)(c % kAhead) * cr * m->out,
           sizeof(float) * (size_t)rows * m->out);
    if (c % per == 0) {
      float ms = 0.f;
      MCHK(hipEventElapsedTime(&ms, m->f0[s], m->f1[s]));
      m->fwd_ms += ms;
    }
    if (c + kAhead < nchunks)
      if (int ierr = enqueue(c + kAhead)) return ierr;
  }
  return SE2W_OK;
}

int se2w_mlp_gradient(se2w_mlp *m, int32_t n, const float *x, const float *target, float *loss, float *grad) {
  if (!m || !x || !target || !grad) return mfail(SE2W_ERR_ARG, "null argument");
  if (n != m->B) return mfail(SE2W_ERR_ARG, "gradient batch must have %d rows", m->B);
  MCHK(hipSetDevice(m->device));
  if (int ierr = stage_batch(m, n, x, target)) return ierr;
  const LossArgs la{m->Ts, m->idx, m->part};
  if (int ierr = forward(m, m->B, &la, nullptr)) return ierr;
  if (int ierr = backward(m)) return ierr;
  hipLaunchKernelGGL(k_sum_parts, dim3(1), dim3(256), 0, m->stream, (const double *)m->part, (long)m->nparts,
                     1.0 / ((double)m->B * m->out), m->loss);
  if (int ierr = weight_gradients(m)) return ierr;
  double l = 0.0;
  MCHK(hipMemcpyAsync(&l, m->loss, sizeof(double), hipMemcpyDeviceToHost, m->stream));
  std::vector<float *> w, b;
  for (MlpLayer &Ly : m->L) { w.push_back(Ly.gW); b.push_back(Ly.gb); }
  if (int ierr = params_copy(m, grad, true, w, b)) return ierr;
  if (loss) *loss = (float)l;
  return SE2W_OK;
}

int se2w_mlp_adam_step(se2w_mlp *m, const float *grad, float lr) {
  if (!m || !grad) return mfail(SE2W_ERR_ARG, "null argument");
  MCHK(hipSetDevice(m->device));
  std::vector<float *> w, b;
  for (MlpLayer &Ly : m->L) { w.push_back(Ly.gW); b.push_back(Ly.gb); }
  if (int ierr = params_copy(m, (float *)grad, false, w, b)) return ierr;
  if (int ierr = adam(m, lr)) return ierr;
  MCHK(hipStreamSynchronize(m->stream));
  return SE2W_OK;
}

int se2w_mlp_set_data(se2w_mlp *m, int32_t n, const float *x, const float *target) {
  if (!m || n < m->B || !x || !target) return mfail(SE2W_ERR_ARG, "need at least one batch of data");
  MCHK(hipSetDevice(m->device));
  if (m->X) hipFree(m->X);
  if (m->T) hipFree(m->T);
  m->X = m->T = nullptr;
  m->ndata = 0;
  MCHK(hipMalloc(&m->X, sizeof(float) * (size_t)n * m->in_pad));
  MCHK(hipMalloc(&m->T, sizeof(float) * (size_t)n * m->out));
  if (int ierr = copy_rows(m, const_cast<float *>(x), m->X, n, m->in, m->in_pad, false)) return ierr;
  MCHK(hipMemcpyAsync(m->T, target, sizeof(float) * (size_t)n * m->out, hipMemcpyHostToDevice, m->stream));
  MCHK(hipStreamSynchronize(m->stream));
  m->ndata = n;
  return SE2W_OK;
}

int se2w_mlp_train(se2w_mlp *m, int32_t epochs, float lr, uint64_t shuffle_seed, float *epoch_loss) {
  if (!m || epochs < 1 || !(lr > 0.f)) return mfail(SE2W_ERR_ARG, "bad training arguments");
  if (m->ndata < m->B) return mfail(SE2W_ERR_STATE, "set the training data first");
  MCHK(hipSetDevice(m->device));
  const int nb = m->ndata / m->B;
  const size_t np = (size_t)nb * m->B;
  if (int ierr = ensure_parts(m, nb)) return ierr;
  if (int ierr = ensure_perm(m, np)) return ierr;
  std::vector<int> perm(m->ndata);
  double *d_loss = nullptr;
  if (hipMalloc(&d_loss, sizeof(double) * epochs) != hipSuccess) return mfail(SE2W_ERR_MEM, "hipMalloc failed");
  int ierr = SE2W_OK;
  uint64_t rng = shuffle_seed;
  if (hipEventRecord(m->e0, m->stream) != hipSuccess) ierr = mfail(SE2W_ERR_HIP, "training setup failed");
  for (int e = 0; e < epochs && !ierr; e++) {
    for (int i = 0; i < m->ndata; i++) perm[i] = i;
    for (int i = m->ndata - 1; i > 0; i--) {  // Fisher-Yates
      const int j = (int)(uniform01(rng) * (i + 1));
      std::swap(perm[i], perm[j]);
    }
    // The permutation goes up on the stream, so the host may run an epoch
    // ahead; the pinned half is free again once its previous copy has gone
    // up (the device half is ordered by the stream).
    const int half = e & 1;
    int *hp = m->perm_host + half * m->perm_cap, *dp = m->perm_dev + half * m->perm_cap;
    if (e >= 2 && hipEventSynchronize(m->perm_up[half]) != hipSuccess) {
      ierr = mfail(SE2W_ERR_HIP, "permutation upload failed");
      break;
    }
    memcpy(hp, perm.data(), sizeof(int) * np);
    if (hipMemcpyAsync(dp, hp, sizeof(int) * np, hipMemcpyHostToDevice, m->stream) != hipSuccess ||
        hipEventRecord(m->perm_up[half], m->stream) != hipSuccess) {
      ierr = mfail(SE2W_ERR_HIP, "permutation upload failed");
      break;
    }
    for (int k = 0; k < nb && !ierr; k++) {
      const int *rows = dp + (size_t)k * m->B;
      hipLaunchKernelGGL(k_gather, dim3(m->B), dim3(128), 0, m->stream, (const float *)m->X, rows, m->B, m->in_pad,
                         m->H0, m->H0t);
      const LossArgs la{m->T, rows, m->part + (size_t)k * m->nparts};
      if ((ierr = forward(m, m->B, &la, nullptr)) || (ierr = backward(m))) break;
      // cosine decay: lr_s = lr (1 + cos(pi s / S)) / 2 over the S steps of this call
      const double frac = (double)(e * nb + k) / ((double)epochs * nb);
      const float lr_s = m->cosine ? (float)(0.5 * lr * (1.0 + std::cos(3.14159265358979323846 * frac))) : lr;
      ierr = weight_update(m, lr_s);
    }
    // the epoch's loss is the mean of its batch losses
    hipLaunchKernelGGL(k_sum_parts, dim3(1), dim3(256), 0, m->stream, (const double *)m->part, (long)nb * m->nparts,
                       1.0 / ((double)m->B * m->out * nb), d_loss + e);
  }
  if (!ierr) {
    if (hipEventRecord(m->e1, m->stream) != hipSuccess || hipStreamSynchronize(m->stream) != hipSuccess) {
      ierr = mfail(SE2W_ERR_HIP, "training failed: %s", hipGetErrorString(hipGetLastError()));
    } else {
      float ms = 0.f;
      hipEventElapsedTime(&ms, m->e0, m->e1);
      m->train_ms = ms;
      if (epoch_loss) {
        std::vector<double> l(epochs);
        hipMemcpy(l.data(), d_loss, sizeof(double) * epochs, hipMemcpyDeviceToHost);
        for (int e = 0; e < epochs; e++) epoch_loss[e] = (float)l[e];
      }
    }
  }
  hipStreamSynchronize(m->stream);
  hipFree(d_loss);
  return ierr;
}

int se2w_mlp_set_lr_schedule(se2w_mlp *m, int32_t cosine) {
  if (!m) return mfail(SE2W_ERR_ARG, "null argument");
  m->cosine = cosine != 0;
  return SE2W_OK;
}

int se2w_mlp_set_weight_decay(se2w_mlp *m, float wd) {
  if (!m || !(wd >= 0.f)) return mfail(SE2W_ERR_ARG, "bad weight decay");
  m->weight_decay = wd;
  return SE2W_OK;
}

int se2w_mlp_get_timing(se2w_mlp *m, double *train_ms, double *forward_ms) {
  if (!m) return mfail(SE2W_ERR_ARG, "null argument");
  if (train_ms) *train_ms = m->train_ms;
  if (forward_ms) *forward_ms = m->fwd_ms;
  return SE2W_OK;
}

int se2w_mlp_destroy(se2w_mlp *m) {
  if (!m) return SE2W_OK;
  hipSetDevice(m->device);
  if (m->stream) hipStreamSynchronize(m->stream);
  for (void *p : m->allocs) hipFree(p);
  if (m->X) hipFree(m->X);
  if (m->T) hipFree(m->T);
  if (m->x_host) hipHostFree(m->x_host);
  if (m->y_host) hipHostFree(m->y_host);
  for (hipEvent_t e : m->y_up)
    if (e) hipEventDestroy(e);
  for (hipEvent_t e : m->x_read)
    if (e) hipEventDestroy(e);
  for (int s = 0; s <= kAhead; s++) {
    if (m->f0[s]) hipEventDestroy(m->f0[s]);
    if (m->f1[s]) hipEventDestroy(m->f1[s]);
  }
  if (m->part) hipFree(m->part);
  if (m->perm_dev) hipFree(m->perm_dev);
  if (m->perm_host) hipHostFree(m->perm_host);
  for (hipEvent_t e : m->perm_up)
    if (e) hipEventDestroy(e);
  if (m->e0) hipEventDestroy(m->e0);
  if (m->e1) hipEventDestroy(m->e1);
  if (m->stream) hipStreamDestroy(m->stream);
  delete m;
  return SE2W_OK;
}

}  // extern "C"
