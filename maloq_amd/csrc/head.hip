// The Fock irreps output head in one pass each way (gfx950): scalar linear, gate,
// per-degree linears and the label gather forward; all their gradients but the
// scalar linear's weights backward.  Reference: Fock_Irreps_Head.process
// (helm/esen_osh.py:894-1052); the formulas are those of irreps_head.hip.
//
// What bounds it: the fp32 MFMA (16x16x4; 107 k products per row at lmax 4, C 128) and
// the exchange through LDS between them, in tiles of 32 rows whose weights each
// workgroup reads again, with one workgroup of eight waves per compute unit.  HBM is
// only the floor: the embeddings (d C floats a row) are read once forward, read and
// their gradient written once backward (20 000 rows at C 128: 150 us at the rate of a
// copy); gated copies, per-degree copies and the outputs before the gather stay in
// registers and LDS.  Forward and backward of those 20 000 rows, 56 copies, as layers
// (gate kernels, a library product and its copies per degree) 2011 us, so 690; 8 rows
// (launches) 1161 and 271.
//
// A workgroup owns 32 rows.  MFMA lanes: i = lane % 16, q = lane / 16; A
// holds row i, B column i, both at k = q; the accumulator's register r is row
// 4 q + r, column i.  Where k runs along memory, step t of block j is k = 16 j +
// 4 q + t, so that a lane reads 16 bytes for four steps.
#include <type_traits>
#include <utility>

#include "common.h"
#include "../../include/maloq_hip.h"

namespace maloq {
namespace head {

constexpr int ROWS = 32;
constexpr int NT = 512, NW = 8;  // forward workgroup
constexpr int MAXL = 6;
constexpr int ZMAX = 256;   // widest row of the per-degree outputs
constexpr int MULMAX = 32;  // most copies of a degree

typedef float f4 __attribute__((ext_vector_type(4)));

struct Args {
  const float* x;           // [R, d, C]
  int64_t R;
  int L, W;                 // W = (1 + L) C
  float scale;              // of every linear: 1 / sqrt(C)
  const float* ws;          // [C, W] scalar linear
  const float* bs;          // [W] or null
  const float* wl[MAXL + 1];  // [C, mul[l]]
  int mul[MAXL + 1], zoff[MAXL + 1];
  const float* b0;          // [mul[0]] or null
  float cst;
  int act;
  float* s;                 // [R, W] scalars: written forward (nullable), read backward
  int Zw, T;
  const int32_t* src;       // forward: label column -> output column (-1: zero)
  const float* sign;
  float* out;               // [R, T]
  // backward
  const float* dout;        // [R, T]
  const int32_t *ptr, *cols;  // CSR of the gather's transpose
  const float* csign;
  float *dx, *ds;           // [R, d, C], [R, W]
  float* part;              // [workgroups, pw]: dW_l [C, mul[l]] at woff[l], then db0
  int woff[MAXL + 2];
  int pw;
};

__device__ __forceinline__ f4 mfma(float a, float b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float act_f(int act, float z) {
  return act ? tanhf(fabsf(z)) : 1.0f / (1.0f + expf(-z));
}
__device__ __forceinline__ float act_df(int act, float z, float f) {
  return act ? (1.0f - f * f) * (z > 0.f ? 1.0f : (z < 0.f ? -1.0f : 0.f)) : f * (1.0f - f);
}
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <class F, int... Is>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, Is...>) {
  (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// C = 16 NJ
template <int NJ>
__global__ __launch_bounds__(NT, 2) void head_fwd_kernel(Args a) {
  constexpr int C = 16 * NJ, GP = C + 4;
  __shared__ alignas(16) float G[ROWS * GP];  // a degree's gate factors (degree 0: its inputs)
  __shared__ alignas(16) float X0[ROWS * GP];  // the l = 0 rows
  __shared__ float Z[ROWS * ZMAX];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, i = lane & 15, q = lane >> 4;
  const int64_t row0 = static_cast<int64_t>(blockIdx.x) * ROWS;
  const int d = (a.L + 1) * (a.L + 1);
  const float* xr[2];  // this lane's rows (past the end: the last one, not stored)
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    const int64_t r = row0 + 16 * rt + i;
    xr[rt] = a.x + (r < a.R ? r : a.R - 1) * d * C + 4 * q;
  }
  for (int u = tid; u < ROWS * NJ * 4; u += NT) {
    const int row = u / (NJ * 4), c4 = u % (NJ * 4) * 4;
    const int64_t r = row0 + row < a.R ? row0 + row : a.R - 1;
    *reinterpret_cast<f4*>(X0 + row * GP + c4) = *reinterpret_cast<const f4*>(a.x + r * d * C + c4);
  }
  for (int l = 0; l <= a.L; ++l) {
    __syncthreads();  // the last degree's factors are read
    for (int nt = wave; nt < NJ; nt += NW) {
      const int c = 16 * nt + i, col = l * C + c;
      // two sums of half the terms each: shorter MFMA chains, less rounding
      f4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}}, acc2[2] = {acc[0], acc[0]};
      float b[NJ][4];
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int t = 0; t < 4; ++t) b[j][t] = a.ws[static_cast<int64_t>(16 * j + 4 * q + t) * a.W + col];
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const f4 v0 = *reinterpret_cast<const f4*>(X0 + i * GP + 16 * j + 4 * q);
        const f4 v1 = *reinterpret_cast<const f4*>(X0 + (16 + i) * GP + 16 * j + 4 * q);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          f4(&s2)[2] = j & 1 ? acc2 : acc;
          s2[0] = mfma(v0[t], b[j][t], s2[0]);
          s2[1] = mfma(v1[t], b[j][t], s2[1]);
        }
      }
      const float bias = a.bs ? a.bs[col] : 0.f;
#pragma unroll
      for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = 16 * rt + 4 * q + r;
          const float z = fmaf(acc[rt][r] + acc2[rt][r], a.scale, bias);
          if (a.s && row0 + row < a.R) a.s[(row0 + row) * a.W + col] = z;
          G[row * GP + c] = l == 0 ? z : a.cst * act_f(a.act, z);
        }
    }
    __syncthreads();
    const int ml = a.mul[l], nm = 2 * l + 1, units = (ml + 15) / 16 * nm;
    for (int u = wave; u < units; u += NW) {
      const int m = u % nm, v = u / nm * 16 + i;
      float b[NJ][4];
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int t = 0; t < 4; ++t) b[j][t] = v < ml ? a.wl[l][(16 * j + 4 * q + t) * ml + v] : 0.f;
      f4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}}, acc2[2] = {acc[0], acc[0]};
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) {
        const float* g = G + (16 * rt + i) * GP + 4 * q;
        const float* xm = xr[rt] + (l * l + m) * C;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          f4 v4 = *reinterpret_cast<const f4*>(g + 16 * j);
          if (l > 0) v4 *= *reinterpret_cast<const f4*>(xm + 16 * j);
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            f4& sum = (j & 1 ? acc2 : acc)[rt];
            sum = mfma(v4[t], b[j][t], sum);
          }
        }
      }
      if (v < ml) {
        const float b0 = l == 0 && a.b0 ? a.b0[v] : 0.f;
#pragma unroll
        for (int rt = 0; rt < 2; ++rt)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            Z[(16 * rt + 4 * q + r) * a.Zw + a.zoff[l] + m * ml + v] = fmaf(acc[rt][r] + acc2[rt][r], a.scale, b0);
      }
    }
  }
  __syncthreads();
  for (int r = wave; r < ROWS && row0 + r < a.R; r += NW)
    for (int t = lane; t < a.T; t += 64) {
      const int sc = a.src[t];
      a.out[(row0 + r) * a.T + t] = sc >= 0 ? a.sign[t] * Z[r * a.Zw + sc] : 0.f;
    }
}

// A wave owns a tile of 16 channels for everything but the last product, so that
// a degree's rows pass through LDS of its own: embeddings in, their gradient out.
// (Eight waves for 96 and 128 channels: two tiles in each of four waves spilled
// 300 bytes per lane and took twice as long.)  Persistent over row tiles: the per-degree weight gradients
// stay in its accumulators and are written once.
constexpr int bwd_waves(int nj) { return nj > 4 ? 8 : 4; }
template <int NJ, int L>
__global__ __launch_bounds__(64 * bwd_waves(NJ), 16 / bwd_waves(NJ)) void head_bwd_kernel(Args a) {
  constexpr int NW = bwd_waves(NJ), TPW = (NJ + NW - 1) / NW, C = 16 * NJ, TP = 20, d = (L + 1) * (L + 1);
  constexpr int NN = MULMAX / 16, NK = MULMAX / 4, W = (L + 1) * C;
  __shared__ alignas(16) float X[NJ * ROWS * TP];  // [channel tile][row][16]: embeddings, then gradients
  __shared__ alignas(16) float G[NJ * ROWS * TP];  // gate factors (degree 0: its inputs)
  __shared__ float Z[ROWS * (ZMAX + 1)];           // output gradients before the gather
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, i = lane & 15, q = lane >> 4;
  const int ZP = a.Zw | 1;
  f4 dw[L + 1][TPW][NN];
#pragma unroll
  for (int l = 0; l <= L; ++l)
#pragma unroll
    for (int k = 0; k < TPW; ++k)
#pragma unroll
      for (int n = 0; n < NN; ++n) dw[l][k][n] = f4{0.f, 0.f, 0.f, 0.f};
  float db0 = 0.f;
  const int64_t ntiles = (a.R + ROWS - 1) / ROWS;
  for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const int64_t row0 = tile * ROWS;
    const int nrow = static_cast<int>(a.R - row0 < ROWS ? a.R - row0 : ROWS);
    __syncthreads();  // the last tile's Z and X are read
    for (int r = wave; r < ROWS; r += NW)
      for (int z = lane; z < a.Zw; z += 64) {
        float v = 0.f;
        if (r < nrow)
          for (int k = a.ptr[z]; k < a.ptr[z + 1]; ++k)
            v = fmaf(a.csign[k], a.dout[(row0 + r) * a.T + a.cols[k]], v);
        Z[r * ZP + z] = v;
      }
    __syncthreads();
    if (tid < a.mul[0])
      for (int r = 0; r < nrow; ++r) db0 += Z[r * ZP + a.zoff[0] + tid];
    f4 dx0[TPW][2];
#pragma unroll
    for (int k = 0; k < TPW; ++k) dx0[k][0] = dx0[k][1] = f4{0.f, 0.f, 0.f, 0.f};
    static_for<L + 1>([&](auto LC) {
      constexpr int l = decltype(LC)::value;
      const int ml = a.mul[l];
      f4 dsum[TPW][2];
      float wt[TPW][NK];  // W_l [channel i][copy 4 kb + q]
#pragma unroll
      for (int k = 0; k < TPW; ++k) {
        const int nt = wave * TPW + k;
        dsum[k][0] = dsum[k][1] = f4{0.f, 0.f, 0.f, 0.f};
        if (nt >= NJ) continue;
#pragma unroll
        for (int kb = 0; kb < NK; ++kb) {
          const int v = 4 * kb + q;
          wt[k][kb] = v < ml ? a.wl[l][(16 * nt + i) * ml + v] : 0.f;
        }
        // four lanes a row, 16 rows at a time
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int row = 16 * h + (lane >> 2), c4 = 4 * (lane & 3);
          f4 z = {0.f, 0.f, 0.f, 0.f};
          if (row < nrow) {
            z = *reinterpret_cast<const f4*>(a.s + (row0 + row) * W + l * C + 16 * nt + c4);
            if (l > 0)
#pragma unroll
              for (int t = 0; t < 4; ++t) z[t] = a.cst * act_f(a.act, z[t]);
          }
          *reinterpret_cast<f4*>(G + (nt * ROWS + row) * TP + c4) = z;
        }
      }
      wave_sync();
      for (int m = 0; m < 2 * l + 1; ++m) {
        const int zc = a.zoff[l] + m * ml;
#pragma unroll
        for (int k = 0; k < TPW; ++k) {
          const int nt = wave * TPW + k;
          if (nt >= NJ) continue;
          float* Xt = X + nt * ROWS * TP;
          const float* Gt = G + nt * ROWS * TP;
          if (l > 0) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const int row = 16 * h + (lane >> 2), c4 = 4 * (lane & 3);
              f4 v = {0.f, 0.f, 0.f, 0.f};
              if (row < nrow)
                v = *reinterpret_cast<const f4*>(a.x + ((row0 + row) * d + l * l + m) * C + 16 * nt + c4);
              *reinterpret_cast<f4*>(Xt + row * TP + c4) = v;
            }
            wave_sync();
          }
          // gradient of the gated rows
          f4 dg[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
          for (int kb = 0; kb < NK; ++kb) {
            if (4 * kb >= ml) break;
            const int v = 4 * kb + q;
#pragma unroll
            for (int rt = 0; rt < 2; ++rt)
              dg[rt] = mfma(v < ml ? Z[(16 * rt + i) * ZP + zc + v] : 0.f, wt[k][kb], dg[rt]);
          }
          dg[0] *= a.scale;
          dg[1] *= a.scale;
          // weight gradient: gated rows (transposed) x output gradients
#pragma unroll
          for (int kk = 0; kk < ROWS / 4; ++kk) {
            const int row = 4 * kk + q;
            const float g = Gt[row * TP + i] * (l > 0 ? Xt[row * TP + i] : 1.0f);
#pragma unroll
            for (int n = 0; n < NN; ++n) {
              if (16 * n >= ml) break;
              const int v = 16 * n + i;
              dw[l][k][n] = mfma(g, v < ml ? Z[row * ZP + zc + v] : 0.f, dw[l][k][n]);
            }
          }
          if (l == 0) {
            dsum[k][0] = dg[0];
            dsum[k][1] = dg[1];
            continue;
          }
          wave_sync();
#pragma unroll
          for (int rt = 0; rt < 2; ++rt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              float* xv = Xt + (16 * rt + 4 * q + r) * TP + i;
              dsum[k][rt][r] = fmaf(dg[rt][r], *xv, dsum[k][rt][r]);
              *xv = dg[rt][r] * Gt[(16 * rt + 4 * q + r) * TP + i];
            }
          wave_sync();
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int row = 16 * h + (lane >> 2), c4 = 4 * (lane & 3);
            if (row < nrow)
              *reinterpret_cast<f4*>(a.dx + ((row0 + row) * d + l * l + m) * C + 16 * nt + c4) =
                  *reinterpret_cast<const f4*>(Xt + row * TP + c4);
          }
          wave_sync();
        }
      }
      // gradient of this degree's scalars, to memory and (all waves') to X
#pragma unroll
      for (int k = 0; k < TPW; ++k) {
        const int nt = wave * TPW + k;
        if (nt >= NJ) continue;
#pragma unroll
        for (int rt = 0; rt < 2; ++rt)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int row = 16 * rt + 4 * q + r;
            float v = 0.f;
            if (row < nrow) {
              const int64_t at = (row0 + row) * W + l * C + 16 * nt + i;
              v = dsum[k][rt][r];
              if (l > 0) {
                const float z = a.s[at];
                v *= a.cst * act_df(a.act, z, act_f(a.act, z));
              }
              a.ds[at] = v;
            }
            X[(nt * ROWS + row) * TP + i] = v;
          }
      }
      __syncthreads();
#pragma unroll
      for (int k = 0; k < TPW; ++k) {
        const int nt = wave * TPW + k;
        if (nt >= NJ) continue;
        const float* w = a.ws + static_cast<int64_t>(16 * nt + i) * W + l * C + 4 * q;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const f4 b = *reinterpret_cast<const f4*>(w + 16 * j);
#pragma unroll
          for (int rt = 0; rt < 2; ++rt) {
            const f4 v = *reinterpret_cast<const f4*>(X + (j * ROWS + 16 * rt + i) * TP + 4 * q);
#pragma unroll
            for (int t = 0; t < 4; ++t) dx0[k][rt] = mfma(v[t], b[t], dx0[k][rt]);
          }
        }
      }
      __syncthreads();
    });
#pragma unroll
    for (int k = 0; k < TPW; ++k) {
      const int nt = wave * TPW + k;
      if (nt >= NJ) continue;
#pragma unroll
      for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = 16 * rt + 4 * q + r;
          if (row < nrow) a.dx[(row0 + row) * d * C + 16 * nt + i] = dx0[k][rt][r] * a.scale;
        }
    }
  }
  float* part = a.part + static_cast<int64_t>(blockIdx.x) * a.pw;
#pragma unroll
  for (int l = 0; l <= L; ++l)
#pragma unroll
    for (int k = 0; k < TPW; ++k) {
      const int nt = wave * TPW + k;
      if (nt >= NJ) continue;
#pragma unroll
      for (int n = 0; n < NN; ++n) {
        const int v = 16 * n + i;
        if (v >= a.mul[l]) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) part[a.woff[l] + (16 * nt + 4 * q + r) * a.mul[l] + v] = dw[l][k][n][r];
      }
    }
  if (tid < a.mul[0]) part[a.woff[L + 1] + tid] = db0;
}

// out[i] = sum over the workgroups' partials, in order
// (times scale for the first nw: the weights').  Loads ahead of the sums, which are
// one chain.
__global__ void head_reduce_kernel(const float* __restrict__ part, int nwg, int pw, int nw, float scale,
                                   float* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= pw) return;
  float s = 0.f;
  int g = 0;
  for (; g + 16 <= nwg; g += 16) {
    float v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) v[k] = part[static_cast<int64_t>(g + k) * pw + i];
#pragma unroll
    for (int k = 0; k < 16; ++k) s += v[k];
  }
  for (; g < nwg; ++g) s += part[static_cast<int64_t>(g) * pw + i];
  out[i] = i < nw ? s * scale : s;
}

static int workgroups(int64_t rows, int c) {
  const int64_t tiles = (rows + ROWS - 1) / ROWS, most = 16 / bwd_waves(c / 16) * device_cus();
  return static_cast<int>(tiles < most ? tiles : most);
}

static int setup(Args& a, int64_t rows, int lmax, int c, const float* const* wl, const int* mul) {
  a.R = rows;
  a.L = lmax;
  a.W = (lmax + 1) * c;
  int z = 0, w = 0;
  for (int l = 0; l <= lmax; ++l) {
    MALOQ_REQUIRE(mul[l] >= 0 && mul[l] <= MULMAX && (mul[l] == 0 || wl == nullptr || wl[l]), "bad copies of degree %d", l);
    a.wl[l] = wl ? wl[l] : nullptr;
    a.mul[l] = mul[l];
    a.zoff[l] = z;
    a.woff[l] = w;
    z += (2 * l + 1) * mul[l];
    w += c * mul[l];
  }
  a.woff[lmax + 1] = w;
  a.pw = w + mul[0];
  a.Zw = z;
  return MALOQ_OK;
}

static bool supported(int lmax, int c, const int* mul) {
  if (lmax < 0 || lmax > MAXL || c <= 0 || c % 32 || c > 128) return false;
  int z = 0;
  for (int l = 0; l <= lmax; ++l) {
    if (mul[l] < 0 || mul[l] > MULMAX) return false;
    z += (2 * l + 1) * mul[l];
  }
  return z > 0 && z <= ZMAX && (lmax == 2 || lmax == 4 || lmax == 6);
}

}  // namespace head
}  // namespace maloq

using namespace maloq;
using namespace maloq::head;

extern "C" int maloq_irreps_head_supported(int lmax, int c, const int* mul) { return supported(lmax, c, mul) ? 1 : 0; }

extern "C" int maloq_irreps_head_fwd(const float* x, int64_t num_rows, int lmax, int c, const float* ws,
                                     const float* bs, const float* const* wl, const int* mul, const float* b0,
                                     float scale, float cst, int act, const int32_t* src, const float* sign, int t,
                                     float* scalars, float* out, void* stream) {
  MALOQ_REQUIRE(mul && supported(lmax, c, mul), "unsupported head shape");
  MALOQ_REQUIRE(num_rows >= 0 && t >= 0 && (act == 0 || act == 1), "bad arguments");
  if (num_rows == 0 || t == 0) return MALOQ_OK;
  MALOQ_REQUIRE(x && ws && wl && src && sign && out, "null pointer");
  Args a{};
  if (setup(a, num_rows, lmax, c, wl, mul)) return MALOQ_EINVAL;
  a.x = x; a.scale = scale; a.ws = ws; a.bs = bs; a.b0 = b0; a.cst = cst; a.act = act; a.s = scalars;
  a.src = src; a.sign = sign; a.T = t; a.out = out;
  const int64_t grid = (num_rows + ROWS - 1) / ROWS;
  MALOQ_REQUIRE(grid < (int64_t(1) << 31), "too many rows");
  const dim3 g(static_cast<unsigned>(grid)), b(NT);
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (c / 16) {
    case 2: hipLaunchKernelGGL(head_fwd_kernel<2>, g, b, 0, s, a); break;
    case 4: hipLaunchKernelGGL(head_fwd_kernel<4>, g, b, 0, s, a); break;
    case 6: hipLaunchKernelGGL(head_fwd_kernel<6>, g, b, 0, s, a); break;
    default: hipLaunchKernelGGL(head_fwd_kernel<8>, g, b, 0, s, a); break;
  }
  return check_launch("head_fwd_kernel");
}

extern "C" int64_t maloq_irreps_head_partials_floats(int64_t num_rows, int lmax, int c, const int* mul) {
  Args a{};
  if (num_rows < 0 || !mul || !supported(lmax, c, mul) || setup(a, num_rows, lmax, c, nullptr, mul)) return -1;
  return static_cast<int64_t>(workgroups(num_rows, c) < 1 ? 1 : workgroups(num_rows, c)) * a.pw;
}

template <int NJ>
static void launch_bwd(int lmax, const dim3& g, hipStream_t s, const Args& a) {
  switch (lmax) {
    case 2: hipLaunchKernelGGL((head_bwd_kernel<NJ, 2>), g, dim3(64 * bwd_waves(NJ)), 0, s, a); break;
    case 4: hipLaunchKernelGGL((head_bwd_kernel<NJ, 4>), g, dim3(64 * bwd_waves(NJ)), 0, s, a); break;
    default: hipLaunchKernelGGL((head_bwd_kernel<NJ, 6>), g, dim3(64 * bwd_waves(NJ)), 0, s, a); break;
  }
}

extern "C" int maloq_irreps_head_bwd(const float* x, int64_t num_rows, int lmax, int c, const float* ws,
                                     const float* const* wl, const int* mul, float scale, float cst, int act,
                                     const float* scalars,
                                     const float* grad_out, int t, const int32_t* ptr, const int32_t* cols,
                                     const float* csign, float* partials, float* grad_x, float* grad_scalars,
                                     float* grad_wl, void* stream) {
  MALOQ_REQUIRE(mul && supported(lmax, c, mul), "unsupported head shape");
  MALOQ_REQUIRE(num_rows > 0 && t > 0 && (act == 0 || act == 1), "bad arguments");
  MALOQ_REQUIRE(x && ws && wl && scalars && grad_out && ptr && cols && csign && partials && grad_x && grad_scalars &&
                grad_wl, "null pointer");
  Args a{};
  if (setup(a, num_rows, lmax, c, wl, mul)) return MALOQ_EINVAL;
  a.x = x; a.scale = scale; a.ws = ws; a.cst = cst; a.act = act; a.s = const_cast<float*>(scalars); a.T = t;
  a.dout = grad_out; a.ptr = ptr; a.cols = cols; a.csign = csign; a.dx = grad_x; a.ds = grad_scalars;
  a.part = partials;
  const int nwg = workgroups(num_rows, c);
  const dim3 g(static_cast<unsigned>(nwg));
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (c / 16) {
    case 2: launch_bwd<2>(lmax, g, s, a); break;
    case 4: launch_bwd<4>(lmax, g, s, a); break;
    case 6: launch_bwd<6>(lmax, g, s, a); break;
    default: launch_bwd<8>(lmax, g, s, a); break;
  }
  int rc = check_launch("head_bwd_kernel");
  if (rc) return rc;
  hipLaunchKernelGGL(head_reduce_kernel, dim3((a.pw + 63) / 64), dim3(64), 0, s, partials, nwg, a.pw,
                     a.woff[lmax + 1], a.scale, grad_wl);
  return check_launch("head_reduce_kernel");
}
