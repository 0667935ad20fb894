// Router GEMMs of fp32 MoC layers (moc/api.py:383-388 of the reference: logits =
// F.linear(z, router) with the softmax / exp after it, and its autograd), the
// fp32 counterparts of moc_router.hip.
//
// All three products have at most 32 routes on one side, so what bounds them is
// one pass over z (and dz) through HBM; a library GEMM tiles for a wide second
// side instead (its drouter product ran 38.6 us for 33.5 MB of z).  The products
// run on the fp32 matrix instruction (v_mfma_f32_16x16x4_f32: 2 N Z K flops each,
// a fifth of the streaming time at 16 routes), operands are read with 16-byte
// accesses in the order the instruction wants them (a contraction may be taken
// in any order if both operands agree: step v of four takes entries 4 q + v), sums
// are fp32 and in a fixed order.  N 8192, Z 1024, 16 routes: forward with the
// softmax 14.4 -> 8.6 us, dz and drouter 50.5 -> 16.9 us (library GEMMs before).
// K % 4 == 0, K <= 32, Z % 64 == 0.

#include "moc_kernels.h"
#include "moc_mfma.h"

namespace moc {
namespace router {

using mfma::Buf;
using mfma::f32x4;
using mfma::kOffNone;

namespace {

__device__ __forceinline__ f32x4 load4(const Buf& b, uint32_t off) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(b.r, static_cast<int>(off), 0, 0));
}
// 16 x 16 x 16 product: lane (i, q) holds entries 4 q + {0..3} of row i of either operand
__device__ __forceinline__ f32x4 mma4(f32x4 a, f32x4 b, f32x4 c) {
#pragma unroll
  for (int v = 0; v < 4; ++v) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[v], b[v], c, 0, 0, 0);
  return c;
}

// ---------------------------------------------------------------------------
// out[t, k] = activation_k(sum_z z[t, z] router[k, z]).  Workgroup: 16 tokens, 4
// waves; wave w sums the 64-wide z chunks w, w + 4, ... with lane (i, q) holding
// columns 16 u + 4 q + {0..3} (u < 4) of token t0 + i and of route 16 kc + i.  The
// waves' tiles are summed in LDS in wave order; 16 or 32 consecutive lanes then
// hold a token's routes and form the activation as the operand preparation
// forms it (moc_mfma_common.hip).
template <int KC>
__global__ void __launch_bounds__(256)
router_f32_fwd_kernel(const float* __restrict__ z, const float* __restrict__ r,
                      float* __restrict__ out, int64_t N, int Z, int K, int routing) {
  constexpr int KP = 16 * KC;
  __shared__ float red[4][16][KP + 1];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int i = lane & 15, q = lane >> 4;
  const int64_t t0 = static_cast<int64_t>(blockIdx.x) * 16;
  const int64_t rows = N - t0 < 16 ? N - t0 : 16;
  // rows past N and routes past K lie outside the buffers and load zeros
  const Buf zb(z + t0 * Z, rows * Z * 4);
  const Buf rb(r, static_cast<int64_t>(K) * Z * 4);
  const int nchunk = Z / 64;
  // one sum per 16 columns of a chunk: chains a quarter as long, for the products
  // in flight and for the rounding of the sums (Z 1024: 1.55e-7 off the 64-bit
  // logits, a library GEMM 2.9e-7; a decode step's y 2.4e-7 -> 1.6e-7)
  f32x4 acc[4][KC];
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int kc = 0; kc < KC; ++kc) acc[u][kc] = f32x4{0.f, 0.f, 0.f, 0.f};
  // two chunks in flight (a chunk past the row loads zeros)
  struct Ops {
    f32x4 z[4], r[KC][4];
  };
  auto load = [&](int c, Ops& o) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const uint32_t col = static_cast<uint32_t>((64 * c + 16 * u + 4 * q) * 4);
      o.z[u] = load4(zb, c < nchunk ? static_cast<uint32_t>(i * Z * 4) + col : kOffNone);
#pragma unroll
      for (int kc = 0; kc < KC; ++kc)
        o.r[kc][u] = load4(rb, c < nchunk ? static_cast<uint32_t>((16 * kc + i) * Z * 4) + col : kOffNone);
    }
  };
  auto mult = [&](const Ops& o) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) acc[u][kc] = mma4(o.z[u], o.r[kc][u], acc[u][kc]);
  };
  Ops a, b;
  load(w, a);
  for (int c = w; c < nchunk; c += 8) {
    load(c + 4, b);
    mult(a);
    load(c + 8, a);
    mult(b);
  }
  // D lane (j, q): route 16 kc + j, tokens 4 q + v
#pragma unroll
  for (int kc = 0; kc < KC; ++kc)
#pragma unroll
    for (int v = 0; v < 4; ++v)
      red[w][4 * q + v][16 * kc + i] = (acc[0][kc][v] + acc[1][kc][v]) + (acc[2][kc][v] + acc[3][kc][v]);
  __syncthreads();
#pragma unroll
  for (int pass = 0; pass < KC; ++pass) {
    const int idx = threadIdx.x + 256 * pass;
    const int tok = idx / KP, k = idx % KP;
    float v = ((red[0][tok][k] + red[1][tok][k]) + red[2][tok][k]) + red[3][tok][k];
    if (routing == ROUTE_SOFTMAX) {
      const float l = k < K ? v : -INFINITY;
      float m = l;
#pragma unroll
      for (int o = KP / 2; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
      const float e = k < K ? __expf(l - m) : 0.f;
      float sum = e;
#pragma unroll
      for (int o = KP / 2; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
      v = e * (1.0f / sum);
    } else if (routing == ROUTE_EXP) {
      v = __expf(v);
    }
    if (k < K && tok < rows) out[(t0 + tok) * K + k] = v;
  }
}

// ---------------------------------------------------------------------------
// dz[t, zc] = sum_k dl[t, k] router[k, zc] and the partial drouter[k, zc] =
// sum_t dl[t, k] z[t, zc] of a token range, either of them skipped when its
// pointer is null.  Workgroup: 64 columns and one range, 4 waves taking blocks of
// 16 tokens in turn.  dz: D rows are columns (tile tl, row 4 q + v: column 16 tl +
// 4 q + v, so a lane stores 16 bytes), D columns are tokens.  drouter: lane (j,
// q) loads columns 4 j + {0..3} of tokens 4 s + q (s < 4), tile v takes column
// 4 j + v.  The waves' drouter tiles are summed in LDS in wave order.
template <int KC>
__global__ void __launch_bounds__(256)
router_f32_bwd_kernel(const float* __restrict__ dl, const float* __restrict__ z,
                      const float* __restrict__ r, float* __restrict__ dz,
                      float* __restrict__ part, int64_t N, int Z, int K, int blocks_per_range) {
  constexpr int KP = 16 * KC;
  __shared__ float red[4][KP][65];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int i = lane & 15, q = lane >> 4;
  const int zs = blockIdx.x * 64;
  const Buf rb(r, static_cast<int64_t>(K) * Z * 4);
  // dz A operands: router[16 kc + 4 q + v][zs + 16 tl + i] (routes past K: zero)
  f32x4 aop[4][KC];
  if (dz != nullptr)
#pragma unroll
    for (int tl = 0; tl < 4; ++tl)
#pragma unroll
      for (int kc = 0; kc < KC; ++kc)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          float e;
          rb.load<4>(static_cast<uint32_t>(((16 * kc + 4 * q + v) * Z + zs + 16 * tl + i) * 4), &e);
          aop[tl][kc][v] = e;
        }
  f32x4 acc[4][KC];
#pragma unroll
  for (int tl = 0; tl < 4; ++tl)
#pragma unroll
    for (int kc = 0; kc < KC; ++kc) acc[tl][kc] = f32x4{0.f, 0.f, 0.f, 0.f};

  // buffers from the range's first token on (rows past N: zeros, dropped)
  const int64_t first = static_cast<int64_t>(blockIdx.y) * blocks_per_range * 16;
  const int64_t rows = N - first < static_cast<int64_t>(blocks_per_range) * 16
                           ? N - first : static_cast<int64_t>(blocks_per_range) * 16;
  const Buf zb(z + first * Z, part != nullptr ? rows * Z * 4 : 0);
  const Buf db(dl + first * K, rows * K * 4);
  const Buf ob(dz + first * Z, dz != nullptr ? rows * Z * 4 : 0);
  struct Regs {
    f32x4 z[4];        // tokens 4 s + q, columns zs + 4 i + {0..3}
    f32x4 b[KC];       // dl[token i][16 kc + 4 q + {0..3}]
    float a[KC][4];    // dl[token 4 s + q][16 kc + i]
  };
  auto load = [&](Regs& g, int blk) {
    const int t = 16 * blk;  // (blocks past the range lie past the buffers)
#pragma unroll
    for (int s = 0; s < 4; ++s)
      g.z[s] = load4(zb, (static_cast<uint32_t>(t + 4 * s + q) * static_cast<uint32_t>(Z) + zs + 4 * i) * 4);
#pragma unroll
    for (int kc = 0; kc < KC; ++kc) {
      g.b[kc] = load4(db, 16 * kc + 4 * q < K ? static_cast<uint32_t>(((t + i) * K + 16 * kc + 4 * q) * 4) : kOffNone);
#pragma unroll
      for (int s = 0; s < 4; ++s)
        db.load<4>(16 * kc + i < K ? static_cast<uint32_t>(((t + 4 * s + q) * K + 16 * kc + i) * 4) : kOffNone,
                   &g.a[kc][s]);
    }
  };
  auto mult = [&](const Regs& g, int blk) {
    if (dz != nullptr) {
#pragma unroll
      for (int tl = 0; tl < 4; ++tl) {
        f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kc = 0; kc < KC; ++kc) o = mma4(aop[tl][kc], g.b[kc], o);
        ob.store<16>((static_cast<uint32_t>(16 * blk + i) * static_cast<uint32_t>(Z) + zs + 16 * tl + 4 * q) * 4, &o);
      }
    }
    if (part != nullptr) {
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int tl = 0; tl < 4; ++tl)
#pragma unroll
          for (int kc = 0; kc < KC; ++kc)
            acc[tl][kc] = __builtin_amdgcn_mfma_f32_16x16x4f32(g.a[kc][s], g.z[s][tl], acc[tl][kc], 0, 0, 0);
    }
  };
  Regs ga, gb;
  load(ga, w);
  for (int b = w; b < blocks_per_range; b += 8) {
    load(gb, b + 4);
    mult(ga, b);
    load(ga, b + 8);
    if (b + 4 < blocks_per_range) mult(gb, b + 4);
  }
  if (part == nullptr) return;
  // D lane (j, q): column 4 j + tl, routes 16 kc + 4 q + v
#pragma unroll
  for (int tl = 0; tl < 4; ++tl)
#pragma unroll
    for (int kc = 0; kc < KC; ++kc)
#pragma unroll
      for (int v = 0; v < 4; ++v) red[w][16 * kc + 4 * q + v][4 * i + tl] = acc[tl][kc][v];
  __syncthreads();
  for (int idx = threadIdx.x; idx < K * 64; idx += 256) {
    const int k = idx / 64, c = idx % 64;
    part[(static_cast<int64_t>(blockIdx.y) * K + k) * Z + zs + c] =
        ((red[0][k][c] + red[1][k][c]) + red[2][k][c]) + red[3][k][c];
  }
}

// drouter = sum of the ranges' partials, in range order, eight loads in flight
__global__ void __launch_bounds__(256)
router_f32_reduce_kernel(const float* __restrict__ part, float* __restrict__ dr, int64_t KZ, int n) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (idx >= KZ) return;
  float s = 0.f;
  int p = 0;
  for (; p + 8 <= n; p += 8) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = part[(p + u) * KZ + idx];
#pragma unroll
    for (int u = 0; u < 8; ++u) s += v[u];
  }
  for (; p < n; ++p) s += part[p * KZ + idx];
  dr[idx] = s;
}

inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

struct F32Plan {
  int64_t ranges, blocks_per_range;
};
// about 1024 workgroups (two resident per CU and their successors), each wave
// with a block at least; a range's rows stay within a buffer's 32-bit offsets
// (the whole of z does: router_f32_supported)
F32Plan f32_plan(int64_t N, int64_t Z) {
  const int64_t nblk = cdiv(N, 16);
  int64_t ranges = cdiv(1024, Z / 64);
  if (ranges > cdiv(nblk, 4)) ranges = cdiv(nblk, 4);
  const int64_t bpr = cdiv(nblk, ranges);
  return F32Plan{cdiv(nblk, bpr), bpr};
}

}  // namespace
}  // namespace router

// The kernels address z and the router with 32-bit byte offsets: n_tokens z_dim and
// the router with its routes padded to a tile (16 or 32 rows, also the 16 token
// rows of a block past the last one) are below 2^29 elements each.
bool router_f32_supported(int64_t N, int64_t Z, int64_t K) {
  const int64_t lim = int64_t(1) << 29;
  return K > 0 && K <= kRouterMaxRoutedK && K % 4 == 0 && Z >= 64 && Z % 64 == 0 && N > 0 &&
         N <= (int64_t(1) << 30) && Z < lim / 16 && N * Z < lim && router::cdiv(K, 16) * 16 * Z < lim;
}

void router_f32_forward(const void* z, const void* r, void* out, int64_t N, int64_t Z, int64_t K,
                        int routing, hipStream_t st) {
  auto kern = K <= 16 ? router::router_f32_fwd_kernel<1> : router::router_f32_fwd_kernel<2>;
  hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(router::cdiv(N, 16))), dim3(256), 0, st,
                     static_cast<const float*>(z), static_cast<const float*>(r),
                     static_cast<float*>(out), N, static_cast<int>(Z), static_cast<int>(K), routing);
}

size_t router_f32_backward_workspace(int64_t N, int64_t Z, int64_t K) {
  return static_cast<size_t>(router::f32_plan(N, Z).ranges * K * Z) * 4;
}

void router_f32_backward(const void* z, const void* r, const void* dl, void* dz, void* dr,
                         int64_t N, int64_t Z, int64_t K, void* workspace, hipStream_t st) {
  const router::F32Plan pl = router::f32_plan(N, Z);
  float* part = dr != nullptr ? static_cast<float*>(workspace) : nullptr;
  auto kern = K <= 16 ? router::router_f32_bwd_kernel<1> : router::router_f32_bwd_kernel<2>;
  hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(Z / 64), static_cast<unsigned>(pl.ranges)),
                     dim3(256), 0, st, static_cast<const float*>(dl), static_cast<const float*>(z),
                     static_cast<const float*>(r), static_cast<float*>(dz), part, N,
                     static_cast<int>(Z), static_cast<int>(K), static_cast<int>(pl.blocks_per_range));
  if (dr != nullptr)
    hipLaunchKernelGGL(router::router_f32_reduce_kernel,
                       dim3(static_cast<unsigned>(router::cdiv(K * Z, 256))), dim3(256), 0, st, part,
                       static_cast<float*>(dr), K * Z, static_cast<int>(pl.ranges));
}

}  // namespace moc
