// Router GEMMs of fp32 MoC layers (moc/api.py:383-388 of the reference: logits =
// F.linear(z, router) with the softmax / exp after it, and its autograd), the
// fp32 counterparts of moc_router.hip.
//
// All three products have at most 32 routes on one side, so what bounds them is
// one pass over z (and dz) through HBM; a library GEMM tiles for a wide second
// side instead.  The products run on the fp32 matrix instruction
// (v_mfma_f32_16x16x4_f32: 2 N Z K flops each, a fifth of the streaming time at 16
// routes, half of it at 32), a contraction in any order both operands agree on
// (step v of four takes entries 4 q + v); sums are fp32 and in a fixed order.
// N 8192, Z 1024, 16 routes, us (a copy of z 13.6): forward with the softmax 10.7,
// the library's 16.0; dz and drouter 22.9, the library's 51.5.
// K % 4 == 0, K <= 32, Z % 64 == 0.

#include "moc_kernels.h"
#include "moc_mfma_launch.h"

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
// out[t, k] = activation_k(sum_z z[t, z] router[k, z]).  Workgroup: 16 tokens, W
// waves; wave w sums the 64-wide z chunks w, w + W, ...  A product's lane (i, q)
// wants 16 bytes of row i, but four neighbouring lanes in four rows cost the
// access path four times what 64 bytes of one row do (16 bytes a clock and CU,
// whatever the stride or the number of waves: what bounded this kernel).  So a
// half chunk's tiles (the tokens', and one per 16 routes) are loaded eight lanes
// to a row of 128 bytes, written to a wave-private LDS tile and read back as
// operands, while the next chunk's same half is loaded.  The waves' sums are
// added in pairs, through LDS; 16 or 32 consecutive lanes then hold a token's routes
// and form the activation as the operand preparation forms it (moc_mfma_common.hip).
//
// Us, operands loaded as they lie -> here: 16 routes, Z 1024, 48 tokens 5.6 -> 3.8,
// 8192 tokens 11.9 -> 11.5; Z 4096, 300 tokens 16.4 -> 8.4, 16384 tokens 68.6 -> 59.1;
// 32 routes, Z 4096, 48 tokens 23.9 -> 12.8, 16384 tokens 97.9 -> 66.5 (z alone 52 at the
// copy rate; a library GEMM 55); Z 512, 16384 tokens 16.0 -> 12.1.  Whole chunks in LDS:
// the same at 16 routes, 14.7 there (fewer workgroups of a CU).  Blocks of 32 tokens
// (half the reads of the router): half again slower up to 4096 tokens, within 10% past.
template <int KC, int W>
__global__ void __launch_bounds__(64 * W)
router_f32_fwd_kernel(const float* __restrict__ z, const float* __restrict__ r,
                      float* __restrict__ out, int64_t N, int Z, int K, int routing) {
  constexpr int KP = 16 * KC, T = 1 + KC;  // tiles of a chunk: tokens, routes
  __shared__ __align__(16) f32x4 st[W][T][128];
  float(*red)[16][KP + 1] = reinterpret_cast<float(*)[16][KP + 1]>(st);
  static_assert(sizeof(float) * W * 16 * (KP + 1) <= sizeof(st), "the sums fit the tiles");
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int i = lane & 15, q = lane >> 4;
  const int64_t t0 = static_cast<int64_t>(blockIdx.x) * 16;
  const int64_t rows = N - t0 < 16 ? N - t0 : 16;
  const int k0 = KP * static_cast<int>(blockIdx.y);  // (first route of this workgroup)
  // rows past N and routes past K lie outside the buffers and load zeros
  const Buf zb(z + t0 * Z, rows * Z * 4);
  const Buf rb(r + static_cast<int64_t>(k0) * Z, static_cast<int64_t>(K - k0) * Z * 4);
  const int nchunk = Z / 64;
  // several sums, each of its 16-column parts of the chunks: short chains, for the
  // products in flight and for the rounding of the sums (Z 1024: 1.55e-7 off the
  // 64-bit logits, a library GEMM 2.9e-7; a decode step's y 2.4e-7 -> 1.6e-7)
  constexpr int US = 16 / W;
  f32x4 acc[US][KC];
#pragma unroll
  for (int u = 0; u < US; ++u)
#pragma unroll
    for (int kc = 0; kc < KC; ++kc) acc[u][kc] = f32x4{0.f, 0.f, 0.f, 0.f};
  // load l of a half tile: row 8 l + lane / 8, of its 32 columns the 16 bytes
  // (lane % 8) ^ (row / 2), to slot 64 l + lane: the 16 rows that a group of lanes
  // reads then lie in 16 different slots modulo 16
  uint32_t off[2];
#pragma unroll
  for (int l = 0; l < 2; ++l) {
    const int row = 8 * l + (lane >> 3);
    off[l] = (static_cast<uint32_t>(row) * Z + 4 * ((lane & 7) ^ (row >> 1))) * 4;
  }
  f32x4 raw[2][T][2];
  auto load = [&](int c, int h) {  // (a chunk past the row loads zeros)
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int l = 0; l < 2; ++l) {
        const uint32_t tile = static_cast<uint32_t>(t > 0 ? 16 * (t - 1) : 0) * Z * 4 + 256 * c + 128 * h;
        raw[h][t][l] = load4(t > 0 ? rb : zb, c < nchunk ? off[l] + tile : kOffNone);
      }
  };
  load(w, 0);
  load(w, 1);
  for (int c = w; c < nchunk; c += W) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int l = 0; l < 2; ++l) st[w][t][64 * l + lane] = raw[h][t][l];
      load(c + W, h);
      __builtin_amdgcn_sched_barrier(0);
      mfma::wave_lds_sync();
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        // row i, columns 32 h + 16 u + 4 q + {0..3}
        const int slot = 64 * (i >> 3) + 8 * (i & 7) + ((4 * u + q) ^ (i >> 1)), a = (2 * h + u) % US;
#pragma unroll
        for (int kc = 0; kc < KC; ++kc) acc[a][kc] = mma4(st[w][0][slot], st[w][1 + kc][slot], acc[a][kc]);
      }
      mfma::wave_lds_sync();
    }
  }
  __syncthreads();
  // D lane (j, q): route 16 kc + j, tokens 4 q + v
#pragma unroll
  for (int kc = 0; kc < KC; ++kc)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      float s = acc[0][kc][v] + acc[1][kc][v];
      if constexpr (US == 4) s += acc[2][kc][v] + acc[3][kc][v];
      red[w][4 * q + v][16 * kc + i] = s;
    }
  __syncthreads();
  for (int idx = threadIdx.x; idx < 16 * KP; idx += 64 * W) {  // (whole waves: 16 KP is 4 or 8 of them)
    const int tok = idx / KP, k = idx % KP;
    float part[W];
#pragma unroll
    for (int ww = 0; ww < W; ++ww) part[ww] = red[ww][tok][k];
#pragma unroll
    for (int d = 1; d < W; d *= 2)
#pragma unroll
      for (int ww = 0; ww < W; ww += 2 * d) part[ww] += part[ww + d];
    float v = part[0];
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
    if (k0 + k < K && tok < rows) out[(t0 + tok) * K + k0 + k] = v;
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
  // eight waves a workgroup while every CU has at most one and each wave a chunk, else
  // four (16 routes, Z 4096, 2000 tokens: 12.3 us with eight, 15.3 with four; 32 routes,
  // Z 512, 16384 tokens: 13.9 and 12.1; below Z 512 four waves' shorter sums are 20%
  // closer to 64 bits for 0.4 us)
  const int64_t blocks = router::cdiv(N, 16);
  const int n_cu = mfma::device_cu_count(), cus = n_cu > 0 ? n_cu : 256;
  const bool eight = blocks <= cus && Z >= 512;
  // more than 16 routes in two workgroups of 16 where half the CUs would be idle and
  // no softmax joins them: a CU's matrix rate bounds a token block (decode step of 16
  // tokens, Z 4096, 32 routes: its router 12.8 -> 8.0 us)
  const bool halves = K > 16 && routing != ROUTE_SOFTMAX && 2 * blocks <= cus;
  const bool one = K <= 16 || halves;
  auto kern = one ? (eight ? router::router_f32_fwd_kernel<1, 8> : router::router_f32_fwd_kernel<1, 4>)
                  : (eight ? router::router_f32_fwd_kernel<2, 8> : router::router_f32_fwd_kernel<2, 4>);
  hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(blocks), halves ? 2 : 1), dim3(eight ? 512 : 256), 0, st,
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
