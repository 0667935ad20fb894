// Fused backward (stage 1) with 2 to 8 taps: bf16 up to 32 routes, fp32 up to 16
// (32 with up to 5 taps).
//
// What bounds it: instruction issue and the latency chains of two to four waves
// per SIMD (four, 128 VGPRs, with 2 to 4 taps and 16 routes; else two, 256 VGPRs).
// A wave holds 16 channels, one per lane, and a workgroup of 8 waves the 128
// channels of bwd_tile's workgroup, so channel groups, range counts and
// partial-sum layouts are those of its grids, and stage 2 is the same.
//
// A range's rows are cut in four streams of 8 n rows, one per 16-lane group of
// the wave (lane (j, q): channel j, stream q), walked in n steps of 8 rows.  So
// what a row shares with its neighbours stays in the lane's registers from step
// to step: the last S - 1 x rows of the window, and the partial dx of the last
// S - 1 rows, to which later rows still add (dx[t - off] += g[t] W_{S-1-off}[t]:
// the same W tile that P uses).  A stream hands what its first rows owe to the
// rows before them to the stream before it at the end.  Against super-blocks of
// 32 consecutive rows (S - 1 rows of each recomputed in the next, S + 7 window
// rows loaded and converted for 8, a second W tile at shifted rows and a
// cross-lane read of g for dx) a row of 4 taps takes 25% fewer vector
// instructions and 8 fewer matrix instructions of 32.  And one pass holds every
// tap and both route chunks, where dx and the m products of more taps or routes
// ran as two passes with g = dy silu'(P) through memory, or once per route chunk.
//
// Both stages, us, before -> here (B4 T4096 D2048, without / with SiLU):
//   taps       2                3                4                6                8
//   16 routes  67.5->66.6       77.7->74.7       80.7->75.2       138.7->99.6      151.8->119
//              72.4->69.7       84.8->77.7       90.6->80.0       157.4->110       201.2->129
//   32 routes  94.5->82.9       127->94          130->102         161->129         194.6->158
//              116->85.7        152->95.5        190->109         217->137         252->169
// and D 4096: 32768 tokens, 16 routes, 4 taps 275 -> 262.6; 16384 tokens, 32
// routes, 8 taps 335 -> 280.  So it serves every bf16 shape it is built for.
//
// fp32 (every product on v_mfma_f32_16x16x4_f32, whose rate is half of what bounds
// it: 96 of them, 3072 cycles, a step and wave at 4 taps, 82 us of the 165 below;
// m needs no split, and its dbasis operand is the lane's own registers).  Backward
// entry, B4 T4096 D2048, 16 routes, without / with SiLU, us, the fused pass of
// bwd_tile or the two passes with g through memory -> here:
//   taps  2            3            4            5            6            8
//         111->(114)   170->132     206->158     249->184     260->209     330->263
//         132->118     180->137     273->165     342->193     352->223     484->282
// B4 T2048 D1024, 4 taps, SiLU: 92 -> 54, its training step 145 -> 108; same
// order at 4 routes, D 4096, and 600 rows of D 3000.  32 routes, to 5 taps (six
// taps' basis tiles are past a CU's LDS), the fused pass (2, 3 taps) or the two
// passes -> here:
//   taps  2            3            4            5
//         226->204     287->237     322->268     424->318
//         253->185     356->228     414->276     546->320
// B4 T2048 D1024, 4 taps, SiLU: 129 -> 85.
//
// Work per step and wave (rows 8 i .. 8 i + 7 of each stream):
//   W_s = alpha . basis_s by MFMA (16x16x16, or 16x16x32 over 32 routes; both
//   operands from LDS, the basis tile read transposed), P = sum_s W_s x_s, g =
//   dy silu'(P); dx as above; m_s = g x_s split in bf16 hi / lo; dbasis +=
//   alpha^T m_s (16x16x32 over the 32 rows, accumulated over the whole range in
//   registers); dalpha += m . basis^T over 16 channels of hi and lo (16x16x32, m
//   read back transposed from a wave-private LDS tile with ds_read_b64_tr_b16);
//   the 8 waves' dalpha tiles summed in LDS in wave order.
//
// Measured and not kept (4 taps, 16 routes, SiLU, 79.9 us): x and dy as one
// 16-byte load per lane through an LDS tile (4x fewer memory instructions, more
// LDS work: 81.9); the rows' scalar offsets in the accesses' soffset (85.8); the
// next rows fetched before the m products (no change where it fits the registers,
// 112 where it spills); the step loop unrolled twice (no change).
#pragma once

#include "moc_mfma.h"

namespace moc {
namespace mfma {

// m tile of one wave for the transposed dalpha reads, one channel per lane.
// Writer lane (j, q) holds, per token block b, m of channel j at the tokens
// 4 g + {0..3} of token group g = 2 q + b: one 8-byte slot.  The dalpha A
// operand wants, in lane i of 16-lane group qq, the channels 4 qq + {0..3} of
// token 16 rb + i; ds_read_b64_tr_b16 gives lane i element i % 4 of the slots
// read by lanes i / 4 + {0, 4, 8, 12} of its group, so reader lane 4 e + a
// reads the slot of channel 4 qq + e, token group 4 rb + a.  Slot (ch, g) sits
// at g 16 + (ch ^ 4 (g & 3)): a writer group covers 16 consecutive slots, a
// reader group 16 distinct slots modulo 16 (no bank conflicts).
struct TrTile1 {
  static constexpr int kSlots = 8 * 16;  // 8 token groups x 16 channels
  static __device__ __forceinline__ int wslot(int j, int q, int b) {
    const int g = 2 * q + b;
    return g * 16 + (j ^ (4 * (g & 3)));
  }
  static __device__ __forceinline__ int rslot(int i, int qq, int rb) {
    const int e = i >> 2, a = i & 3;
    const int g = 4 * rb + a;
    return g * 16 + ((4 * qq + e) ^ (4 * a));
  }
};

constexpr int kLeanWPG = 8;        // waves per workgroup (8 x 16 = 128 channels)
constexpr int kLeanCW = 16;        // channels per wave

// Shapes the lean pass serves (fp32 with 2 taps and no activation, where there is
// little to form or share: 111 us in the fused pass of bwd_tile, 114 here)
constexpr bool bwd_lean(int S, int KC, bool act, bool bf) {
  return S >= 2 && (bf ? KC <= 2 && S <= 8 : (KC == 1 && S <= 8 && (act || S > 2)) || (KC == 2 && S <= 5));
}
// Waves per SIMD it is built for: four (128 VGPRs, two workgroups per CU) with 2
// to 4 taps and 16 routes in bf16, else two (256 VGPRs and up to 156 KB of LDS,
// one workgroup per CU)
constexpr int lean_waves(int S, int KC, bool bf = true) { return bf && S <= 4 && KC == 1 ? 4 : 2; }

// LDS tiles of the fp32 form: rows of 16 floats, the 4-float chunk c of row r at
// chunk c ^ sw, and 16 floats of padding after every P rows.  Tiles that 16
// lanes read 16 bytes each down 16 rows, and that the wave writes or reads a
// float per lane across four row groups P apart, touch every bank once.
template <int P>
__device__ __forceinline__ int f32_slot(int row, int chunk, int sw) {
  return row * 16 + (row / P) * 16 + 4 * (chunk ^ sw);
}
// routing weights (rows 8 q + r), m (likewise) and the basis (routes)
__device__ __forceinline__ int f32_aslot(int row, int chunk) { return f32_slot<8>(row, chunk, row >> 3); }
__device__ __forceinline__ int f32_mslot(int row, int chunk) { return f32_slot<8>(row, chunk, (row >> 2) & 3); }
__device__ __forceinline__ int f32_bslot(int row, int chunk) { return f32_slot<4>(row, chunk, row >> 2); }
constexpr int kF32Rows = 32 * 16 + 3 * 16, kF32Basis = 16 * 16 + 3 * 16;  // floats of a tile

// Rows of a row-major tensor walked with the scalar unit: next(bytes) is a buffer
// from the current row on (`left` bytes; at most 0 past the end: loads give
// zero, stores drop) and moves `bytes` on.  A lane's byte offset (its stream's
// first row and its channel) is then the same in every step.  (Opaque after each
// move: the compiler otherwise precomputes one 64-bit offset per row, more
// scalars than there are.)
struct RowWalk {
  const char* p;
  int32_t left;
  __device__ __forceinline__ Buf next(uint32_t bytes, bool on = true) {
    const Buf b(p, on ? left : 0);
    p += bytes;
    left -= static_cast<int32_t>(bytes);
    asm volatile("" : "+s"(p), "+s"(left));
    return b;
  }
};

// The work of workgroup (bx, by) of one layer; the __global__ wrappers below
// map a single launch's 2-D grid or a grouped launch's 1-D grid onto it.
template <int S, int KC, int ACT, bool DY1, bool BF>
__device__ __forceinline__ void
bwd_lean_tile(const void* __restrict__ xv, const void* __restrict__ dyv, int64_t dys,
              const typename CT<BF>::elem* __restrict__ a_c,
              const typename CT<BF>::elem* __restrict__ b_c, void* __restrict__ dxv, float* __restrict__ part_da, float* __restrict__ part_db,
              SeqLayout seq, int64_t D, int bx, int by, int gy, int gy1, int n_old, int n_total,
              bool act_rt = false) {
  const bool act = ACT == kActRuntime ? act_rt : ACT != 0;  // (uniform)
  using C = CT<BF>;
  using E = typename C::elem;
  using Op = typename C::opnd;
  constexpr int NB = 2, R = 8, TB = 32, H = S - 1, W = R + H;
  constexpr int KP = 16 * KC, WPG = kLeanWPG, CW = kLeanCW;
  constexpr int ESZ = sizeof(E);
  static_assert(S >= 2 && S <= 8 && KC <= 2, "lean backward: 2 to 8 taps, up to 32 routes");
  // the four-wave form leaves what a stream owes its predecessor in LDS
  constexpr bool kC0Lds = lean_waves(S, KC, BF) == 4;
  // The next step's rows are loaded where this step's have been converted in the
  // two-wave form (a SIMD has one other wave to cover the loads: 16 routes, 8
  // taps 80.9 -> 77.1 us, 32 routes, 4 taps 115.4 -> 109.0), after the m products
  // in the others (four waves cover them; 8 taps with 32 routes would spill, 167
  // -> 204 us)
  constexpr bool kFetchEarly = lean_waves(S, KC, BF) == 2 && !(S == 8 && KC == 2);

  // routing-weight rows of a step, unpadded: row rho = 8 q + r is row r of
  // stream q; the 8-byte chunk c (4 routes) of row rho sits at chunk c ^ asw(rho)
  // (W operand, transposed and staging accesses without bank conflicts)
  auto asw = [](int row) -> int {
    return KC == 1 ? (row >> 3) & 3 : ((row >> 1) & 1) | (((row >> 3) & 3) << 1);
  };
  __shared__ __align__(16) E a_lds[2][BF ? TB : KC][BF ? KP : kF32Rows];
  __shared__ __align__(16) Op m_tr[BF ? WPG : 1][2][TrTile1::kSlots];  // [wave][hi / lo]
  __shared__ __align__(16) float m_f32[BF ? 1 : WPG][kF32Rows];        // fp32: rows x channels
  // basis tile of each wave, b_lds[wave][s][kc][route j][4 channels, chunk q ^
  // (j / 4)] (a 16-lane group of a read touches 16 distinct slots)
  __shared__ __align__(16) Op b_lds[WPG][S][KC][BF ? 16 * 4 : kF32Basis / 4];
  // (fp32 over 32 routes: one buffer, the two of them past the CU's LDS, and a
  // second barrier in a step)
  constexpr int DAB = BF || KC == 1 ? 2 : 1;
  __shared__ float da_lds[DAB][WPG][NB][KC][16][17];
  __shared__ float c0_lds[kC0Lds ? H : 1][kC0Lds ? 64 * WPG : 1];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 15, q = lane >> 4;
  const int64_t N = seq.n_tokens;
  const int64_t d0 = (static_cast<int64_t>(bx) * WPG + wave) * CW;
  const bool wave_on = d0 < D;
  const int64_t dl = d0 + j;
  const bool ch_ok = wave_on && dl < D;

  // steps [sb_lo, sb_hi) of this range (ranges by < gy1 share the first n_old),
  // n of them: rows [first, first + 32 n), the last S - 1 not its own
  const int64_t sb_lo = by < gy1 ? static_cast<int64_t>(by) * n_old / gy1
                                 : n_old + static_cast<int64_t>(by - gy1) * (n_total - n_old) / (gy - gy1);
  const int64_t sb_hi = by < gy1 ? static_cast<int64_t>(by + 1) * n_old / gy1
                                 : n_old + static_cast<int64_t>(by + 1 - gy1) * (n_total - n_old) / (gy - gy1);
  const int n = static_cast<int>(sb_hi - sb_lo);
  const int64_t first = sb_lo * TB - static_cast<int64_t>(by) * H;
  const int64_t end = first + static_cast<int64_t>(n) * TB;
  const int64_t row_hi = end < N ? end : N;            // rows read
  const int64_t own_hi = end - H < N ? end - H : N;    // rows owned
  const int srow = R * n * q;                          // first row of this lane's stream
  const uint32_t rb = static_cast<uint32_t>(D * ESZ);
  const uint32_t col = static_cast<uint32_t>(dl * ESZ);
  const uint32_t vx = ch_ok ? static_cast<uint32_t>(srow) * rb + col : kOffNone;
  RowWalk xwalk{static_cast<const char*>(xv) + first * rb, static_cast<int32_t>((row_hi - first) * rb)};
  RowWalk dxw{static_cast<const char*>(dxv) + (first - H) * rb,
              static_cast<int32_t>((own_hi - first + H) * rb)};
  // dy rows dys elements apart (D; 0: one row for all tokens; -1: one element
  // for every token and channel, the expanded gradient of a sum).  DY1 (dys =
  // -1 in every layer of the launch): the element is read once.  Otherwise a -1
  // of one layer reads the element in place of every row (rows 0 bytes apart,
  // no channel offset)
  const bool dy_one = DY1 || dys < 0;
  const uint32_t drb = static_cast<uint32_t>((dy_one ? 0 : dys) * ESZ);
  const uint32_t vdy = ch_ok ? static_cast<uint32_t>(srow) * drb + (dy_one ? 0u : col) : kOffNone;
  // (the bytes after row w: rows up to row_hi, the last one D elements long)
  RowWalk dyw{static_cast<const char*>(dyv) + first * drb,
              static_cast<int32_t>(dy_one ? ESZ
                                          : (row_hi > first ? (row_hi - first - 1) * drb + D * ESZ : 0))};
  float dy1 = 0.f;
  if constexpr (DY1) {
    E e;
    Buf(dyv, ESZ).load<ESZ>(ch_ok ? 0u : kOffNone, &e);
    dy1 = C::to_f(e);
  }
  const Buf bb(b_c, static_cast<int64_t>(KP) * S * D * ESZ);

  // dalpha B operands: basis[j, s, d0 + 4 q + {0..3}] (channels past D,
  // with D % 4 == 2 the last two of the final group, zero: the load reaches into
  // the next row)
  {
    const int64_t ch = d0 + 4 * q;
    const bool on = wave_on && ch < D;
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) {
        Op bda;
        bb.load<4 * ESZ>(row_off((16 * kc + j) * S + s, 0, rb, static_cast<uint32_t>(ch * ESZ), on), &bda);
        if (ch + 2 >= D) {
          bda[2] = 0;
          bda[3] = 0;
        }
        b_lds[wave][s][kc][BF ? j * 4 + (q ^ (j >> 2)) : f32_bslot(j, q) / 4] = bda;
      }
  }
  f32x4 dbacc[S][KC];
#pragma unroll
  for (int s = 0; s < S; ++s)
#pragma unroll
    for (int kc = 0; kc < KC; ++kc) dbacc[s][kc] = f32x4{0.f, 0.f, 0.f, 0.f};

  // raw rows of one step
  E xr[R], dr[DY1 ? 1 : R];
  // (two rows per buffer: one more vector add against six scalar instructions)
  auto fetch_xdy = [&]() {
#pragma unroll
    for (int r = 0; r < R; r += 2) {
      const Buf b = xwalk.next(2 * rb);
      b.load<ESZ>(vx, &xr[r]);
      b.load<ESZ>(vx + rb, &xr[r + 1]);
    }
    if constexpr (!DY1) {
#pragma unroll
      for (int r = 0; r < R; r += 2) {
        const Buf b = dyw.next(2 * drb);
        b.load<ESZ>(vdy, &dr[r]);
        b.load<ESZ>(vdy + drb, &dr[r + 1]);
      }
    }
  };
  // routing-weight rows of a step: 32 rows, 4 routes per thread of the first 2 KC
  // waves (row rho: thread 4 KC rho + chunk)
  // (the per-lane terms are formed where they are used, from an opaque copy of
  // the thread id: hoisted out of the loop they outgrow the register budget)
  auto opaque_tid = [&]() {
    int t = tid;
    asm volatile("" : "+v"(t));
    return t;
  };
  static_assert(TB * KP / 4 == 128 * KC, "2 KC waves fetch a step's routing weights");
  RowWalk aw{reinterpret_cast<const char*>(a_c + first * KP), static_cast<int32_t>((row_hi - first) * KP * ESZ)};
  E arw[4];
  auto fetch_a = [&]() {
    const Buf ab = aw.next(R * KP * ESZ);
    if (wave < 2 * KC) {
      const int t = opaque_tid(), row = t / (4 * KC);
      ab.load<4 * ESZ>(static_cast<uint32_t>(((R * n * (row >> 3) + (row & 7)) * KP + (t % (4 * KC)) * 4) * ESZ),
                       arw);
    }
  };
  auto stage_alpha = [&](int buf) {
    if (wave < 2 * KC) {
      const int t = opaque_tid(), row = t / (4 * KC);
      if constexpr (BF) Vec<E, 4>::store(&a_lds[buf][row][((t % (4 * KC)) ^ asw(row)) * 4], arw);
      else Vec<E, 4>::store(&a_lds[buf][KC == 1 ? 0 : t % (4 * KC) / 4][f32_aslot(row, t % 4)], arw);
    }
  };

  // the window rows before the stream: rows first + srow - H + w
  float xw[W];
#pragma unroll
  for (int w = 0; w < H; ++w) {
    const int64_t u = first + srow - H + w;
    E e;
    const int64_t lo = first - H > 0 ? first - H : 0;
    Buf(static_cast<const char*>(xv) + lo * rb, (row_hi - lo) * rb).load<ESZ>(row_off(u, lo, rb, col, ch_ok), &e);
    xw[R + w] = C::to_f(e);
  }
  fetch_xdy();
  fetch_a();
  stage_alpha(0);
  __syncthreads();

  // the next segment start at or after this lane's window (rows from `first`;
  // the token axis's end counts as one), searched again once a window passed it
  const int32_t n_rel = static_cast<int32_t>(N - first < (int64_t(1) << 30) ? N - first : int64_t(1) << 30);
  auto start_from = [&](int64_t rel) -> int32_t {
    const int64_t st = seq.next_start(first + rel) - first;
    return static_cast<int32_t>(st < n_rel ? st : n_rel);
  };
  int32_t ns = start_from(srow - (S - 2));

  // dx rows -(S-1) .. R-1 of a step: dxa[w] is row w - (S-1); the first S-1 carry
  // over from the step before.  c0 / c0_lds: what a stream's first rows add to
  // the rows before it, which the stream before takes at the end
  float dxa[W], c0[H];
#pragma unroll
  for (int e = 0; e < H; ++e) dxa[R + e] = c0[e] = 0.f;

  // dalpha partials of this channel group from row `first` on (own rows)
  RowWalk pdw{reinterpret_cast<const char*>(part_da + (static_cast<int64_t>(bx) * N + first) * KP),
              static_cast<int32_t>((own_hi - first) * KP * 4)};

  auto step = [&](int i, auto mask_tag) {
    constexpr bool MASK = decltype(mask_tag)::value;
    const int tl = opaque_tid();
    const int j = tl & 15, q = (tl >> 4) & 3;
    const int buf = i & 1;
    const bool more = i + 1 < n;
#pragma unroll
    for (int w = 0; w < H; ++w) {
      xw[w] = xw[R + w];
      dxa[w] = dxa[R + w];
    }
    float g[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      xw[H + r] = C::to_f(xr[r]);
      g[r] = DY1 ? dy1 : C::to_f(dr[DY1 ? 0 : r]);
    }
    // (unconditionally, also after the last step: rows past the buffer load zeros)
    fetch_a();
    if constexpr (kFetchEarly) {
      __builtin_amdgcn_sched_barrier(0);
      fetch_xdy();
      __builtin_amdgcn_sched_barrier(0);
    }

    // alpha operand of token block b: row 8 (j / 4) + 4 b + j % 4, chunk 4 kc + q
    Op aop[NB][KC];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) {
        const int row = R * (j >> 2) + 4 * b + (j & 3);
        if constexpr (BF)
          aop[b][kc] = *reinterpret_cast<const Op*>(&a_lds[buf][row][((4 * kc + q) ^ asw(row)) * 4]);
        else
          aop[b][kc] = *reinterpret_cast<const Op*>(&a_lds[buf][kc][f32_aslot(row, q)]);
      }

    f32x4 dacc[NB][KC];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) dacc[b][kc] = f32x4{0.f, 0.f, 0.f, 0.f};

    {
      // bit k of `sbm`: window row t0 - (S-1) + k starts a segment; bit r of
      // `rv`: row t0 + r is a token (< N); tap s of row r is valid when the row
      // is a token and no segment starts in window rows r + s + 1 .. r + S - 1
      uint32_t sbm = 0, rv = 0;
      if constexpr (MASK) {
        const int32_t t0 = R * n * q + R * i;  // this lane's first row (from `first`)
        const int32_t u0 = t0 - H, lo_next = t0 + R - (S - 2);
        int32_t st = ns;
        while (st <= t0 + R - 1 && st < n_rel) {
          const int32_t k = st - u0;
          if (k > 0) sbm |= 1u << k;
          const int32_t nx = start_from(static_cast<int64_t>(st) + 1);
          if (st < lo_next) ns = nx;
          st = nx;
        }
        const int32_t nrow = n_rel - t0;  // rows r < nrow are tokens
        rv = nrow >= R ? 0xffu : (nrow <= 0 ? 0u : ((1u << nrow) - 1u));
      }
      auto tap_ok = [&](int r, int s) -> bool {
        if constexpr (MASK) {
          const uint32_t span = ((1u << (S - 1 - s)) - 1u) << (r + s + 1);
          return ((rv >> r) & 1u) && (sbm & span) == 0;
        } else {
          return true;
        }
      };

      // W of tap s for this lane's rows; the basis operand (routes 16 kc + 4 q + v,
      // channel j) is the tile's rows read transposed.  With the activation P and
      // dx read the same W tiles; without, over 32 routes, dx forms each where it
      // reads it
      auto form_w = [&](int s, f32x4 (&w)[NB]) {
        Op bop[KC];
#pragma unroll
        for (int kc = 0; kc < KC; ++kc) {
          if constexpr (BF) {
            bop[kc] = TrTile<NB, 2>::read(&b_lds[wave][s][kc][(4 * q + (j >> 2)) * 4 + ((j & 3) ^ q)]);
          } else {
            const float* bt = reinterpret_cast<const float*>(&b_lds[wave][s][kc][0]);
#pragma unroll
            for (int v = 0; v < 4; ++v) bop[kc][v] = bt[f32_bslot(4 * q + v, j >> 2) + (j & 3)];
          }
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
          if constexpr (KC == 2 && !BF) w[b] = C::mma(aop[b][1], bop[1], C::mma(aop[b][0], bop[0], zero));
          else if constexpr (KC == 2) w[b] = mma32(aop[b][0], aop[b][1], bop[0], bop[1], zero);
          else w[b] = C::mma(aop[b][0], bop[0], zero);
        }
      };
      constexpr bool kKeepW = ACT != 0 || KC == 1;
      f32x4 w4[kKeepW ? S : 1][NB];
      if constexpr (kKeepW)
#pragma unroll
        for (int s = 0; s < S; ++s) form_w(s, w4[s]);

      if constexpr (ACT != 0) if (act) {  // (act: uniform; always with a fixed ACT)
        float p[R];
#pragma unroll
        for (int r = 0; r < R; ++r) p[r] = 0.f;
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
          for (int r = 0; r < R; ++r)
            if (tap_ok(r, s)) p[r] = fmaf(xw[r + s], w4[kKeepW ? s : 0][r >> 2][r & 3], p[r]);
        // g *= silu'(P) = sg (1 + P (1 - sg)), sg = sigmoid(P) as sigmoid_f forms it
        float sg[R];
#pragma unroll
        for (int r = 0; r < R; ++r) sg[r] = __builtin_amdgcn_exp2f(-p[r] * 1.4426950408889634f);
#pragma unroll
        for (int r = 0; r < R; ++r) sg[r] = __builtin_amdgcn_rcpf(1.0f + sg[r]);
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const float v = fmaf(-sg[r], sg[r], sg[r]);
          g[r] = g[r] * fmaf(p[r], v, sg[r]);
        }
      }

      // dx[t - off] += g[t] W_{S-1-off}[t], nearest rows first
      if (dxv != nullptr) {
#pragma unroll
        for (int r = 0; r < R; ++r) dxa[H + r] = 0.f;
#pragma unroll
        for (int off = 0; off < S; ++off) {
          const int s = S - 1 - off;
          if constexpr (!kKeepW) form_w(s, w4[0]);
#pragma unroll
          for (int r = 0; r < R; ++r)
            if (tap_ok(r, s))
              dxa[H + r - off] = fmaf(g[r], w4[kKeepW ? s : 0][r >> 2][r & 3], dxa[H + r - off]);
        }
        if (i == 0) {
#pragma unroll
          for (int e = 0; e < H; ++e) {
            if constexpr (kC0Lds) c0_lds[e][tl] = dxa[e];
            else c0[e] = dxa[e];
          }
        }
        // rows -(S-1) .. R-S of the step are complete; before the first step's
        // they belong to the stream (or range) before
#pragma unroll
        for (int w = 0; w < R; ++w) {
          const E o = C::from_f(dxa[w]);
          dxw.next(rb, w >= H || i > 0).store<ESZ>(vx, &o);
        }
      }

      // alpha^T operands of the dbasis MFMA, own rows only (the last step's
      // final S-1 rows of stream 3 are the next range's; rows past N are zero):
      // at[b][v] = alpha[row 8 q + 4 b + v, j] (transposed read of the staged rows)
      Op at[NB][KC];
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int kc = 0; kc < KC; ++kc) {
          const int row = R * q + 4 * b + (j >> 2);
          if constexpr (BF) {
            at[b][kc] = TrTile<NB, 2>::read(&a_lds[buf][row][((4 * kc + (j & 3)) ^ asw(row)) * 4]);
          } else {
#pragma unroll
            for (int v = 0; v < 4; ++v)
              at[b][kc][v] = a_lds[buf][kc][f32_aslot(R * q + 4 * b + v, j >> 2) + (j & 3)];
          }
        }
      if (!more) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          constexpr int kOwn = R - H;  // rows of stream 3 that are still this range's
          const int n_ok = kOwn - 4 * b < 0 ? 0 : (kOwn - 4 * b < 4 ? kOwn - 4 * b : 4);
          if constexpr (BF) {
            const uint64_t keep = q == 3 && n_ok < 4 ? ((1ull << (16 * n_ok)) - 1ull) : ~0ull;
#pragma unroll
            for (int kc = 0; kc < KC; ++kc)
              at[b][kc] = __builtin_bit_cast(Op, __builtin_bit_cast(uint64_t, at[b][kc]) & keep);
          } else {
#pragma unroll
            for (int kc = 0; kc < KC; ++kc)
#pragma unroll
              for (int v = 0; v < 4; ++v)
                if (q == 3 && v >= n_ok) at[b][kc][v] = 0.f;
          }
        }
      }
      if constexpr (BF) {
        // m of tap s -> hi / lo operands -> this wave's tile, dbasis MFMAs
        auto stage_m = [&](int s) {
          Op mh[NB], ml[NB];
#pragma unroll
          for (int b = 0; b < NB; ++b) {
            uint32_t hbits[4];
            float lo[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
              const int r = 4 * b + v;
              const float mval = tap_ok(r, s) ? g[r] * xw[r + s] : 0.f;
              hbits[v] = __float_as_uint(mval) & 0xffff0000u;
              lo[v] = mval - __uint_as_float(hbits[v]);
            }
            mh[b] = pack4_hi(hbits[0], hbits[1], hbits[2], hbits[3]);
            ml[b] = pack4_bf16(lo[0], lo[1], lo[2], lo[3]);
            m_tr[wave][0][TrTile1::wslot(j, q, b)] = mh[b];
            m_tr[wave][1][TrTile1::wslot(j, q, b)] = ml[b];
          }
#pragma unroll
          for (int kc = 0; kc < KC; ++kc) {
            dbacc[s][kc] = mma32(mh[0], mh[1], at[0][kc], at[1][kc], dbacc[s][kc]);
            dbacc[s][kc] = mma32(ml[0], ml[1], at[0][kc], at[1][kc], dbacc[s][kc]);
          }
        };
        // dalpha contracts 16 channels of the hi and of the lo part in one
        // 16x16x32 MFMA against the basis operand twice.  The transposed reads of
        // a tap (ra[rb][h] = m[16 rb + i][4 qq + {0..3}]) are issued before the next
        // tap's m values are formed and written (a wave's LDS operations complete
        // in issue order, so one tile serves)
        Op ra[NB][2], bda[KC];
        stage_m(0);
#pragma unroll
        for (int s = 0; s < S; ++s) {
          wave_lds_sync();
#pragma unroll
          for (int r2 = 0; r2 < NB; ++r2)
#pragma unroll
            for (int h = 0; h < 2; ++h)
              ra[r2][h] = TrTile<NB, 2>::read(&m_tr[wave][h][TrTile1::rslot(j, q, r2)]);
#pragma unroll
          for (int kc = 0; kc < KC; ++kc) bda[kc] = b_lds[wave][s][kc][j * 4 + (q ^ (j >> 2))];
          __builtin_amdgcn_sched_barrier(0);
          if (s + 1 < S) stage_m(s + 1);
#pragma unroll
          for (int r2 = 0; r2 < NB; ++r2)
#pragma unroll
            for (int kc = 0; kc < KC; ++kc)
              dacc[r2][kc] = mma32(ra[r2][0], ra[r2][1], bda[kc], bda[kc], dacc[r2][kc]);
        }
      } else {
        // fp32: m is the dbasis A operand as it lies (row r of every stream in
        // one 16x16x4 product), its transpose for dalpha goes through the tile
        auto stage_m = [&](int s) {
#pragma unroll
          for (int r = 0; r < R; ++r) {
            const float mval = tap_ok(r, s) ? g[r] * xw[r + s] : 0.f;
            m_f32[wave][f32_mslot(R * q + r, j >> 2) + (j & 3)] = mval;
#pragma unroll
            for (int kc = 0; kc < KC; ++kc)
              dbacc[s][kc] =
                  __builtin_amdgcn_mfma_f32_16x16x4f32(mval, at[r >> 2][kc][r & 3], dbacc[s][kc], 0, 0, 0);
          }
        };
        Op ra[NB], bda[KC];
        stage_m(0);
#pragma unroll
        for (int s = 0; s < S; ++s) {
          wave_lds_sync();
#pragma unroll
          for (int r2 = 0; r2 < NB; ++r2)
            ra[r2] = *reinterpret_cast<const Op*>(&m_f32[wave][f32_mslot(16 * r2 + j, q)]);
#pragma unroll
          for (int kc = 0; kc < KC; ++kc) bda[kc] = b_lds[wave][s][kc][f32_bslot(j, q) / 4];
          __builtin_amdgcn_sched_barrier(0);
          if (s + 1 < S) stage_m(s + 1);
#pragma unroll
          for (int r2 = 0; r2 < NB; ++r2)
#pragma unroll
            for (int kc = 0; kc < KC; ++kc) dacc[r2][kc] = C::mma(ra[r2], bda[kc], dacc[r2][kc]);
        }
      }
      wave_lds_sync();
    }
    // (unconditionally, as fetch_a above); after the m products, where the fewest
    // registers are live
    if constexpr (!kFetchEarly) fetch_xdy();

#pragma unroll
    for (int r2 = 0; r2 < NB; ++r2)
#pragma unroll
      for (int kc = 0; kc < KC; ++kc)
#pragma unroll
        for (int v = 0; v < 4; ++v) da_lds[buf % DAB][wave][r2][kc][4 * q + v][j] = dacc[r2][kc][v];
    if (more) stage_alpha(buf ^ 1);
    __syncthreads();
    // sum the 8 waves' dalpha tiles in wave order; rows past the own ones drop
    {
      const int r2 = tl >> 8, row = (tl >> 4) & 15, c = tl & 15, rho = tl >> 4;
      const Buf pdb = pdw.next(R * KP * 4);
      const uint32_t off = static_cast<uint32_t>(((R * n * (rho >> 3) + (rho & 7)) * KP + c) * 4);
      float tv[KC][WPG];
#pragma unroll
      for (int kc = 0; kc < KC; ++kc)
#pragma unroll
        for (int w = 0; w < WPG; ++w) tv[kc][w] = da_lds[buf % DAB][w][r2][kc][row][c];
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) {
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < WPG; ++w) sum += tv[kc][w];
        pdb.store<4>(off + 64 * kc, &sum);
      }
      if constexpr (DAB == 1) __syncthreads();
    }
  };
  // plain steps in a loop of their own: the accumulators stay in their registers
  // there (with both forms joined in one loop body they were moved every step)
  for (int i = 0; i < n; ++i) {
    for (; i < n && __builtin_amdgcn_ballot_w64(ns <= srow + R * i + R - 1) == 0; ++i)
      step(i, std::false_type{});
    if (i < n) step(i, std::true_type{});
  }

  // the last S-1 rows of a stream: what its own rows gave them, and what the next
  // stream's first rows did (stream 3's are past the own rows and drop)
  if (dxv != nullptr) {
#pragma unroll
    for (int e = 0; e < H; ++e) {
      const int from = (lane + 16) & 63;
      const float owed = kC0Lds ? c0_lds[kC0Lds ? e : 0][kC0Lds ? (tid & ~63) | from : 0] : __shfl(c0[e], from, 64);
      const E o = C::from_f(dxa[R + e] + owed);
      dxw.next(rb).store<ESZ>(vx, &o);
    }
  }

  // this workgroup's dbasis partial: dbacc[s][kc][v] is (k = 16 kc + j, s, channel
  // d0 + 4 q + v); with D % 4 == 2 the rows are 8-byte aligned and the last group
  // of 4 half past D
  if (wave_on && d0 + 4 * q < D) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) {
        const f32x4 v = dbacc[s][kc];
        float* dst = part_db + ((static_cast<int64_t>(by) * KP + 16 * kc + j) * S + s) * D + d0 + 4 * q;
        if (D % 4 == 0) {
          *reinterpret_cast<f32x4*>(dst) = v;
        } else {
          *reinterpret_cast<f32x2*>(dst) = f32x2{v[0], v[1]};
          if (d0 + 4 * q + 2 < D) *reinterpret_cast<f32x2*>(dst + 2) = f32x2{v[2], v[3]};
        }
      }
  }
}

template <int S, int KC, bool ACT, bool DY1, bool BF>
__global__ void __launch_bounds__(64 * kLeanWPG) __attribute__((amdgpu_waves_per_eu(lean_waves(S, KC, BF))))
bwd_lean_kernel(const void* __restrict__ xv, const void* __restrict__ dyv, int64_t dys,
                const typename CT<BF>::elem* __restrict__ a_c,
                const typename CT<BF>::elem* __restrict__ b_c, void* __restrict__ dxv, float* __restrict__ part_da, float* __restrict__ part_db,
                SeqLayout seq, int64_t D, int gy, int gy1, int n_old, int n_total) {
  bwd_lean_tile<S, KC, ACT, DY1, BF>(xv, dyv, dys, a_c, b_c, dxv, part_da, part_db, seq, D,
                        static_cast<int>(blockIdx.x), static_cast<int>(blockIdx.y), gy, gy1, n_old,
                        n_total);
}

// Several layers in one launch (1-D grid, the layers' grids one after another,
// as bwd_layers_kernel maps them), so that a grouped launch returns the
// per-layer calls' results bit for bit.
template <int S, int KC, int ACT, bool DY1>
__global__ void __launch_bounds__(64 * kLeanWPG) __attribute__((amdgpu_waves_per_eu(lean_waves(S, KC))))
bwd_lean_layers_kernel(BwdLayers ly, SeqLayout seq) {
  const int blk = static_cast<int>(blockIdx.x);
  const BwdLayer* Lp = &ly.l[layer_index(ly, blk)];
  int local = blk - Lp->blk0, row = 0;
  const int gxl = Lp->gx;
  while (local >= gxl) {  // scalar: local < gx gy, at most gy - 1 steps
    local -= gxl;
    ++row;
  }
  bwd_lean_tile<S, KC, ACT, DY1, true>(Lp->x, Lp->dy, Lp->dys, static_cast<const uint16_t*>(Lp->a),
                        static_cast<const uint16_t*>(Lp->b), Lp->dx, Lp->part_da, Lp->part_db, seq,
                        Lp->D, local, row, Lp->gy, Lp->gy1, Lp->n_old, Lp->n_total, Lp->act != 0);
}

}  // namespace mfma
}  // namespace moc
