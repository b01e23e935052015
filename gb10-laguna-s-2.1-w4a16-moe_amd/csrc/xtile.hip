// Grouped GEMM with exact int4 weights on bf16 MFMA: the experts of a call
// that runs every expert on exact weights and has too many pairs to route
// itself (the sort has run).
//
// Reference kernels: _w4a16_moe_w1_fused_kernel (kernels/w4a16_moe.py:374-499)
// and _w4a16_moe_w2_kernel (:502-634).
//
// The weight operand is the integer 128 + code, exact in bf16 and one
// v_and_or_b32 per two codes (as in gemv_item.hpp); the scale multiplies the
// fp32 sum of its group, and the offset is taken off where the sum starts:
//     y += s_g * (sum_k (128 + c_k) x_k  -  136 sum_k x_k).
// v_mfma_f32_16x16x32_bf16 reduces 32 elements, one group of 32, so a group's
// sum is one MFMA (two or four of them for groups of 64 and 128) whose C
// operand is -136 sum x: another MFMA, of the activations with a constant
// -136 operand, shared by all row blocks of a wave.  A weight word costs 7
// VALU instructions (8 with the lane transposition of groups of 32) plus 4,
// 2 or 1 multiply-adds per 16 tokens by group size, where the kernel of
// mfma_item.hpp spends 17 to form bf16((c - 8) s); the result has no weight
// rounding.
//
// Activations are the A operand, weights B: lane l holds word l / 16 of a
// group of weight row l % 16 and D gives it 4 tokens of that row, so one
// register holds the row's scale.  A lane reads 16 bytes (a whole group of
// 32): the 16-row block's four lane quarters hold four different groups of
// their row.  Groups of 32 are transposed between the quarters
// (v_permlane32_swap, v_permlane16_swap: one instruction per word) so that
// each MFMA sees one group; groups of 64 take half of that, groups of 128
// none.
//
// A workgroup of 4 waves owns one tile of an expert (at most 16 TBMAX of its
// sorted pairs) and one or more row tiles of 256 weight rows, run in turn.
// A wave has 4 blocks of 16 rows, interleaved so that a lane's four rows are
// neighbours in the output (w13: 2 gate and the matching 2 up rows).  The
// tile's activation rows go through two LDS buffers of one step (128
// elements), permuted to the words' code order and stored in fragment order;
// one barrier per step.
//
// Bounds: with many pairs per expert no one unit (E=256, K=3072, N=128, 80
// pairs: w13 80 us, VALU busy 47 % and MFMA 23 % of the SIMDs' time, 433
// instructions per wave and step of which 192 are the groups' multiply-adds;
// w2 61 us, VALU 35 %, its 126 MB of partial rows at 2 TB/s), with 10 the
// memory (N=1024: w13 192 us, 4.7 TB/s of weights), with few in all the chain
// of a tile's steps (few_pairs_gemv below).
#include <limits.h>

#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "gemv_item.hpp"

namespace w4a16 {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

constexpr int kWaves = 4;
constexpr int kRB = 4;            // 16-row blocks per wave
constexpr int kXcds = 8;
constexpr int kGemvLds = 76 * 1024;

// LDS of one workgroup for tiles of at most TBMAX token blocks: two
// activation buffers of one step, each wave's packed weights of a pair of
// steps (256 bytes x 16 rows x 4 blocks, the second step's half set off by
// 128 bytes, see the weights below) and its scale window (kWin scales of 64 rows,
// 16 bytes of padding a row).
template <int TBMAX>
struct XGeo {
  static constexpr int kTBMax = TBMAX;
  static constexpr int kTileM = 16 * TBMAX;
  static constexpr int kHalf = 4096 + 128;
  static constexpr int kW = 2 * kHalf;
  static constexpr int kWin = TBMAX <= 2 ? 32 : 16;  // scales of a row per window
  static constexpr int kSRow = 2 * kWin + 16;
  static constexpr int kS = 64 * kSRow;
  static constexpr int kOffW = 2 * TBMAX * 4096;
  static constexpr int kOffS = kOffW + kWaves * kW;
  // (at least what the GEMV's items stage of rows of up to 7,360 elements)
  static constexpr int kLds = kOffS + kWaves * kS > kGemvLds ? kOffS + kWaves * kS : kGemvLds;
  static_assert(2 * (kLds + kTileM * 8) <= 160 * 1024, "two workgroups per CU");
};

__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  const f32x2_t v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}

// LDS barrier: the wave's LDS accesses are complete, its global loads stay in
// flight (a __syncthreads() fence would wait for the weight prefetch).
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

__device__ __forceinline__ float silu(float g) {
  return g * __builtin_amdgcn_rcpf(1.0f + __expf(-g));
}

// Octet (8 elements) of a step that lane quarter q meets in MFMA j, by group
// size: the quarter's word of group j (32), of group pair j / 2 (64), or word
// j of its own chunk (128).
template <int GS>
__device__ __forceinline__ int frag_octet(int j, int q) {
  if constexpr (GS == 0) return 4 * j + q;
  else if constexpr (GS == 1) return 4 * ((j & 2) | (q & 1)) + ((j & 1) | (q & 2));
  else return 4 * q + j;
}

// One tile of TB token blocks (16 slots each).  GS = log2(group / 32).  SP:
// scales per load: a row's scales are whole, aligned pieces of 8 (16 bytes) or
// 4 (8 bytes), else they are loaded one by one.
// kStaged = false: the reduction has at most two steps, which stay in the two
// buffers: the loop loads no activations and needs no barrier.
template <int MODE, int GS, int SP, int TB, class X, bool kStaged>
__device__ __forceinline__ void run_xtile(const XtileLaunch& a, int e, int rt0, int nrt,
                                          const int* s_f, const float* s_wt, int count,
                                          unsigned char* lds) {
  constexpr int kBuf = TB * 4096;   // one step of TB x 16 rows
  constexpr int kSc = GS == 0 ? 4 : GS == 1 ? 2 : 1;  // scales of a row per step
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int n = lane & 15;
  const int q = lane >> 4;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int G = a.kdim >> 5;           // 16-byte chunks of a weight row
  const int T = (G + 3) >> 2;          // steps (128 elements) of a row tile
  const int TP = (T + 1) >> 1;         // pairs of steps
  const int gpr = a.kdim / a.group;
  const int rows_total = MODE == 0 ? 2 * a.n_out : a.n_out;

  // ---- activations: thread -> row tid / 16 of every token block, octet tid % 16
  const int at = tid >> 4, ao = tid & 15;
  const char* arow[TB];
#pragma unroll
  for (int b = 0; b < TB; ++b) {
    int f = s_f[16 * b + at];
    if (16 * b + at >= count) f = s_f[0];  // padding slots: a row to load, not used
    const int64_t row = MODE == 0 ? f / a.topk : f;
    arow[b] = reinterpret_cast<const char*>(a.act + row * a.ld_act);
  }
  // Padding slots (of the last block) are zeros: their MFMAs draw less power.
  const bool pad = 16 * (TB - 1) + at >= count;
  const int n_oct = a.kdim >> 3;
  // With two register sets in turn, a step's rows are written to LDS two
  // steps after their loads were issued: loads return in order, so the wait
  // for them leaves the weight loads of two steps in flight.  (Tall tiles of
  // the larger groups have registers for one set: one step.)
  constexpr int kSets = TB <= 2 ? 2 : 1;
  constexpr bool kWhole = SP > 1 || GS == 2;  // K is a multiple of 128: no partial steps
  u32x4_t ars[kSets][TB];
  int ka = 0;  // local step of the next activation load
  bool ar_oks[kSets];
  auto load_act = [&](u32x4_t (&ar)[TB], bool& ar_ok) {
    const int o = 16 * ka + ao;
    ar_ok = o < n_oct;
    const uint32_t off = ar_ok ? (uint32_t)o * 16u : 0u;  // past the row: octet 0, not used
    ka = ka + 1 < 2 * TP ? ka + 1 : 0;
#pragma unroll
    for (int b = 0; b < TB; ++b)
      ar[b] = *reinterpret_cast<const u32x4_t*>(arow[b] + off);
  };
  // Writer position: fragment j, quarter qw of octet ao; the row is xor-ed
  // with the octet so that the 16 threads of a row write 16 bank groups.
  int aw;
  {
    const int c = ao >> 2, w = ao & 3;
    int j, qw;
    if (GS == 0) j = c, qw = w;
    else if (GS == 1) j = (c & 2) | (w & 1), qw = (c & 1) | (w & 2);
    else j = w, qw = c;
    aw = (j * 64 + qw * 16 + (at ^ ao)) * 16;
  }
  auto write_act = [&](const u32x4_t (&ar)[TB], bool ar_ok, int buf) {
#pragma unroll
    for (int b = 0; b < TB; ++b) {
      const bool ok = (kWhole || ar_ok) && (b < TB - 1 || !pad);
      const u32x4_t d = ok ? ar[b] : u32x4_t{0u, 0u, 0u, 0u};
      u32x4_t p;
      p[0] = __builtin_amdgcn_perm(d[2], d[0], 0x05040100u);  // (x0, x4)
      p[1] = __builtin_amdgcn_perm(d[2], d[0], 0x07060302u);  // (x1, x5)
      p[2] = __builtin_amdgcn_perm(d[3], d[1], 0x05040100u);  // (x2, x6)
      p[3] = __builtin_amdgcn_perm(d[3], d[1], 0x07060302u);  // (x3, x7)
      *reinterpret_cast<u32x4_t*>(lds + buf + b * 4096 + aw) = p;
    }
  };
  int rd[4];
#pragma unroll
  for (int j = 0; j < 4; ++j)
    rd[j] = (j * 64 + q * 16 + (n ^ frag_octet<GS>(j, q))) * 16;

  // ---- weights ----------------------------------------------------------------
  const char* const wexp =
      reinterpret_cast<const char*>(a.w) + (int64_t)e * rows_total * G * 16;
  const char* const sexp =
      reinterpret_cast<const char*>(a.s) + (int64_t)e * rows_total * gpr * 2;
  // Weight row of position m of block rb in row tile rt, clamped to the last
  // (rows past the end are computed and not stored).
  auto wrow = [&](int rt, int rb, int m) {
    if (MODE == 0) {
      const int col = (rt * kWaves + wid) * 32 + 2 * m + (rb & 1);
      return min(col, a.n_out - 1) + (rb < 2 ? 0 : a.n_out);
    }
    return min((rt * kWaves + wid) * 64 + 4 * m + rb, a.n_out - 1);
  };
  // Loads: a pair of steps at a time, lane l on chunk l % 8 of row l / 8 (and
  // 8 + l / 8), so that one instruction reads whole 128-byte lines, which the
  // launch never reads again: non-temporal, as the GEMV's.  (Lane l on row
  // l % 16, as the MFMA wants them, makes every lane a line of its own, and
  // lines read in halves lose with the hint: 210 against 286 us.)
  // The words go through this wave's own LDS to lane (n, q): 16-byte position
  // c of row m holds chunk c ^ ((m / 4) % 4) of its step, which spreads a
  // read of 16 rows over all banks; the 128 bytes between the steps' halves
  // do it for the writes.
  const int lm = lane >> 3, lc = lane & 7;
  unsigned char* const w_lds = lds + X::kOffW + wid * X::kW;
  int ww[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int m = 8 * h + lm;
    ww[h] = (lc >> 2) * X::kHalf + m * 64 + ((lc & 3) ^ ((m >> 2) & 3)) * 16;
  }
  const int wr = n * 64 + (q ^ ((n >> 2) & 3)) * 16;
  uint32_t woff[kRB][2];
  auto set_rows = [&](int rt) {
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        woff[rb][h] = (uint32_t)wrow(rt, rb, 8 * h + lm) * (uint32_t)G * 16u;
  };
  u32x4_t wb[kRB][2];
  int rt_l = rt0, k_l = 0;  // row tile and step pair of the next weight load
  set_rows(rt0);
  auto load_w = [&]() {
    const uint32_t c = (uint32_t)min(8 * k_l + lc, G - 1) * 16u;
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        wb[rb][h] =
            __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(wexp + (woff[rb][h] + c)));
    // the next pair; past the item's last, the expert's first line (the loads
    // stay unconditional, see below)
    if (++k_l == TP) {
      k_l = 0;
      if (++rt_l < rt0 + nrt) {
        set_rows(rt_l);
      } else {
#pragma unroll
        for (int rb = 0; rb < kRB; ++rb) woff[rb][0] = woff[rb][1] = 0;
      }
    }
  };
  auto store_w = [&]() {
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        *reinterpret_cast<u32x4_t*>(w_lds + rb * 1024 + ww[h]) = wb[rb][h];
  };
  u32x4_t wq[kRB];
  auto read_w = [&](int half) {
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb)
      wq[rb] = *reinterpret_cast<const u32x4_t*>(w_lds + half * X::kHalf + rb * 1024 + wr);
  };

  // ---- scales -----------------------------------------------------------------
  // A window of kWin scales of each of the wave's 64 rows at a time, into the
  // wave's own LDS, loaded a window ahead.  Loading each step's few scales on
  // their own cost a cache line per row and step (w13 of 256 experts with 10
  // pairs each, K=3072, N=1024: 302 us, 196 without the scale loads).
  constexpr int kWin = SP == 8 ? X::kWin : 8;  // scales of a row per window
  constexpr int kWinSteps = kWin / kSc;   // steps per window
  constexpr int kPc = kWin / 8;           // 16-byte pieces of a row's window
  const int n_win = (T + kWinSteps - 1) / kWinSteps;
  unsigned char* const s_lds = lds + X::kOffS + wid * X::kS;
  u32x4_t sreg[kPc];
  int rt_s = rt0, w_s = 0;  // row tile and window of the next scale load
  auto load_scales = [&]() {
    if constexpr (SP == 8) {  // piece lane % kPc of rows lane / kPc, ...
#pragma unroll
      for (int i = 0; i < kPc; ++i) {
        const int m = (64 / kPc) * i + lane / kPc;  // row of the wave: block m / 16
        const uint32_t r = (uint32_t)wrow(rt_s, m >> 4, m & 15);
        const uint32_t c = (uint32_t)min(kPc * w_s + lane % kPc, (gpr >> 3) - 1);
        sreg[i] = *reinterpret_cast<const u32x4_t*>(sexp + (r * (uint32_t)gpr * 2u + c * 16u));
      }
    } else if constexpr (SP == 4) {  // one row per lane
      const uint32_t r = (uint32_t)wrow(rt_s, q, n);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint32_t c = (uint32_t)min(2 * w_s + i, (gpr >> 2) - 1);
        const u32x2_t v =
            *reinterpret_cast<const u32x2_t*>(sexp + (r * (uint32_t)gpr * 2u + c * 8u));
        sreg[0][2 * i] = v[0], sreg[0][2 * i + 1] = v[1];
      }
    } else {  // any alignment: one row per lane
      const uint32_t r = (uint32_t)wrow(rt_s, q, n);
      uint32_t h[8];
#pragma unroll
      for (int i = 0; i < 8; ++i)
        h[i] = *reinterpret_cast<const uint16_t*>(
            sexp + (r * (uint32_t)gpr + (uint32_t)min(8 * w_s + i, gpr - 1)) * 2u);
#pragma unroll
      for (int i = 0; i < 4; ++i) sreg[0][i] = h[2 * i] | (h[2 * i + 1] << 16);
    }
    if (++w_s == n_win) w_s = 0, rt_s = min(rt_s + 1, rt0 + nrt - 1);
  };
  auto store_scales = [&]() {
#pragma unroll
    for (int i = 0; i < kPc; ++i)
      *reinterpret_cast<u32x4_t*>(s_lds + ((64 / kPc) * i + lane / kPc) * X::kSRow +
                                  (lane % kPc) * 16) = sreg[i];
  };
  uint32_t sc[kRB][kSc > 2 ? 2 : 1];  // the step's scales
  auto read_scales = [&](int ks) {    // ks: step within the window
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb) {
      const unsigned char* p = s_lds + (rb * 16 + n) * X::kSRow + ks * (2 * kSc);
      if constexpr (kSc == 4) {
        const u32x2_t v = *reinterpret_cast<const u32x2_t*>(p);
        sc[rb][0] = v[0], sc[rb][kSc > 2] = v[1];
      } else if constexpr (kSc == 2) {
        sc[rb][0] = *reinterpret_cast<const uint32_t*>(p);
      } else {
        sc[rb][0] = *reinterpret_cast<const uint16_t*>(p);
      }
    }
  };
  auto scale_of = [&](int rb, int i) {
    const uint32_t v = sc[rb][i >> 1];
    return __uint_as_float((i & 1) ? (v & 0xFFFF0000u) : (v << 16));
  };

  const uint32_t mask = a.nib_mask;
  uint32_t magic;
  asm volatile("v_mov_b32 %0, %1" : "=v"(magic) : "s"(a.nib_magic));
  const u32x4_t m136 = {0xC308C308u, 0xC308C308u, 0xC308C308u, 0xC308C308u};  // bf16 -136
  const bf16x8_t neg = __builtin_bit_cast(bf16x8_t, m136);

  f32x4_t acc[kRB][TB];
  auto clear = [&]() {
#pragma unroll
    for (int rb = 0; rb < kRB; ++rb)
#pragma unroll
      for (int b = 0; b < TB; ++b) acc[rb][b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  };
  clear();

  // Quarter transposition of a block's four words (see above).
  auto spread = [&](u32x4_t& w) {
    if constexpr (GS <= 1) {
      auto r0 = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
      auto r1 = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
      w[0] = r0[0], w[2] = r0[1], w[1] = r1[0], w[3] = r1[1];
    }
    if constexpr (GS == 0) {
      auto r0 = __builtin_amdgcn_permlane16_swap(w[0], w[1], false, false);
      auto r1 = __builtin_amdgcn_permlane16_swap(w[2], w[3], false, false);
      w[0] = r0[0], w[1] = r0[1], w[2] = r1[0], w[3] = r1[1];
    }
  };
  auto dequant = [&](uint32_t w) {
    const u32x4_t o = {(w & mask) | magic, ((w >> 4) & mask) | magic, ((w >> 8) & mask) | magic,
                       ((w >> 12) & mask) | magic};
    return __builtin_bit_cast(bf16x8_t, o);
  };
  constexpr int kJ = GS == 0 ? 1 : GS == 1 ? 2 : 4;  // MFMAs per group
  // Per group and row block: the MFMAs, the next block's dequantization while
  // they run, then the multiply-adds of their sums.  The scheduling barriers
  // keep the compiler from issuing every MFMA of the step first, whose sums
  // would not fit the registers.
  auto compute = [&](int buf) {
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    bf16x8_t wv[2];
    auto next_weights = [&](int i) {  // MFMA j of block rb of group g, i = (g kRB + rb) kJ + j
      const int j = i % kJ, rb = i / kJ % kRB, g = i / kJ / kRB;
      if (g == 0 && j == 0) spread(wq[rb]);
      wv[i & 1] = dequant(wq[rb][g * kJ + j]);
    };
    constexpr int kAf = TB <= 2 ? 2 : 1;  // fragments of the next group read ahead
    bf16x8_t af[kAf][kJ][TB];
    f32x4_t c[TB];
    auto read_af = [&](int g) {
#pragma unroll
      for (int j = 0; j < kJ; ++j)
#pragma unroll
        for (int b = 0; b < TB; ++b)
          af[kAf == 2 ? g & 1 : 0][j][b] =
              *reinterpret_cast<const bf16x8_t*>(lds + buf + b * 4096 + rd[g * kJ + j]);
    };
    auto offsets = [&](int g) {  // c = -136 sum x of group g
#pragma unroll
      for (int b = 0; b < TB; ++b) {
        c[b] = zero;
#pragma unroll
        for (int j = 0; j < kJ; ++j)
          c[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[kAf == 2 ? g & 1 : 0][j][b], neg, c[b], 0, 0, 0);
      }
    };
    constexpr int kG = 4 / kJ;  // groups of a step
    read_af(0);
    next_weights(0);
    offsets(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < kG; ++g) {
      if (kAf == 2 && g + 1 < kG) read_af(g + 1);
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb) {
        f32x4_t p[TB];
#pragma unroll
        for (int b = 0; b < TB; ++b) p[b] = c[b];
#pragma unroll
        for (int j = 0; j < kJ; ++j) {
          const int i = (g * kRB + rb) * kJ + j;
#pragma unroll
          for (int b = 0; b < TB; ++b)
            p[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[kAf == 2 ? g & 1 : 0][j][b], wv[i & 1], p[b], 0, 0,
                                                           0);
          if (j == kJ - 1 && rb == kRB - 1 && g + 1 < kG) {
            if (kAf == 1) read_af(g + 1);
            offsets(g + 1);
          }
          if (i + 1 < kG * kRB * kJ) next_weights(i + 1);
        }
        const float sf = scale_of(rb, g);
#pragma unroll
        for (int b = 0; b < TB; ++b)
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[rb][b][r] = fmaf(sf, p[b][r], acc[rb][b][r]);
        // pinned here: left alone, the compiler sinks the multiply-adds
        // towards the epilogue and keeps every sum alive
#pragma unroll
        for (int b = 0; b < TB; ++b) asm volatile("" : "+v"(acc[rb][b]));
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  // Outputs of row tile rt: lane (q, n) holds tokens 16 b + 4 q + r of its
  // rows; its neighbouring rows make one store per token.
  auto write_out = [&](int rt) {
    const int first = (rt * kWaves + wid) * (MODE == 0 ? 32 : 64) + (MODE == 0 ? 2 : 4) * n;
    const bool rows_ok = first < a.n_out;
    const int elt = MODE == 1 && !a.partial_bf16 ? 4 : 2;
    char* const base = static_cast<char*>(a.out) + (int64_t)first * elt;
    const int pitch = a.n_out * elt;
#pragma unroll
    for (int b = 0; b < TB; ++b) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = 16 * b + 4 * q + r;
        char* const o = base + (int64_t)s_f[t] * pitch;
        if (MODE == 0) {
          const float h0 = silu(acc[0][b][r]) * acc[2][b][r];
          const float h1 = silu(acc[1][b][r]) * acc[3][b][r];
          if (t < count && rows_ok) *reinterpret_cast<uint32_t*>(o) = pack2(h0, h1);
        } else {
          const float wt = s_wt[t];
          const float v0 = acc[0][b][r] * wt, v1 = acc[1][b][r] * wt;
          const float v2 = acc[2][b][r] * wt, v3 = acc[3][b][r] * wt;
          if (t < count && rows_ok) {
            if (a.partial_bf16)
              *reinterpret_cast<u32x2_t*>(o) = u32x2_t{pack2(v0, v1), pack2(v2, v3)};
            else
              *reinterpret_cast<f32x4_t*>(o) = f32x4_t{v0, v1, v2, v3};
          }
        }
      }
    }
  };

  // Step s: write the activations of step s + 1 (loaded kSets steps ago) into
  // the other buffer -- last read in step s - 1, before its barrier -- load
  // those of step s + 1 + kSets, compute.  The second step of a pair, once it
  // has read its weights, stores the next pair's and loads those of the pair
  // after.  The loads are unconditional, so that the compiler's waits leave
  // the newer ones in flight on every path.
  static_assert(kWinSteps % 2 == 0, "scale windows end with a pair of steps");
  load_scales();
  load_w();
  load_act(ars[0], ar_oks[0]);
  if (kSets == 2) load_act(ars[kSets - 1], ar_oks[kSets - 1]);
  // (in the order of the loop's second step: the compiler's waits are the
  // strictest over the ways into the loop, and with the weights issued before
  // the activations here each step waited for the weights just issued)
  write_act(ars[0], ar_oks[0], 0);
  load_act(ars[0], ar_oks[0]);
  store_scales();
  store_w();
  load_w();
  load_scales();
  read_w(0);
  if (!kStaged && T == 2) write_act(ars[kSets - 1], ar_oks[kSets - 1], kBuf);
  lds_barrier();
  int k = 0, ks = 0, rt = rt0;
  for (int gp = nrt * TP; gp > 0; --gp) {
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      if constexpr (kStaged) {
        constexpr int kS1 = kSets - 1;
        write_act(ars[(p + 1) & kS1], ar_oks[(p + 1) & kS1], p ? 0 : kBuf);
        load_act(ars[(p + 1) & kS1], ar_oks[(p + 1) & kS1]);
      }
      if (p == 1) {
        store_w();
        load_w();
      }
      if (p == 0 || k < T) {
        read_scales(ks);
        compute(p ? kBuf : 0);
      }
      ++k, ++ks;
      if (p == 1 && k >= T) {
        write_out(rt);
        clear();
        k = 0, ks = kWinSteps;
        ++rt;
      }
      // the next scale window, behind the newest weight loads (windows are an
      // even number of steps)
      if (p == 1 && ks == kWinSteps) {
        store_scales();
        load_scales();
        ks = 0;
      }
      read_w(p ? 0 : 1);
      if constexpr (kStaged) lds_barrier();
    }
  }
}

// ---- calls with few pairs per expert -----------------------------------------
// The host lays out a call by all its pairs; where most of them belong to
// experts elsewhere (one GPU's share of the experts), an expert is left with a
// pair or two and a tile's chain of steps is the launch: 27 us for w13 at
// K=3072 however few tiles there are, where the GEMV takes 8 to 20.  Such a
// launch runs the GEMV's items instead, its workgroups taking them in turn,
// by the counts that the sort left in the header:
//   cost   few_pairs_cost summed,
//   over   experts of more than one pass (kFewPairsOver each: of more than two),
//   experts  routed experts (one sorted block each, as over < kFewPairsOver).
// w13: while the GEMV is not bound by throughput (few_cost, by what its passes
// and a tile's steps take: set_few_pairs), or nearly every expert has one or
// two pairs.  E=32 of 256, K=3072, N=128, 25 and 48 tokens of top-10: w13 27.1
// -> 10 us, 27.2 -> 18 (the GEMV's own launch 9.8 and 17.0); the calls 44.5 ->
// 30.6 and 45.0 -> 36.7.
// w2: while no expert takes a second pass (N=1056, K=3072: 20 experts of 1, 4
// and 8 pairs 13, 17 and 29 us against 28 to 29; 240 of them 123, 151 and 297
// against 154 to 164) and, for short rows, whose tiles are short too, the
// items are few.  The branch costs the launches that run their tiles 0 to 0.3
// us, those of 16-slot tiles with groups of 64 (other registers) 0.3 to 0.7.
template <int MODE>
__device__ __forceinline__ bool few_pairs_gemv(const XtileLaunch& a, int experts, int cost,
                                               int over) {
  if (MODE == 1) return over == 0 && cost <= a.few_cost[0];
  return over < kFewPairsOver && (cost <= a.few_cost[over > 0] ||
                                  (a.few_cost[0] >= 0 && over == 0 && 4 * cost <= 9 * experts));
}

// The GEMV's shape: that of its passes of four rows (two where four do not
// fit the LDS).
constexpr int gemv_rpl(int mode) { return mode == 0 ? W4A16_W13_RPL_T4 : W4A16_W2_RPL_T4; }
constexpr int gemv_pf(int mode) { return mode == 0 ? W4A16_W13_PF_T4 : W4A16_W2_PF_T4; }
__host__ __device__ constexpr int gemv_groups(int mode, int n_out) {
  return (n_out + 8 * gemv_rpl(mode) * kWaves - 1) / (8 * gemv_rpl(mode) * kWaves);
}

// A function of its own, which gets the launch's arguments by their address
// and the workgroup's LDS by its offset, both uniform: inlined, it took scalar
// registers from the tiles (w2 of 64-slot tiles spilled 64, now 21) and a call
// of 2,048 tokens at N=128 1 us; the call costs the GEMV's launches 0.4 us.
template <int MODE, int TC>
__device__ __attribute__((noinline)) void run_gemv(uint32_t args_lo, uint32_t args_hi,
                                                   uint32_t lds_at, int first, int stride,
                                                   int experts) {
  static_assert(gemv_dev::kGemvWaves == kWaves, "workgroups of one size");
  auto uniform = [](uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); };
  const auto* a = (const __attribute__((address_space(4))) XtileLaunch*)(
      (uint64_t)uniform(args_lo) | (uint64_t)uniform(args_hi) << 32);
  auto* lds =
      (gemv_dev::u32x4_t*)(__attribute__((address_space(3))) gemv_dev::u32x4_t*)uniform(lds_at);
  GemvLaunch g{};
  g.act = a->act;
  g.ld_act = a->ld_act;
  g.w = a->w;
  g.s = a->s;
  g.sorted = a->sorted;
  g.expert_ids = a->expert_ids;
  g.header = a->header;
  g.topk_w = a->topk_w;
  g.out = a->out;
  g.partial_bf16 = a->partial_bf16;
  g.n_tok = a->n_tok;
  g.topk = a->topk;
  g.n_out = a->n_out;
  g.kdim = a->kdim;
  g.block = 16;
  g.group = a->group;
  g.nib_mask = a->nib_mask;
  g.nib_magic = a->nib_magic;
  const int items = (int)uniform(experts) * gemv_groups(MODE, g.n_out);
  const int step = (int)uniform(stride);
  for (int i = (int)uniform(first); i < items; i += step)
    gemv_dev::gemv_item<MODE, gemv_rpl(MODE), gemv_pf(MODE), TC, kWaves, 0, false, 1, 8>(g, i,
                                                                                         lds);
}

template <int MODE, int GS, int SP, class X>
__global__ __launch_bounds__(kWaves * 64) __attribute__((amdgpu_waves_per_eu(2)))
void xtile_kernel(const XtileLaunch a) {
  __shared__ __align__(16) unsigned char lds[X::kLds];
  __shared__ int s_f[X::kTileM];
  __shared__ float s_wt[X::kTileM];
  __shared__ int s_count;
  const int bid = (int)blockIdx.x;
  const int rows_per_tile = MODE == 0 ? kWaves * 32 : kWaves * 64;
  const int n_rt = (a.n_out + rows_per_tile - 1) / rows_per_tile;
  const int items = (n_rt + a.row_tiles - 1) / a.row_tiles;
  // Tiles are dealt over the 8 XCDs in rounds that alternate direction, and
  // the items of one tile run back to back on its XCD (as in mfma_item).
  const int xcd = bid % kXcds, slot = bid / kXcds;
  const int round = slot / items;
  const int tile = kXcds * round + ((round & 1) ? kXcds - 1 - xcd : xcd);
  const int experts = a.header[0] >> 4;
  if (few_pairs_gemv<MODE>(a, experts, a.header[4], a.header[5])) {
    const uint64_t args = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();  // = &a
    const uint32_t at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds;
    if (MODE == 1 || gemv_dev::gemv_lds_bytes(4, a.kdim) <= kGemvLds)
      run_gemv<MODE, 4>((uint32_t)args, (uint32_t)(args >> 32), at, (int)blockIdx.x,
                        (int)gridDim.x, experts);
    else
      run_gemv<MODE, MODE == 0 ? 2 : 4>((uint32_t)args, (uint32_t)(args >> 32), at,
                                        (int)blockIdx.x, (int)gridDim.x, experts);
    return;
  }
  if (tile >= a.header[2]) return;
  const int rt0 = (slot - round * items) * a.row_tiles;
  const int nrt = min(a.row_tiles, n_rt - rt0);
  const int info = a.tiles[tile];
  const int start = (info & 0x0FFFFFFF) << 4;
  const int blocks = min(info >> 28, X::kTBMax);
  const int e = __builtin_amdgcn_readfirstlane(a.expert_ids[start >> 4]);
  static_assert(X::kTileM <= 64, "one wave lists the tile's pairs");
  if (threadIdx.x < 64) {  // the tile's pairs are a prefix of its slots
    const int i = threadIdx.x;
    const int f = i < 16 * blocks ? a.sorted[start + i] : a.n_tok;
    const bool live = f < a.n_tok;
    if (i < X::kTileM) {
      s_f[i] = f;
      s_wt[i] = (MODE == 1 && live) ? a.topk_w[f] : 0.0f;
    }
    const int c = __popcll(ballot(live));
    if (i == 0) s_count = c;
  }
  __syncthreads();
  const int count = __builtin_amdgcn_readfirstlane(s_count);
  // (w2 of a layer sliced to N <= 256; a hidden size is not that short)
  const bool short_k = a.kdim <= 256;
#define W4A16_XTILE(TB_)                                                                   \
  case TB_:                                                                                \
    if constexpr (TB_ <= X::kTBMax) {                                                      \
      if (MODE == 1 && short_k)                                                            \
        run_xtile<MODE, GS, SP, TB_, X, MODE == 0>(a, e, rt0, nrt, s_f, s_wt, count, lds); \
      else                                                                                 \
        run_xtile<MODE, GS, SP, TB_, X, true>(a, e, rt0, nrt, s_f, s_wt, count, lds);      \
    }                                                                                      \
    break;
  switch ((count + 15) >> 4) {
    W4A16_XTILE(1)
    W4A16_XTILE(2)
    W4A16_XTILE(3)
    W4A16_XTILE(4)
    default: break;
  }
#undef W4A16_XTILE
}

template <int MODE, int GS, class X>
void launch_sp(const XtileLaunch& a, dim3 g, hipStream_t stream) {
  const dim3 b(kWaves * 64);
  const int gpr = a.kdim / a.group;
  const uintptr_t s = reinterpret_cast<uintptr_t>(a.s);
  if (gpr % 8 == 0 && s % 16 == 0)
    hipLaunchKernelGGL((xtile_kernel<MODE, GS, 8, X>), g, b, 0, stream, a);
  else if (gpr % 4 == 0 && s % 8 == 0)
    hipLaunchKernelGGL((xtile_kernel<MODE, GS, 4, X>), g, b, 0, stream, a);
  else
    hipLaunchKernelGGL((xtile_kernel<MODE, GS, 1, X>), g, b, 0, stream, a);
}

// Tiles of at most 32 slots, else of 64 (48 for groups of 128).
template <int MODE, int GS>
hipError_t launch_geo(const XtileLaunch& a, dim3 g, hipStream_t stream) {
  using Tall = XGeo<GS == 2 ? 3 : 4>;
  if (a.tile_m <= XGeo<2>::kTileM)
    launch_sp<MODE, GS, XGeo<2>>(a, g, stream);
  else if (a.tile_m <= Tall::kTileM)
    launch_sp<MODE, GS, Tall>(a, g, stream);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

// Costs up to which few_pairs_gemv takes the GEMV, for experts of at most one
// and two passes.  w13: a tile's chain takes about 3.5 + 7.6e-3 K us, the
// GEMV 0.6 of its own chain (3 + 2.75e-3 K us a pass) and 0.095 us per unit of
// cost and million weights (N K); fitted to K from 1,024 to 6,144 and N from
// 96 to 1,408, 4 to 240 experts of 1, 4 and 8 pairs (the sum of a call whose
// experts mix one and two passes stays lower: 128 of 256 experts, N=128, 64
// tokens, cost 320, GEMV 59.1 us per call, tiles 57.4).  w2: rows of one step
// (N <= 128) and of two, by their number of rows (N=128, K=3072: 20 experts
// of 1 and 4 pairs 5.6 and 7.1 us against 7.2, 48 of them 10.5 and 13.4
// against 10.3; N=192, K=6144: 48 experts 17.7 and 22.8 against 22.6 and
// 23.7, 60 of them 22.2 against 18.9); longer rows always.
template <int MODE>
void set_few_pairs(XtileLaunch& a) {
  using gemv_dev::gemv_lds_bytes;
  const bool four = gemv_lds_bytes(4, a.kdim) <= kGemvLds;
  a.few_cost[0] = a.few_cost[1] = -1;
  if (MODE == 0 && gemv_lds_bytes(2, a.kdim) <= kGemvLds) {
    const int steps = 18000000 / a.kdim;
    const int one = (62000 + steps) / a.n_out, two = (32000 + steps) / a.n_out;
    a.few_cost[0] = four ? one : two;  // (two-row passes: twice as many)
    a.few_cost[1] = four ? two : -1;
  } else if (MODE == 1 && four) {
    a.few_cost[0] = a.kdim <= 128 ? 160000 / a.n_out : a.kdim <= 256 ? 600000 / a.n_out : INT_MAX;
  }
}

template <int MODE>
hipError_t launch_xtile(const XtileLaunch& a_in, hipStream_t stream) {
  XtileLaunch a = a_in;
  a.nib_mask = 0x000F000Fu;
  a.nib_magic = 0x43004300u;  // bf16 (128, 128)
  if (a.kdim < 32 || a.kdim % 32 != 0 || a.n_out < 32 || a.n_out % 32 != 0 || a.row_tiles < 1 ||
      a.max_tiles < 0 || a.tile_m < 16)
    return hipErrorInvalidValue;
  const int rows_per_tile = MODE == 0 ? kWaves * 32 : kWaves * 64;
  const int n_rt = (a.n_out + rows_per_tile - 1) / rows_per_tile;
  const int items = (n_rt + a.row_tiles - 1) / a.row_tiles;
  int64_t grid = (int64_t)(a.max_tiles + kXcds - 1) / kXcds * kXcds * items;
  if (grid <= 0) return hipSuccess;
  set_few_pairs<MODE>(a);
  if (a.few_cost[0] >= 0)  // enough for the GEMV's items: two workgroups per CU
    grid = std::max(grid, std::min<int64_t>(512, (int64_t)a.max_tiles *
                                                     gemv_groups(MODE, a.n_out)));
  if (grid > INT32_MAX) return hipErrorInvalidValue;
  const dim3 g((unsigned)grid);
  switch (a.group) {
    case 32: return launch_geo<MODE, 0>(a, g, stream);
    case 64: return launch_geo<MODE, 1>(a, g, stream);
    case 128: return launch_geo<MODE, 2>(a, g, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

hipError_t launch_w13_xtile(const XtileLaunch& a, hipStream_t stream) {
  return launch_xtile<0>(a, stream);
}

hipError_t launch_w2_xtile(const XtileLaunch& a, hipStream_t stream) {
  return launch_xtile<1>(a, stream);
}

}  // namespace w4a16
