// eqf_lex.hip -- lexicographic Gauss-Seidel (lin_solve, fluid.rs:301-325) of
// the exact mode on gfx950, bit for bit.
//
// Work split.  The grid of S x S cells (ring included) is cut into strips of
// 63 rows.  A workgroup takes one strip of one lin_solve through up to
// LEX_KMAX = 20 sweeps (a round): lane r of a wave owns a row, each of four or
// eight waves runs up to five or three consecutive sweeps, two steps apart.  The strip moves
// up by one row from sweep to sweep: in sweep k lane r holds row j = 63 s - 1 +
// r - k.  A cell of sweep k at step t is column c = t - r - 2k.  Then everything
// a cell reads comes from its own lane or the lane before it, at an earlier
// step:
//   left  x_k(c-1, j)      own lane, step t-1
//   up    x_k(c, j-1)      lane r-1, step t-1
//   down  x_{k-1}(c, j+1)  own lane, its value after set_boundaries at t-1
//   right x_{k-1}(c+1, j)  lane r-1, the same
// Lane 0 repeats the last row of the strip above: its updated values come from
// there instead of x0, and with the rules of its row they give its final ones.
// So sweeps hand values on in registers, waves through LDS, and a strip needs
// only the strip above it (lane 63 of every sweep), never the one below: x and
// x0 are read once and x is written once for all the sweeps of a round.  The
// row shift costs K - 1 more rows per round.  Strips that do not move have to
// wait out a round trip with the strip below in every sweep, which kept the
// sweeps of a strip 32 to 64 steps apart and moved 12 bytes per cell and sweep
// through the caches: one workgroup per scene, 28.7 ms per frame at N=1024,
// 0.86 at N=128, 0.44 at N=30 (16 sweeps), 11.0 for 512 scenes of N 64..512;
// with moving strips on a CU each 1.45, 0.26, 0.12 and 5.4 ms (the other phases
// of a frame included).
//
// Lane 0 as a row of its own (63 rows per strip, one select per update) does
// away with the first lane's neighbours as operands of their own: the lane
// shifts become operands of the additions, 107 registers instead of 168 hold
// a wave of five sweeps, and two workgroups share a CU.  With 64 rows, two values
// per cell in the hand-off and the shifts as moves a frame took 2.20, 0.44, 0.18
// and 8.1 ms, where this took 1.90, 0.39, 0.16 and 5.8.
//
// AdjustRow's walls are the left / right neighbours, known one step after the
// cell: its final value is formed then (hence two steps from sweep to sweep).
// AdjustColumn runs the same code with rows and columns exchanged (the scan
// order along anti-diagonals is symmetric), so that its walls are left / right
// too.  Ring cells are cells like the others whose "update" is their fixed
// value, or in Passive the copy of the interior neighbour.  Which of these a
// block of eight steps can hold decides among four forms of the step (Class).
//
// Four or five more waves bring operands into LDS by anti-diagonals, where a step of a
// wave reads 64 neighbours, write the results, and exchange lane 63's values
// with the strips above and below, which run on other CUs: agent-scope stores
// and loads in device memory, and a progress count per strip.  (Two waves took
// 4400 cycles per block for that and three 2900, when the sweeps took 3000 and
// 2000.)  A strip trails the one above it by about 90 steps: 64 of skew, the
// blocks of 8, a store and a load; taking lane 0's values a block earlier than
// they are needed made it 8 more (N=1024 1.75 ms per frame, then 1.60).  Workgroups
// take their strip from a ticket counter whose
// order puts every strip after the one it reads from, so a waiting workgroup
// always waits for one that already runs: the launch ends whatever share of
// it is resident.
//
// Bound: a launch that fills the device by instruction issue.  For 512 scenes of N
// 64..512 and 20 sweeps the SIMDs issue a VALU instruction in 73% of their cycles
// (LDS is accessed in 25%, 7% are bank conflicts).  An update of a plain cell takes 8
// of them (6 of arithmetic, of which two shift a lane, one for lane 0, one that
// gathers lane 63's value), 180 M of a launch's 520 M; the others are steps of
// the skew and of rows beyond the grid, cells beside walls and the ring, and the waves
// that move data.  A plain block of 5 sweeps x 8 steps takes 2800 cycles with a wave
// alone on its SIMD, of which 500 are LDS reads of x0.  A lone scene is bound by its
// chain of S + 63 + 2K steps plus about 90 per strip.
//
// With few sweeps a launch that fills the device is bound by the length of a block
// (1.1 us at N=128 with one sweep, 2.0 with 20; 512 scenes: VALU 77% of the cycles with
// 20 sweeps, 49 with 4, 26 with one): the data waves' chains from barrier to barrier
// and their loads and stores of 32 bytes of a row (33 bytes per cell and solve at 2.2
// TB/s where 13 would do; without any of the fields' loads and stores a frame takes 10%
// less at N=128, 27% at N=256).  There walking the grid once per sweep, a workgroup per scene, was faster;
// us per frame then and now: 512 scenes of N=128 564 and 875 (one sweep), 763 and 961
// (4), 960 and 1060 (8), 1528 and 1556 (20); of N=256 2203 and 2997, 3115 and 3115,
// 4115 and 3229, 6886 and 3986; of N=512 7.2 and 11.3 ms, 9.6 and 11.5, 13.2 and 11.8.
// More workgroups do not help: four of two waves of sweeps per CU, for up to 8 sweeps,
// took 0.92 to 1.32 of the time of these.
//
// Compiled with -ffp-contract=off: rustc does not contract a*b+c.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "eqf_internal.h"

namespace eqf {
namespace lex {

typedef __attribute__((address_space(3))) float lf;
typedef __attribute__((address_space(3))) uint32_t lu;
typedef __attribute__((address_space(3))) uint8_t lb;
typedef uint32_t u4 __attribute__((ext_vector_type(4)));
typedef uint32_t u2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) f2 lf2;

__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }

// lane i <- lane i-1 (DPP wave_shr:1; lane 0, which has no use for it, 0).
// Where its one use is an addition the compiler makes it that addition's operand.
__device__ __forceinline__ float from_prev_lane(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x138, 0xf, 0xf, true));
}

// Lane 63 - n of `acc` <- lane 63 of v (n < 16; a constant).  Lanes below it in
// its group of four change too: called with n ascending.
template <int N>
__device__ __forceinline__ float put_lane_n(float acc, float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, acc), __builtin_bit_cast(int, v),
                                                               N == 0 ? 0xe4 : 0x100 + N, 8, 8 >> (N / 4), false));
}
__device__ __forceinline__ float put_lane(float acc, float v, int n) {
  switch (n) {
#define EQF_LANE(N) case N: return put_lane_n<N>(acc, v);
    EQF_LANE(0) EQF_LANE(1) EQF_LANE(2) EQF_LANE(3) EQF_LANE(4) EQF_LANE(5) EQF_LANE(6) EQF_LANE(7)
    EQF_LANE(8) EQF_LANE(9) EQF_LANE(10) EQF_LANE(11) EQF_LANE(12) EQF_LANE(13) EQF_LANE(14) EQF_LANE(15)
#undef EQF_LANE
  }
  return acc;
}

typedef __amdgpu_buffer_rsrc_t rsrc_t;
__device__ __forceinline__ rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  const uint64_t a = (uint64_t)(uintptr_t)base;
  const uint64_t au = (uint64_t)(uint32_t)uni((int)(uint32_t)a) | ((uint64_t)(uint32_t)uni((int)(a >> 32)) << 32);
  return __builtin_amdgcn_make_buffer_rsrc((void*)(uintptr_t)au, (short)0, uni((int)bytes), 0x00020000);
}

template <class T>
__device__ __forceinline__ T agent_load(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ void agent_store(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A workgroup with W waves of sweeps.
template <int W>
struct Lex {
static constexpr int QMAX = (LEX_KMAX + W - 1) / W, KMAX = LEX_KMAX, B = LEX_B;
// Waves that move data: with four waves of sweeps four (16 waves of two
// workgroups fill a CU), else the final values have one of their own (with the
// hand-off they took up to 3700 cycles per block, the sweeps 2600).
static constexpr int NH = W == 4 ? 4 : 5;
static constexpr int NT = 64 * (W + NH);
static_assert(QMAX <= 5 && W <= 16 && B == 8, "waves of up to five sweeps, blocks of 8 steps");
// x0 in LDS by anti-diagonals: row u = c + j - 63 s + 1 of a ring of XR rows,
// position p = j - 63 s + KMAX (sweep k at step t reads row t - 3k, lane r
// position r - k + KMAX - 1: 64 neighbours; lane 0 its value from the strip
// above, at CP + k).  Rows are numbered u + UOFF >= 0.
// A block of 8 steps may start anywhere in the ring, so the first 8 rows are
// held twice.  Live at block b (W = 4): rows 8b - 20 .. 8b + 79 (the last wave's
// last sweep, words of four rules; the rows loaded during the block).
static constexpr int CP = 84, XP = CP + KMAX, XR = (3 * (KMAX - 1) + B * W + 11 + B - 1) / B * B, UOFF = 64;
static_assert(CP >= 64 + KMAX - 1, "positions");
static constexpr int CR = XR / 4;  // rule words: four rows of one position per word, first two rows held twice
// hand-off from wave to wave: 16 step rows of 64 values; a pitch of 72 keeps the transposing accesses (8 steps x 8 lanes per
// 64) in distinct banks
static constexpr int RP = 72, RR = 16;
// LDS layout (4-byte words)
static constexpr int L_X0 = 0;
static constexpr int L_CODE = L_X0 + (XR + B) * XP;
static constexpr int L_RING = L_CODE + (CR + 2) * CP;
static constexpr int EN = W * QMAX * B;
static constexpr int L_P = L_RING + (W + 1) * RR * RP;  // lane 63's updated values: [block & 1][wave][sweep][8 steps]
static constexpr int L_CL = L_P + 2 * EN;  // class of the waves' blocks of steps, a byte each: [block & 3]
static constexpr int L_MISC = L_CL + 16;
static constexpr int L_WORDS = L_MISC + 4;
static_assert(L_WORDS * 4 <= (W == 4 ? 80 : 160) * 1024, "two workgroups per CU with four waves of sweeps");

// Selector of a cell in LDS: 0 a plain cell; ROW / COL (logical): 1 -(left),
// 2 -(right), 3 a plain one too, 4 ring (keeps its value); PASSIVE ring: 8 keeps its value, 9
// copies the left, 10 the right, 11 the upper, 12 the lower neighbour.
template <int MODE>
static __device__ __forceinline__ uint32_t selectors(uint32_t c) {  // four rule bytes -> four selectors
  if constexpr (MODE == M_PASSIVE) return ((c >> R_PAS_SHIFT) & 0x07070707u) | ((~c & 0x01010101u) << 3);
  else return ((c >> (MODE == M_COL ? R_COL_SHIFT : R_ROW_SHIFT)) & 0x03030303u) | ((~c & 0x01010101u) << 2);
}

// Values a wave carries from block to block.
struct Carry {
  float r1[QMAX];     // the cell updated at the last step
  float f2[QMAX];     // final value of the cell updated the step before it
  float lp[QMAX];     // left neighbour used at the last step
  uint32_t sp[QMAX];  // selector of the cell updated at the last step
  float in;           // the previous wave's final value of the last step
  int row;            // x0 ring row of the next block's first step, sweep k0
};

// What the cells of a block of steps may be besides plain ones:
//   C_ROWS  ring cells of the first and last row, each a fixed lane of a sweep
//           (strips at the grid's top and bottom)
//   C_RING  (Passive, every row and column holding a NoWall cell) ring cells
//           of the first and last column too: the lane whose column it is
//   C_ALL   anything, by the selectors in LDS
enum Class { C_PLAIN = 0, C_ROWS = 1, C_RING = 2, C_ALL = 3 };

// What a strip's waves know about its place.
struct Place {
  int S, base, lane;
  float a, cr;
};

// Eight steps of Q consecutive sweeps k0 .. k0+Q-1 (block m = b - w: steps 8m
// .. 8m+7).  Where no cell has a rule, a cell's final value is the updated
// one.
template <int MODE, int Q, int CLS>
static __device__ __forceinline__ void steps(lf* L, Carry& s, int b, int w, int k0, const Place& pl) {
  constexpr bool GEN = CLS == C_ALL;
  constexpr bool FIN = GEN && MODE != M_PASSIVE;  // final values other than the updated ones
  constexpr int G = 2;
  const int m = b - w, lane = pl.lane;
  const float a = pl.a, cr = pl.cr;
  const lf* x0p[Q];
  uint32_t cw[Q][2];
  bool top[Q], bot[Q];
  int c0[Q], cN[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    int row = s.row - 3 * q;
    row += row < 0 ? XR : 0;
    const int pos = KMAX - 1 - (k0 + q) + lane;
    x0p[q] = L + (L_X0 + row * XP) + (lane == 0 ? CP + k0 + q : pos);
    if constexpr (CLS == C_ROWS || CLS == C_RING) {
      top[q] = lane == k0 + q - pl.base;
      bot[q] = lane == k0 + q - pl.base + pl.S - 1;
      if constexpr (CLS == C_RING) {  // minus the columns at the block's first step
        c0[q] = lane + 2 * (k0 + q) - m * B;
        cN[q] = c0[q] + pl.S - 1;
      }
    }
    if constexpr (GEN) {
      const lu* cp = (const lu*)L + (L_CODE + (row >> 2) * CP) + pos;
      const uint32_t w0 = cp[0], w1 = cp[CP], w2 = cp[2 * CP];
      const uint32_t sh = (uint32_t)(row & 3);
      cw[q][0] = __builtin_amdgcn_alignbyte(w1, w0, sh);
      cw[q][1] = __builtin_amdgcn_alignbyte(w2, w1, sh);
    }
  }
  const lf* ri = L + (L_RING + (w * RR + (m & 1) * B) * RP) + lane;
  lf* ro = L + (L_RING + ((w + 1) * RR + (m & 1) * B) * RP) + lane;
  lf* po = L + L_P + (b & 1) * EN + w * QMAX * B;
  // Operands of G steps are read from LDS while the G before them are computed,
  // ahead of those steps' writes (the compiler cannot tell that reads and
  // writes do not overlap).
  float xin[2][G], x0v[Q][2][G];
  auto fetch = [&](int g) {
    const int h = g & 1;
#pragma unroll
    for (int ii = 0; ii < G; ++ii) {
#pragma unroll
      for (int q = 0; q < Q; ++q) x0v[q][h][ii] = x0p[q][(g * G + ii) * XP];
      xin[h][ii] = ri[(g * G + ii) * RP];
    }
  };
  fetch(0);
  float in = s.in, last[(Q + 1) / 2];
#pragma unroll
  for (int q = 0; q < Q; q += 2) last[q / 2] = 0.0f;
#pragma unroll
  for (int g = 0; g < B / G; ++g) {
    const int h = g & 1;
    if (g + 1 < B / G) fetch(g + 1);
    float out[G];
#pragma unroll
    for (int ii = 0; ii < G; ++ii) {
      const int i = g * G + ii;
      // The sweeps of a step are independent; the update goes through them
      // operation by operation, so that no instruction waits for the one
      // before it (a dependent one issues 8 cycles later instead of 4).
      float dn[Q], lt[Q], t[Q], rt[Q], up[Q], nv[Q], fin[Q];
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        dn[q] = q == 0 ? in : s.f2[q - 1];
        lt[q] = s.r1[q];
        fin[q] = s.r1[q];
        rt[q] = from_prev_lane(dn[q]);
        up[q] = from_prev_lane(s.r1[q]);
      }
      // fluid.rs:315-320; AdjustColumn: logical right / left are down / up
#pragma unroll
      for (int q = 0; q < Q; ++q) t[q] = MODE == M_COL ? up[q] + dn[q] : rt[q] + lt[q];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < Q; ++q) t[q] = MODE == M_COL ? rt[q] + t[q] : t[q] + dn[q];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < Q; ++q) t[q] = MODE == M_COL ? t[q] + lt[q] : up[q] + t[q];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < Q; ++q) t[q] = a * t[q];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < Q; ++q) t[q] = x0v[q][h][ii] + t[q];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < Q; ++q) nv[q] = t[q] * cr;
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (CLS == C_ROWS || CLS == C_RING) {
        // ring cells: their fixed value, in Passive the interior neighbour
        // (before the first sweep the ring holds what it held, not copies of
        // the right / lower neighbours)
#pragma unroll
        for (int q = 0; q < Q; ++q) {
          const bool first = q == 0 && k0 == 0;
          if constexpr (MODE == M_PASSIVE) {
            nv[q] = top[q] ? (first ? x0v[q][h][ii] : dn[q]) : nv[q];
            nv[q] = bot[q] ? up[q] : nv[q];
            if constexpr (CLS == C_RING) {
              nv[q] = c0[q] == i ? (first ? x0v[q][h][ii] : rt[q]) : nv[q];
              nv[q] = cN[q] == i ? lt[q] : nv[q];
            }
          } else {
            nv[q] = (top[q] || bot[q]) ? x0v[q][h][ii] : nv[q];
          }
        }
      }
      if constexpr (GEN) {
#pragma unroll
        for (int q = 0; q < Q; ++q) {
          const uint32_t sel = (cw[q][i >> 2] >> (8 * (i & 3))) & 255u;
          if constexpr (MODE == M_PASSIVE) {
            // before the first sweep the ring holds what it held, not copies
            // of the right / lower neighbours
            float rv = x0v[q][h][ii];
            rv = sel == 9u ? lt[q] : rv;
            rv = sel == 11u ? up[q] : rv;
            if (k0 + q > 0) {
              rv = sel == 10u ? rt[q] : rv;
              rv = sel == 12u ? dn[q] : rv;
            }
            nv[q] = sel == 0u ? nv[q] : rv;
          } else {
            nv[q] = (sel & 4u) ? x0v[q][h][ii] : nv[q];
          }
        }
      }
#pragma unroll
      for (int q = 0; q < Q; ++q) nv[q] = lane == 0 ? x0v[q][h][ii] : nv[q];
      if constexpr (FIN) {
#pragma unroll
        for (int q = 0; q < Q; ++q) {
          fin[q] = s.sp[q] == 1u ? -s.lp[q] : fin[q];
          fin[q] = s.sp[q] == 2u ? -nv[q] : fin[q];
          s.sp[q] = (cw[q][i >> 2] >> (8 * (i & 3))) & 255u;
          s.lp[q] = lt[q];
        }
      }
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        last[q / 2] = put_lane(last[q / 2], nv[q], (q & 1) * B + i);
        s.f2[q] = fin[q];
        s.r1[q] = nv[q];
      }
      out[ii] = s.f2[Q - 1];
      in = xin[h][ii];
    }
#pragma unroll
    for (int ii = 0; ii < G; ++ii) ro[(g * G + ii) * RP] = out[ii];
  }
  // lane 63's values: lane 63 - i holds step i of an even sweep, lane 55 - i of the odd one after it
#pragma unroll
  for (int q = 0; q < Q; q += 2)
    if (lane >= (q + 1 < Q ? 64 - 2 * B : 64 - B)) po[q * B + 63 - lane] = last[q / 2];
  s.in = in;
  s.row += B;
  s.row -= s.row >= XR ? XR : 0;
  if constexpr (!GEN && MODE != M_PASSIVE) {
#pragma unroll
    for (int q = 0; q < Q; ++q) s.sp[q] = 0;  // plain cells
  }
}

template <int MODE, int Q>
static __device__ __forceinline__ void steps_c(int cls, lf* L, Carry& s, int b, int w, int k0, const Place& pl) {
  if (cls == C_PLAIN) steps<MODE, Q, C_PLAIN>(L, s, b, w, k0, pl);
  else if (cls == C_ROWS) steps<MODE, Q, C_ROWS>(L, s, b, w, k0, pl);
  else if (MODE == M_PASSIVE && cls == C_RING) steps<M_PASSIVE, Q, C_RING>(L, s, b, w, k0, pl);
  else steps<MODE, Q, C_ALL>(L, s, b, w, k0, pl);
}
template <int MODE>
static __device__ __forceinline__ void steps_q(int Q, int cls, lf* L, Carry& s, int b, int w, int k0, const Place& pl) {
  if (Q == 1) steps_c<MODE, 1>(cls, L, s, b, w, k0, pl);
  else if (Q == 2) steps_c<MODE, 2>(cls, L, s, b, w, k0, pl);
  else if (QMAX == 3 || Q == 3) steps_c<MODE, 3>(cls, L, s, b, w, k0, pl);
  else if constexpr (QMAX > 3) {
    if (Q == 4) steps_c<MODE, 4>(cls, L, s, b, w, k0, pl);
    else steps_c<MODE, 5>(cls, L, s, b, w, k0, pl);
  }
}

// The sweeps of wave w of K: first sweep, count, and its first and last block of
// steps, `steps` the last step of the first sweep.
struct Part {
  int k0, Q, mlo, mhi;
};
static __device__ __forceinline__ Part part_of(int w, int steps, int K) {
  const int Wn = min(W, K);
  Part r;
  r.Q = w < Wn ? K / Wn + (w < K % Wn ? 1 : 0) : 0;
  r.k0 = w * (K / Wn) + min(w, K % Wn);
  r.mlo = max(0, (2 * r.k0 - 1) >> 3);
  r.mhi = w < Wn ? (steps + 2 * (r.k0 + r.Q - 1)) >> 3 : -1;
  return r;
}

// One strip of one round (K sweeps) of a lin_solve.  Waves 0..W-1 run the
// sweeps; waves W and on bring operands into LDS a block ahead, write the
// results, and talk to the neighbouring strips, so that their loads'
// latencies and the waits for the strip above stay out of the sweeps.
// In block b of the workgroup wave w runs block m = b - w of its steps.
template <int MODE>
static __device__ __forceinline__ void strip_task(lf* L, const RbScene& sc, const LexTask& tk, const LexSpec& sp, int K,
                                           uint32_t* __restrict__ flags,
                                           uint32_t* __restrict__ err, uint32_t polls) {
  const SceneDesc& d = sc.d;
  const int S = d.S;
  const int tid = threadIdx.x, lane = tid & 63, w = uni(tid >> 6);
  const int base = LEX_ROWS * tk.strip - 1;  // lane 0: the last row of the strip above
  const int Wn = min(W, K);
  // The last lane that has a row in some sweep bounds the steps (fewer than 64 in
  // the last strip: a frame of N=30 0.139 -> 0.130 ms, N=128 0.361 -> 0.332).
  const int steps0 = S + min(63, S - 1 + K - 1 - base);  // of the first sweep
  const int NB = ((steps0 + 2 * (K - 1)) >> 3) + 1;
  const int NI = NB + Wn;
  // LDS before the first block: lane 0's values, which nothing writes in the first strip
  for (int e = tid; e < (XR + B) * KMAX; e += NT) L[L_X0 + e / KMAX * XP + CP + e % KMAX] = 0.0f;
  if (tid < L_MISC - L_CL) ((lu*)L)[L_CL + tid] = 0;
  __syncthreads();

  if (w < W) {  // the sweeps
    const Part pt = part_of(w, steps0, K);
    const Place pl{S, base, lane, sp.coef == 0 ? d.a_visc : sp.coef == 1 ? d.a_diff : 1.0f,
                   sp.coef == 0 ? d.cr_visc : sp.coef == 1 ? d.cr_diff : 0.25f};
    Carry s;
#pragma unroll
    for (int q = 0; q < QMAX; ++q) {
      s.r1[q] = s.f2[q] = s.lp[q] = 0.0f;
      s.sp[q] = 0;
    }
    s.in = 0.0f;
    s.row = (pt.mlo * B + UOFF - 3 * pt.k0) % XR;
    for (int b = -1; b < NI; ++b) {
      const int m = b - w;
      if (m >= pt.mlo && m <= pt.mhi) {
        const int cls = uni((int)((const lb*)(L + L_CL))[(b & 3) * 16 + w]);
        steps_q<MODE>(pt.Q, cls, L, s, b, w, pt.k0, pl);
      }
      __syncthreads();
    }
    return;
  }

  float* x = d.fld + (int64_t)sp.x_role * d.fstride;
  const float* x0 = d.fld + (int64_t)sp.x0_role * d.fstride;
  // Range-checked views from FLD_PAD floats before the field (the scene's
  // allocation holds as many before field 0) to 4 floats past it: every
  // 4-element load that touches a cell of the grid lies inside.
  const uint32_t fbytes = (uint32_t)(d.fstride + FLD_PAD + 4) * 4u;
  const rsrc_t rx = make_rsrc(x - FLD_PAD, fbytes);
  const int stepc = MODE == M_COL ? S : 1;  // memory step of a logical column
  auto is_ring = [&](int c, int j) { return c == 0 || c == S - 1 || j == 0 || j == S - 1; };

  // Items of four values that follow each other in memory, which are four
  // rows of the anti-diagonal layout.  ROW / PASSIVE: one position, columns
  // c .. c+3; COL: one logical column c, positions p .. p+3.  A pass z of a
  // wave takes items 64 z + lane; a block's addresses are a lane's constant
  // plus a uniform step per block.
  const bool has_prev = tk.strip > 0, has_next = tk.strip + 1 < tk.nstrips;
  const int T = lex_blocks(S, KMAX) * B;
  // hand-off: value 64 z + lane of the EN per block, [wave][sweep][step]
  int ew[3], ek[3], ei[3], elo[3], ehi[3];
#pragma unroll
  for (int z = 0; z < 3; ++z) {
    const int e = 64 * z + lane;
    ew[z] = e / (QMAX * B);
    const Part pt = part_of(ew[z], steps0, K);
    const int q = e / B % QMAX;
    ek[z] = pt.k0 + q;
    ei[z] = e % B;
    const bool on = e < EN && q < pt.Q;
    elo[z] = on ? pt.mlo : 1;
    ehi[z] = on ? pt.mhi : 0;
  }
  const bool ring_copies = MODE == M_PASSIVE && d.ring_copies == 4 * d.N;  // every ring cell copies its neighbour
  const int hf = (lane & 1) * 4;  // the item's first row of the block's eight
  constexpr int ZI = MODE == M_COL ? 3 : 2;                          // passes
  constexpr int NIN = MODE == M_COL ? 2 * (64 + B - 1) : 2 * 64;     // items
  // x before the round, as "sweep -1": row t of ring 0, lane r: x(t + 1 - r, base + r + 1)
  int ir[ZI], ioff[ZI], oc[ZI], oj[ZI];
#pragma unroll
  for (int z = 0; z < ZI; ++z) {
    const int it = (64 * z + lane) >> 1;
    ir[z] = MODE == M_COL ? hf + it - (B - 1) : it;
    const int ic = MODE == M_COL ? B - it : hf + 1 - it;  // + 8 m
    ioff[z] = (MODE == M_COL ? ic * S + base + ir[z] + 1 : (base + ir[z] + 1) * S + ic) * 4 + FLD_PAD * 4;
    // final values have the same shape
    oc[z] = (MODE == M_COL ? B - 2 - it : hf - 1 - it) - 2 * (K - 1);  // + 8 m
    oj[z] = base + ir[z] - (K - 1);
  }
  // Final values of the round's last sweep (ring Wn, the block before) to x:
  // interior cells, and in Passive the ring cells that copy them.
  auto final_values = [&](int b) {
    if (b < Wn) return;
    const int m = b - Wn;
#pragma unroll
    for (int z = 0; z < ZI; ++z) {
      if (64 * z + lane >= NIN) continue;
      const lf* ring = L + (L_RING + (Wn * RR + (m & 1) * B) * RP) + hf * RP;
      const int c = oc[z] + m * B, j = oj[z];
      typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
      float v[4];
      bool ok[4], all = true, some = false;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int ci = MODE == M_COL ? c : c + i, ji = MODE == M_COL ? j + i : j;
        const int ri = MODE == M_COL ? min(max(ir[z] + i, 0), 63) : ir[z];
        v[i] = ring[i * RP + ri];
        ok[i] = ci >= 1 && ci <= S - 2 && ji >= 1 && ji <= S - 2 && (uint32_t)(ir[z] + (MODE == M_COL ? i : 0) - 1) < 63u;
        all = all && ok[i];
        some = some || ok[i];
      }
      f4u vv;
#pragma unroll
      for (int i = 0; i < 4; ++i) vv[i] = v[i];
      float* o = x + (MODE == M_COL ? c * S + j : j * S + c);
      if (all) {
        *(f4u*)o = vv;
      } else if (some) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (ok[i]) o[i] = v[i];
      }
      if constexpr (MODE == M_PASSIVE) {
        const int Sc = rm_code_stride(S);
        if (some && (j == 1 || j == S - 2)) {  // the rows above / below the interior
          for (int side = 0; side < 2; ++side) {
            if (j != (side ? S - 2 : 1)) continue;
            const int y = side ? S - 1 : 0;
            if (all && ring_copies) {
              *(f4u*)(x + y * S + c) = vv;
            } else {
#pragma unroll
              for (int i = 0; i < 4; ++i)
                if (ok[i] && (ring_copies || (d.code[y * Sc + c + i] >> R_PAS_SHIFT))) x[y * S + c + i] = v[i];
            }
          }
        }
        if (some && c <= 1) {  // the column left of it (c + 3 >= 1: some cell is in the interior)
          float e = v[0];
#pragma unroll
          for (int i = 1; i < 4; ++i) e = c + i == 1 ? v[i] : e;
          if (ring_copies || (d.code[j * Sc] >> R_PAS_SHIFT)) x[j * S] = e;
        }
        if (some && c + 3 >= S - 2) {  // the column right of it
          float e = v[0];
#pragma unroll
          for (int i = 1; i < 4; ++i) e = c + i == S - 2 ? v[i] : e;
          if (ring_copies || (d.code[j * Sc + S - 1] >> R_PAS_SHIFT)) x[j * S + S - 1] = e;
        }
      }
    }
  };

  if (w == W) {  // x0
    const rsrc_t rx0 = make_rsrc(x0 - FLD_PAD, fbytes);
    constexpr int NX = 2 * (CP - 1) + (MODE == M_COL ? 2 * (B - 1) : 0);
    static_assert(NX <= 192, "three passes");
    int xp0[3], xc[3], xj[3], xoff[3];
    bool xring[3];  // a ring cell by its row(s)
#pragma unroll
    for (int z = 0; z < 3; ++z) {
      const int it = (64 * z + lane) >> 1;
      xp0[z] = MODE == M_COL ? hf + it - (B - 1) : it;  // position of the first value
      xc[z] = (MODE == M_COL ? KMAX - 1 + B - 1 - it : hf - it + KMAX - 1) - UOFF;  // + 8 ub: its logical column
      xj[z] = base + xp0[z] - (KMAX - 1);                                          // its logical row
      xoff[z] = (MODE == M_COL ? xc[z] * S + xj[z] : xj[z] * S + xc[z]) * 4 + FLD_PAD * 4;
      xring[z] = MODE == M_COL ? (uint32_t)(xj[z] + 3) <= 3u || (uint32_t)(S - 1 - xj[z]) <= 3u : xj[z] == 0 || xj[z] == S - 1;
    }
    struct Rows {
      u4 x0[3], ring[3];
      bool ring_w[3];  // some item of the pass holds a ring cell (wave-uniform)
    };
    auto load = [&](Rows& t, int ub) {  // rows 8 ub - UOFF .. of x0 (for ring cells, the value they hold)
#pragma unroll
      for (int z = 0; z < 3; ++z) {
        const int c = xc[z] + ub * B, off = xoff[z] + ub * B * stepc * 4;
        // holds a ring cell (or one beyond the grid)
        const bool rg = xring[z] || (MODE == M_COL ? c == 0 || c == S - 1 : (uint32_t)(c + 3) <= 3u || (uint32_t)(S - 1 - c) <= 3u);
        t.ring_w[z] = __builtin_amdgcn_ballot_w64(rg) != 0;
        t.x0[z] = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(rx0, off, 0, 0));
        t.ring[z] = (u4)(0);
        if (t.ring_w[z]) t.ring[z] = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(rx, off, 0, 0));
      }
    };
    auto put = [&](const Rows& t, int ub) {
      const int row = (ub * B) % XR;
#pragma unroll
      for (int z = 0; z < 3; ++z) {
        uint32_t v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = t.x0[z][i];
        if (t.ring_w[z]) {
          const int c = xc[z] + ub * B;
#pragma unroll
          for (int i = 0; i < 4; ++i)
            v[i] = is_ring(MODE == M_COL ? c : c + i, MODE == M_COL ? xj[z] + i : xj[z]) ? t.ring[z][i] : v[i];
        }
        lu* q = (lu*)L + (L_X0 + row * XP) + hf * XP;
        if (64 * z + lane < NX) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            // (COL: positions outside the row go to its last slot, which nobody reads)
            const int pi = MODE == M_COL ? ((uint32_t)(xp0[z] + i) < (uint32_t)CP ? xp0[z] + i : CP - 1) : xp0[z];
            q[i * XP + pi] = v[i];
            if (row == 0) q[(XR + i) * XP + pi] = v[i];
          }
        }
      }
    };
    // First the rows of the cells left of column 0's diagonal (5 .. 7), two groups
    // in flight: a launch's start is a few memory latencies, of a solve of 32 us at
    // N=30.
    static_assert(UOFF / B == 8, "rows before the first block");
    Rows g0, g1;
    load(g0, 5);
    load(g1, 6);
    put(g0, 5);
    load(g0, 7);
    put(g1, 6);
    load(g1, 8);
    put(g0, 7);
    for (int b = -1; b < NI; ++b) {
      if (b + 1 < NB) put(g1, b + 1 + UOFF / B);
      if (b + 2 < NB) load(g1, b + 2 + UOFF / B);
      __syncthreads();
    }
    return;
  }

  if (NH > 4 && w == W + 4) {
    for (int b = -1; b < NI; ++b) {
      final_values(b);
      __syncthreads();
    }
    return;
  }

  if (w == W + 2) {  // lane 63's values for the strip below (and the final values)
    float* hout = tk.hand;
    uint32_t* fown = flags + tk.flag;
    for (int b = -1; b < NI; ++b) {
      if (has_next && b > 0) {
#pragma unroll
        for (int z = 0; z < 3; ++z) {
          const int m = b - 1 - ew[z], pb = (b - 1) & 1;
          if (m >= elo[z] && m <= ehi[z]) agent_store(hout + (ek[z] * T + m * B + ei[z]), L[L_P + pb * EN + 64 * z + lane]);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the stores are in memory: publish them
        if (lane == 0) agent_store(fown, (uint32_t)b);
      }
      if constexpr (NH == 4) final_values(b);
      __syncthreads();
    }
    if (has_next) {
      if (lane == 0) agent_store(fown, 0x7fffffffu);
      // in memory before this workgroup counts as ended (the flags are cleared then)
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    return;
  }

  if (w == W + 3) {  // the rules
    const int Sc = rm_code_stride(S);
    // the rule bytes, transposed for COL, from CODE_PAD bytes before to 8 after them
    const rsrc_t rc = make_rsrc(d.code + (MODE == M_COL ? rm_code_bytes(S) : 0) - CODE_PAD, rm_code_used(S) + CODE_PAD + 8);
    constexpr int NC = 2 * (CP - 1);
    static_assert(NC <= 192, "three passes");
    int coff[3], cc[3];
    struct Words {
      u2 c[3];
    };
#pragma unroll
    for (int z = 0; z < 3; ++z) {
      const int it = (64 * z + lane) >> 1;
      cc[z] = hf - it + KMAX - 1 - UOFF;  // + 8 ub: first logical column
      coff[z] = min(max(base + it - (KMAX - 1), 0), S - 1) * Sc + hf - it + KMAX - 1 - UOFF + CODE_PAD;
    }
    auto load = [&](Words& t, int ub) {
#pragma unroll
      for (int z = 0; z < 3; ++z)
        t.c[z] = __builtin_bit_cast(u2, __builtin_amdgcn_raw_buffer_load_b64(rc, (coff[z] + ub * B) & ~3, 0, 0));
    };
    uint32_t h_rule = 0, h_col = 0;
    auto put = [&](const Words& t, int ub) {
      const int row = (ub * B) % XR;
      uint32_t any = 0;
      bool cols = false;
#pragma unroll
      for (int z = 0; z < 3; ++z)
        if (64 * z + lane < NC) {
          const uint32_t sel = selectors<MODE>(__builtin_amdgcn_alignbyte(t.c[z].y, t.c[z].x, (uint32_t)((coff[z] + ub * B) & 3)));
          lu* cq = (lu*)L + (L_CODE + (row >> 2) * CP) + (hf >> 2) * CP + ((64 * z + lane) >> 1);
          cq[0] = sel;
          if (row == 0) cq[CR * CP] = sel;
          any |= MODE == M_PASSIVE ? sel : sel ^ (sel >> 1);  // (3 keeps its value)
          const int c = cc[z] + ub * B;
          cols = cols || (uint32_t)(c + 3) <= 3u || (uint32_t)(S - 1 - c) <= 3u;
        }
      const bool rules = MODE == M_PASSIVE ? !ring_copies && any != 0 : (any & 0x01010101u) != 0;
      h_rule = (h_rule << 1) | (__builtin_amdgcn_ballot_w64(rules) != 0 ? 1u : 0u);
      h_col = (h_col << 1) | (__builtin_amdgcn_ballot_w64(cols) != 0 ? 1u : 0u);
    };
    // Classes of the blocks that the waves run in block nb of the workgroup,
    // by the rows of x0 (8 to a bit, the newest, 8 (nb + 8), lowest) of their
    // cells and of those finished in them.
    const bool rows = base < KMAX || base + 64 > S - 1;  // a sweep holds a ring row
    uint32_t cmask;  // lane w: the bits of wave w
    {
      const Part pt = part_of(min(lane, W - 1), steps0, K);
      const int newest = 8 + min(lane, W - 1) - ((B - 1 - 3 * pt.k0 + UOFF) >> 3);
      const int oldest = 8 + min(lane, W - 1) - ((-1 - 3 * (pt.k0 + pt.Q - 1) + UOFF) >> 3);
      cmask = ((2u << oldest) - 1u) & ~((1u << newest) - 1u);
    }
    auto classes = [&](int nb) {
      uint32_t c = rows ? C_ROWS : C_PLAIN;
      c = (h_col & cmask) ? (MODE == M_PASSIVE ? C_RING : C_ALL) : c;
      c = (h_rule & cmask) ? C_ALL : c;
      if (lane < W) ((lb*)(L + L_CL))[(nb & 3) * 16 + lane] = (uint8_t)c;
    };
    Words g5, g6, g7, g;
    load(g5, 5);
    load(g6, 6);
    load(g7, 7);
    load(g, 8);
    put(g5, 5);
    put(g6, 6);
    put(g7, 7);
    for (int b = -1; b < NI; ++b) {
      if (b + 1 < NB) {
        put(g, b + 1 + UOFF / B);
      } else {
        h_rule <<= 1;
        h_col <<= 1;
      }
      classes(b + 1);
      if (b + 2 < NB) load(g, b + 2 + UOFF / B);
      __syncthreads();
    }
    return;
  }

  // x before the round, and lane 0's values from the strip above: these only in
  // the block before they are needed, since every block that they come earlier
  // puts every strip that much further behind the one above.
  const float* hin = tk.hand - (has_prev ? KMAX * T : 0);
  const uint32_t* fprev = flags + (has_prev ? tk.flag - 1 : tk.flag);
  u4 gin[ZI];
  float gu[3];
  int erow[3];  // x0 ring row of lane 0's values of the next block to be written
#pragma unroll
  for (int z = 0; z < 3; ++z) erow[z] = (ei[z] - 3 * ek[z] + UOFF + XR - B * ew[z]) % XR;
#pragma unroll
  for (int z = 0; z < ZI; ++z) gin[z] = (u4)(0);
  uint32_t credit = 0, fnext = 0;  // the strip above has published this many blocks
  bool dead = false;
  // operands of block nb of the workgroup (past the last: whatever is there, range-checked)
  auto load_in = [&](int nb) {
#pragma unroll
    for (int z = 0; z < ZI; ++z)
      gin[z] = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(rx, ioff[z] + nb * B * stepc * 4, 0, 0));
  };
  auto load_edge = [&](int nb) {
    // lane 0's values were made by the strip above in blocks up to nb + 8:
    // nb + 9 published blocks are needed
    if (has_prev) {
      const uint32_t need = (uint32_t)(nb + 9);
      credit = max(credit, (uint32_t)uni((int)fnext));
      uint32_t spins = 0;
      while (credit < need && !dead) {
        credit = (uint32_t)uni((int)agent_load(fprev));
        if (credit < need) {
          __builtin_amdgcn_s_sleep(1);
          if (++spins > polls) {  // cannot happen (see the file comment); never wait for ever
            dead = true;
            if (lane == 0) __hip_atomic_store(err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
          }
        }
      }
      asm volatile("" ::: "memory");
#pragma unroll
      for (int z = 0; z < 3; ++z) {
        const int m = nb - ew[z];
        gu[z] = 0.0f;
        // lane 0's value of step tau was made by the strip above in step tau + 63
        if (m >= elo[z] && m <= ehi[z]) {
          const int tau = m * B + ei[z];
          gu[z] = agent_load(hin + ek[z] * T + min(tau + 63, T - 1));
        }
      }
      fnext = agent_load(fprev);
    }
  };
  load_in(0);
  for (int b = -1; b < NI; ++b) {
    if (b + 1 < NB) {
#pragma unroll
      for (int z = 0; z < ZI; ++z) {
        lu* q = (lu*)L + (L_RING + ((b + 1) & 1) * B * RP) + hf * RP;
        if (64 * z + lane < NIN) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int ri = MODE == M_COL ? ((uint32_t)(ir[z] + i) < 64u ? ir[z] + i : RP - 1) : ir[z];
            const uint32_t v = gin[z][i];
            q[i * RP + ri] = v;
          }
        }
      }
    }
    load_edge(b + 1);
    load_in(b + 2);
    if (has_prev) {
#pragma unroll
      for (int z = 0; z < 3; ++z)
        if (elo[z] <= ehi[z]) {
          lf* e = L + (L_X0 + CP) + erow[z] * XP + ek[z];
          e[0] = gu[z];
          if (erow[z] < B) e[XR * XP] = gu[z];
          erow[z] += B;
          erow[z] -= erow[z] >= XR ? XR : 0;
        }
    }
    __syncthreads();
  }
}
};

template <int W>
__global__ void __launch_bounds__(Lex<W>::NT, W == 4 ? 4 : 3)
    k_lex(const RbScene* __restrict__ scs, const LexTask* __restrict__ tasks, int ntasks, LexArgs args,
          uint32_t* __restrict__ ctl, uint32_t* __restrict__ flags, int nflags, uint32_t* __restrict__ err) {
  typedef Lex<W> X;
  extern __shared__ float lex_lds[];
  lf* L = (lf*)lex_lds;
  if (threadIdx.x == 0) ((lu*)L)[X::L_MISC] = atomicAdd(&ctl[0], 1u);
  __syncthreads();
  const int t = uni((int)((lu*)L)[X::L_MISC]);
  if (t >= ntasks) {  // the counters were not zero at the start: nothing is sound then
    if (threadIdx.x == 0) __hip_atomic_store(err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    return;
  }
  const LexTask tk = tasks[t];
  const RbScene& sc = scs[tk.scene];
  const LexSpec sp = args.sp[tk.slot];
  const int K = lex_round_sweeps(args.press ? sc.d.press_iters : sc.d.diff_iters, args.round);
  if (K > 0) {
    if (sp.mode == M_ROW) X::template strip_task<M_ROW>(L, sc, tk, sp, K, flags, err, args.polls);
    else if (sp.mode == M_COL) X::template strip_task<M_COL>(L, sc, tk, sp, K, flags, err, args.polls);
    else X::template strip_task<M_PASSIVE>(L, sc, tk, sp, K, flags, err, args.polls);
  }
  // The last workgroup to end leaves the counters as the next launch needs them.
  __syncthreads();
  if (threadIdx.x == 0) ((lu*)L)[X::L_MISC] = atomicAdd(&ctl[1], 1u);
  __syncthreads();
  if (uni((int)((lu*)L)[X::L_MISC]) == ntasks - 1) {
    for (int i = threadIdx.x; i < nflags; i += X::NT) agent_store(flags + i, 0u);
    if (threadIdx.x < 2) agent_store(ctl + threadIdx.x, 0u);
  }
}

}  // namespace lex

void lex_launch(hipStream_t st, const RbScene* scs, const LexTask* tasks, int ntasks, const LexArgs& args,
                uint32_t* ctl, int nflags, uint32_t* err, int maxN, int cus) {
  if (ntasks <= 0) return;
  auto launch = [&](auto w) {
    typedef lex::Lex<decltype(w)::value> X;
    hipLaunchKernelGGL(lex::k_lex<decltype(w)::value>, dim3((unsigned)ntasks), dim3(X::NT), X::L_WORDS * 4, st, scs, tasks,
                       ntasks, args, ctl, ctl + 2, nflags, err);
  };
  // Up to one workgroup per CU the chain of blocks bounds the
  // launch: eight waves of up to three sweeps take a block faster than four of up
  // to five (a frame of N=1024 1.48 ms instead of 1.76, N=128 0.265 instead of
  // 0.318, N=30 0.120 instead of 0.131; seven 1.58 at N=1024, ten as eight).
  // Two workgroups of four fit a CU, one of eight does not leave room for
  // another, but up to three per CU the faster blocks still win (64 scenes of
  // N=256 0.93 ms instead of 1.02, 24 of N=1024 3.42 instead of 3.81, a mix of 130
  // 1.79 instead of 1.95; also where the large ones are few: one of N=200 beside 200 of
  // N=30 0.387 instead of 0.456, of N=62 0.530 instead of 0.542, four of N=400 beside
  // 200 of N=128 1.14 instead of 1.18) unless the strips are so short that filling eight
  // waves weighs (100 scenes of N=128 0.595 instead of 0.565, 300 of N=64 0.574
  // instead of 0.552).  Beyond that four waves win (the mix of 512 5.38 ms, 6.04
  // with eight).
  if (ntasks <= cus || (ntasks <= 3 * cus && maxN >= 192)) launch(std::integral_constant<int, 8>());
  else launch(std::integral_constant<int, 4>());
}

}  // namespace eqf
