// eqf_frame.hip -- the Stam frame step (fluid.rs:437-524) of one scene or of a
// group of scenes: every kernel of a frame covers all scenes of the group.
//
// The lin_solves run in the mode of the group: exact (lexicographic order,
// eqf_lex.hip) or red-black (below).
//
// Red-black: every lin_solve (fluid.rs:301-325) updates the (i+j)-even cells of a sweep
// first and the odd cells second, then applies set_boundaries, so all cells
// of one colour are independent and the whole grid is updated in parallel by
// many workgroups.  Sweeps are temporally blocked in registers (k_rb_band):
// a workgroup loads a region (its output tile plus a halo of 2T or 3T cells on
// the sides that face other tiles, band_halo_x / _y), runs T full sweeps (red, black,
// set_boundaries) on it, and writes the tile back, so x and x0 cross HBM once
// per T sweeps instead of once per sweep.  Each full sweep shrinks the valid
// region by 2 cells on every side with cells beyond it, red reading black
// neighbours and black the new red ones, and by a third one in the direction in
// which AdjustRow / AdjustColumn copy a wall neighbour.  (3 on all sides made a
// frame of N=4096 with 40 sweeps 2.72 ms instead of 2.45, N=1501 0.460 instead
// of 0.433: T=5 sweeps compute 1.6 to 1.9 times the output tile, not 2.1.)  A
// side on the grid's edge has nothing beyond it, so the first and last tiles of
// a row or column of tiles reach the edge
// with no halo there.  A pass reads one buffer and writes another (ping-pong).
//
// The other phases (divergence, gradient, advection with its row `break`, each
// with its set_boundaries, and the copy) are grid-wide kernels.  One frame is captured
// once as a HIP graph and replayed.  Results are identical to the red-black
// f32 CPU oracle bit for bit and are compared with its f64 version for
// accuracy.  Compiled with -ffp-contract=off like the exact mode.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <string>
#include <vector>

#include "eqf_internal.h"

#define GAS __attribute__((address_space(1)))



namespace eqf {
namespace rb {

__device__ __forceinline__ float rclamp(float x, float lo, float hi) {
  if (x < lo) x = lo;
  if (x > hi) x = hi;
  return x;
}
__device__ __forceinline__ int sat_idx(float f, int S) {
  if (!(f > 0.0f)) return 0;
  if (f >= (float)(S - 1)) return S - 1;
  return (int)f;
}

// Lane shifts (DPP wave_shr:1 / wave_shl:1); the lane without a source reads
// 0 (bound_ctrl).  The empty asm keeps each shift where it is written,
// executed by the whole wave (a shift moved under a divergent branch would
// read disabled lanes), and keeps selects on its result from being folded
// into the move.
__device__ __forceinline__ float from_prev_lane(float v) {
  float r = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x138, 0xf, 0xf, true));
  asm volatile("" : "+v"(r));
  return r;
}
__device__ __forceinline__ float from_next_lane(float v) {
  float r = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x130, 0xf, 0xf, true));
  asm volatile("" : "+v"(r));
  return r;
}
// Unpinned shifts for straight-line code with every lane active and no
// select on the result: the compiler may fold them into the add that uses them.
__device__ __forceinline__ float prev_lane_add(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ float next_lane_add(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x130, 0xf, 0xf, true));
}

// set_boundaries rule of one cell in one mode (k_rb_band): low nibble of the
// per-cell byte, bit 4 = the cell is interior (updated by the sweeps).
enum BandSel : uint32_t {
  BS_KEEP = 0,
  BS_NEG_LEFT = 1, BS_NEG_RIGHT = 2,   // AdjustRow, right wins (fluid.rs:151-164)
  BS_NEG_UP = 3, BS_NEG_DOWN = 4,      // AdjustColumn, up wins (fluid.rs:165-177)
  BS_LEFT = 5, BS_RIGHT = 6, BS_UP = 7, BS_DOWN = 8,  // Passive ring copies (fluid.rs:179-187)
  BS_UPD = 16,
};

// A workgroup finds its scene and its place in it with one load from a map
// of the launch's work units (band tile or block of CELL_BLOCK cells, ring
// included -> {scene, index in the scene}; segments of rows: seg_of).
// Field roles in kernel arguments: F_* (eqf_layout.h), the ping-pong fields, or none.
constexpr int ROLE_TMP = NFIELDS;  // .. + 2
constexpr int ROLE_NONE = -1;
// cells per workgroup of the whole-field kernels (256 threads x 4 cells)
constexpr int CELL_K = 4;
constexpr int CELL_BLOCK = 256 * CELL_K;

// The kernels over interior cells give a wave up to SEG cells of one row, cell
// 64 k + lane of them to lane `lane`, so that a row's place is scalar arithmetic
// and a cell costs few address instructions: with cells dealt out in row-major
// order regardless of rows, these took longer than the memory (a VALU
// instruction per cell is 0.43 us at N=4096, and a division in 64 bits per wave
// 0.3 us of a small launch).
constexpr int SEG_K = 4, SEG = 64 * SEG_K;
struct Seg {
  int j, c0, n;  // row, first column, columns (<= 0: none)
};
// Wave w's segment of a workgroup.  at: {scene, row and segment of the first
// wave's, segments per row}.
__device__ __forceinline__ Seg seg_of(const int4& at, int w, int N) {
  int j = at.y, s = at.z + w;
  while (s >= at.w) {
    s -= at.w;
    ++j;
  }
  const int c0 = 1 + s * SEG;
  return Seg{j, c0, j <= N ? min(SEG, N + 1 - c0) : 0};
}
// Element i of an array: a scalar base and a 32-bit offset (a field has at most
// 2^30 floats).
__device__ __forceinline__ float ld(const float* p, uint32_t i) {
  return *(const GAS float*)((const GAS char*)(const GAS float*)p + (size_t)(i << 2));
}
__device__ __forceinline__ void stg(float* p, uint32_t i, float v) {
  *(GAS float*)((GAS char*)(GAS float*)p + (size_t)(i << 2)) = v;
}
__device__ __forceinline__ float* role_ptr(const RbScene& s, int role) {
  return role >= ROLE_TMP ? s.tmp[role - ROLE_TMP] : s.d.fld + (int64_t)role * s.d.fstride;
}
// Tiles along one dimension of S cells for regions of W cells and output
// tiles of TX: region b starts at b*TX; the first needs no halo before it
// (the grid's edge), the last must reach the far edge.
__host__ __device__ __forceinline__ int band_span(int S, int W, int TX) {
  return S <= W ? 1 : (S - W + TX - 1) / TX + 1;
}

// Cells that T sweeps make invalid at a side of a region with cells beyond it:
// red reads black neighbours, black the new red ones, and AdjustRow /
// AdjustColumn a wall cell beside the cell in their direction.  (Passive only
// writes the grid's own ring, from the cells inside it.)
__host__ __device__ constexpr int band_halo_x(int mode, int T) { return (mode == M_ROW ? 3 : 2) * T; }
__host__ __device__ constexpr int band_halo_y(int mode, int T) { return (mode == M_COL ? 3 : 2) * T; }

// lin_solve coefficients (a, 1/c) of a scene: velocity diffusion, density
// diffusion, pressure (fluid.rs:286-294, 311, 356).
__device__ __forceinline__ void coefs(const SceneDesc& d, int coef, float& a, float& cr) {
  a = coef == 0 ? d.a_visc : coef == 1 ? d.a_diff : 1.0f;
  cr = coef == 0 ? d.cr_visc : coef == 1 ? d.cr_diff : 0.25f;
}

// A lin_solve in a pass of k_rb_band: its tiles (workgroup -> {scene, tile}),
// field roles and coefficients.
struct BandSlot {
  const int2* tmap;
  int nt, mode, src, dst, x0, coef;
};
struct BandArgs {
  BandSlot s[3];
};

// Red-black Gauss-Seidel with set_boundaries, T full sweeps per launch, all
// in registers.  A workgroup of NW waves owns a region of 128 columns x
// NW*R rows: lane l holds columns 2l and 2l+1 of its wave's band of R rows
// (x, x0 and the cell's rule byte in registers).  Horizontal neighbours come
// from the lane's other column or the neighbouring lane (DPP), vertical ones
// from the band's next register row; only the band's first and last rows
// cross waves, through LDS (double-buffered, one barrier per exchange).
// Red cells have (x + y) even; the region origin is chosen so that row i of
// every band has its red cell in column (i & 1) of the lane.  Sweeps make cells
// invalid from the sides that have cells beyond them (band_halo_x / _y), so the
// launch stores the (128 - 2 HX) x (NW*R - 2 HY) interior of its
// region, extended to the grid's edge on the sides where the region reaches
// it (tile b of a dimension: region origin b*TX, so the first region starts
// at the edge and the last one passes the far edge); the region reads one
// buffer and the tile is written to the other (ping-pong).  Corners are set
// once after the lin_solve (nothing reads them during the sweeps).
template <int MODE, int T, int NW, int R>
__device__ __forceinline__ void band_tile(float (&edg)[2][2][2][NW][64], const RbScene* __restrict__ scs,
                                          const BandSlot& sl, int L, int nsweeps) {
  const int2* __restrict__ tmap = sl.tmap;
  const int nt = sl.nt, src_role = sl.src, dst_role = sl.dst, x0_role = sl.x0, coef = sl.coef;
  constexpr int HX = band_halo_x(MODE, T), HY = band_halo_y(MODE, T), W = 128, RH = NW * R;
  constexpr int TX = W - 2 * HX, TY = RH - 2 * HY;
  static_assert(TX > 0 && TY > 0 && TX % 2 == 0 && TY % 2 == 0 && R % 2 == 0, "band geometry");
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // Tile order: workgroup L of the slot's nt, one per tile; they are dealt to
  // the 8 XCDs round-robin by linear id;
  // XCD k takes a contiguous run of the row-major tiles (scene after scene)
  // instead, so tiles that share halo columns run together on one L2.
  int t;
  {
    const int per = nt >> 3, rem = nt & 7, xcd = L & 7;
    t = __builtin_amdgcn_readfirstlane(xcd * per + min(xcd, rem) + (L >> 3));
  }
  const int2 tm = tmap[t];
  const int js = __builtin_amdgcn_readfirstlane(tm.x), tl = __builtin_amdgcn_readfirstlane(tm.y);
  const RbScene& sc = scs[js];
  const SceneDesc& d = sc.d;
  const int S = d.S, N = d.N;
  const int tiles_x = band_span(S, W, TX), tiles_y = band_span(S, RH, TY);
  const int bx = tl % tiles_x, by = tl / tiles_x;
  // Global-memory views: a row's base address is wave-uniform (scalar
  // registers), a lane's column a 32-bit offset.
  GAS const float* __restrict__ src = (GAS const float*)role_ptr(sc, src_role);
  GAS float* __restrict__ dst = (GAS float*)role_ptr(sc, dst_role);
  GAS const float* __restrict__ x0g = (GAS const float*)role_ptr(sc, x0_role);
  GAS const uint8_t* __restrict__ code = (GAS const uint8_t*)d.code;
  float a, cr;
  coefs(d, coef, a, cr);
  const int gx0 = bx * TX;  // region origin; gx0 + gy0 is even (TX, TY, R even)
  const int gyb = by * TY;
  const int gy0 = gyb + w * R;          // this wave's band
  const int gxa = gx0 + 2 * lane;
  // whether this lane's two columns are in the grid (cells outside it are
  // replaced by 0 after the loads)
  bool cin[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) cin[b] = gxa + b < S;  // gxa >= 0
  float x[R][2], x0[R][2];
  uint32_t cd[R];
  // Loads first, all of them, so that one wait covers every load of the
  // region.  Addresses: the tile's first row as one wave-uniform base per
  // array, a row's cells as a 32-bit offset from it (rows clamped into the
  // grid).  A lane's column pair is one 8-byte load per field at
  // min(gxa, S - 2) (gxa >= 0 is even): a pair that straddles the far edge
  // (odd S, gxa = S - 1) reads (S - 2, S - 1) and takes column S - 1 from the
  // second half; pairs past the edge read in-grid cells that are zeroed below.
  // The pair's rule bytes are one 2-byte load (rule rows have an even
  // stride Sc, so min(gxa, Sc - 2) is even; the straddling pair reads column
  // S - 1 and the row's pad byte).
  const int Sc = rm_code_stride(S);
  const uint32_t pc = (uint32_t)min(gxa, S - 2), pcc = (uint32_t)min(gxa, Sc - 2);
  const bool hi = gxa > S - 2;
  GAS const char* sb = (GAS const char*)(src + (int64_t)gyb * S);  // gyb <= S - 1
  GAS const char* xb = (GAS const char*)(x0g + (int64_t)gyb * S);
  GAS const uint8_t* cb = code + (int64_t)gyb * Sc;
  typedef float f2 __attribute__((ext_vector_type(2), aligned(4)));
  uint32_t cw[R];  // rule bytes of the pair, first column low
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const uint32_t rr = (uint32_t)(min(gy0 + i, S - 1) - gyb);  // gy0 >= gyb
    const uint32_t eo = rr * (uint32_t)S + pc;
    const f2 xv = *(GAS const f2*)(sb + 4u * eo);
    const f2 x0v = *(GAS const f2*)(xb + 4u * eo);
    x[i][0] = hi ? xv.y : xv.x;
    x[i][1] = xv.y;
    x0[i][0] = hi ? x0v.y : x0v.x;
    x0[i][1] = x0v.y;
    cw[i] = *(GAS const uint16_t*)(cb + (rr * (uint32_t)Sc + pcc));
  }
  // The rule byte (eqf_layout.h RuleBits) of each cell, as this mode's
  // selector; cells outside the grid (clamped loads) get none.
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int gy = gy0 + i;
    const bool rin = gy >= 0 && gy < S;  // wave-uniform
    uint32_t c2 = 0;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const bool inside = rin && cin[b];
      x[i][b] = inside ? x[i][b] : 0.0f;
      x0[i][b] = inside ? x0[i][b] : 0.0f;
      const uint32_t c = (cw[i] >> (8 * b)) & 255u;
      uint32_t sel = (c & R_INTERIOR) ? (uint32_t)BS_UPD : 0u;
      if constexpr (MODE == M_ROW) {
        const uint32_t r = (c >> R_ROW_SHIFT) & 3u;  // BS_NEG_LEFT / BS_NEG_RIGHT
        sel |= r != R_SOURCE ? r : 0u;
      }
      if constexpr (MODE == M_COL) {
        const uint32_t r = (c >> R_COL_SHIFT) & 3u;
        sel |= r && r != R_SOURCE ? r + (BS_NEG_UP - R_NEG_FIRST) : 0u;
      }
      if constexpr (MODE == M_PASSIVE) {
        const uint32_t r = (c >> R_PAS_SHIFT) & 7u;
        sel |= r ? r + (BS_LEFT - R_COPY_LEFT) : 0u;
      }
      c2 |= (inside ? sel : 0u) << (8 * b);
    }
    cd[i] = c2;
  }
  // Wave-uniform shortcuts: a band whose cells are all interior needs no
  // update mask, and one without set_boundaries rules skips that phase.
  uint32_t allu = 0xffffffffu, anys = 0;
#pragma unroll
  for (int i = 0; i < R; ++i) {
    allu &= cd[i];
    anys |= cd[i];
  }
  // two rows' selectors per register (row 2k low half, 2k+1 high half)
  uint32_t cp[R / 2];
#pragma unroll
  for (int k = 0; k < R / 2; ++k) cp[k] = cd[2 * k] | (cd[2 * k + 1] << 16);
  const bool full = __builtin_amdgcn_ballot_w64((allu & (BS_UPD | (BS_UPD << 8))) != (BS_UPD | (BS_UPD << 8))) == 0;
  const bool rules = __builtin_amdgcn_ballot_w64((anys & 0x0f0fu) != 0) != 0;

  int par = 0;
  // nsweeps >= 1: a loop without an entry test keeps the x0 loads above in the
  // first block (a skippable loop lets them sink below the other loads' wait)
  int k = 0;
  do {
#pragma unroll
    for (int ph = 0; ph < 3; ++ph) {  // red, black, set_boundaries
      // the rule bytes are loop-invariant; keeping the compilers from hoisting
      // every per-cell lane mask out of the sweep loop (into scalar registers)
#pragma unroll
      for (int k = 0; k < R / 2; ++k) asm volatile("" : "+v"(cp[k]));
      float2 ab = make_float2(0.0f, 0.0f), be = make_float2(0.0f, 0.0f);  // rows above / below the band
      if (ph < 2 || MODE != M_ROW) {
        edg[par][0][0][w][lane] = x[0][0];
        edg[par][0][1][w][lane] = x[0][1];
        edg[par][1][0][w][lane] = x[R - 1][0];
        edg[par][1][1][w][lane] = x[R - 1][1];
        __syncthreads();
        if (w > 0) ab = make_float2(edg[par][1][0][w - 1][lane], edg[par][1][1][w - 1][lane]);
        if (w < NW - 1) be = make_float2(edg[par][0][0][w + 1][lane], edg[par][0][1][w + 1][lane]);
        par ^= 1;
      }
      if (ph < 2) {
        // one colour: fluid.rs:315-320 on every cell with (x + y) % 2 == ph
        if (full) {
#pragma unroll
          for (int i = 0; i < R; ++i) {
            const int b = (i + ph) & 1;
            const float left = b ? x[i][0] : prev_lane_add(x[i][1]);
            const float right = b ? next_lane_add(x[i][0]) : x[i][1];
            const float up = i > 0 ? x[i - 1][b] : (b ? ab.y : ab.x);
            const float down = i < R - 1 ? x[i + 1][b] : (b ? be.y : be.x);
            x[i][b] = (x0[i][b] + a * (((right + left) + down) + up)) * cr;
          }
        } else {
#pragma unroll
          for (int i = 0; i < R; ++i) {
            const int b = (i + ph) & 1;
            const float left = b ? x[i][0] : from_prev_lane(x[i][1]);
            const float right = b ? from_next_lane(x[i][0]) : x[i][1];
            const float up = i > 0 ? x[i - 1][b] : (b ? ab.y : ab.x);
            const float down = i < R - 1 ? x[i + 1][b] : (b ? be.y : be.x);
            float nv = (x0[i][b] + a * (((right + left) + down) + up)) * cr;
            asm volatile("" : "+v"(nv));  // a select, not a branch around the update
            x[i][b] = (cp[i >> 1] & (BS_UPD << (16 * (i & 1) + 8 * b))) ? nv : x[i][b];
          }
        }
      } else if constexpr (MODE == M_PASSIVE) {
        // Passive set_boundaries (fluid.rs:179-187) writes ring cells only,
        // each from its interior neighbour (column 0 from column 1, column
        // S-1 from S-2, row 0 from row 1, row S-1 from S-2, where the rule
        // byte says its row / column holds a NoWall cell; corners have none),
        // so only the tiles on the grid's edge have work, at known places.
        if (bx == 0) {  // column 0: the first column of lane 0
#pragma unroll
          for (int i = 0; i < R; ++i) x[i][0] = ((cp[i >> 1] >> (16 * (i & 1))) & 15u) == BS_RIGHT ? x[i][1] : x[i][0];
        }
        if (bx == tiles_x - 1) {  // column S-1
          if (S & 1) {  // the first column of its lane: its left neighbour is in the lane before
#pragma unroll
            for (int i = 0; i < R; ++i) {
              const float l = from_prev_lane(x[i][1]);
              x[i][0] = ((cp[i >> 1] >> (16 * (i & 1))) & 15u) == BS_LEFT ? l : x[i][0];
            }
          } else {
#pragma unroll
            for (int i = 0; i < R; ++i) x[i][1] = ((cp[i >> 1] >> (16 * (i & 1) + 8)) & 15u) == BS_LEFT ? x[i][0] : x[i][1];
          }
        }
        if (gy0 == 0) {  // row 0 (R >= 2)
#pragma unroll
          for (int b = 0; b < 2; ++b) x[0][b] = ((cp[0] >> (8 * b)) & 15u) == BS_DOWN ? x[1][b] : x[0][b];
        }
        if (gy0 + R > S - 1) {  // row S-1 (only its cells carry BS_UP)
#pragma unroll
          for (int i = R - 1; i >= 0; --i) {
#pragma unroll
            for (int b = 0; b < 2; ++b) {
              const float up = i > 0 ? x[i - 1][b] : (b ? ab.y : ab.x);
              x[i][b] = ((cp[i >> 1] >> (16 * (i & 1) + 8 * b)) & 15u) == BS_UP ? up : x[i][b];
            }
          }
        }
      } else if (rules) {
        // set_boundaries AdjustRow / AdjustColumn (fluid.rs:141-178): writes
        // only NoWall cells and reads only walls, so in place is safe
#pragma unroll
        for (int i = 0; i < R; ++i) {
#pragma unroll
          for (int b = 0; b < 2; ++b) {
            const uint32_t sel = (cp[i >> 1] >> (16 * (i & 1) + 8 * b)) & 15u;
            float v = x[i][b];
            if constexpr (MODE == M_ROW) {
              const float left = b ? x[i][0] : from_prev_lane(x[i][1]);
              const float right = b ? from_next_lane(x[i][0]) : x[i][1];
              v = sel == BS_NEG_RIGHT ? -right : (sel == BS_NEG_LEFT ? -left : v);
            } else {
              const float up = i > 0 ? x[i - 1][b] : (b ? ab.y : ab.x);
              const float down = i < R - 1 ? x[i + 1][b] : (b ? be.y : be.x);
              v = sel == BS_NEG_UP ? -up : (sel == BS_NEG_DOWN ? -down : v);
            }
            x[i][b] = v;
          }
        }
      }
    }
  } while (++k < nsweeps);

  // (columns recomputed here rather than kept live through the sweeps)
  // Output tile: [gx0 + HX, gx0 + HX + TX) x [gyb + HY, gyb + HY + TY), from the
  // grid's edge for the first tile of a dimension and to its far edge for
  // the last one.
  const int gxl = bx * TX + 2 * (int)(threadIdx.x & 63);
  const int xlo = bx == 0 ? 0 : bx * TX + HX, xhi = bx == tiles_x - 1 ? S : bx * TX + HX + TX;
  const int ylo = by == 0 ? 0 : gyb + HY, yhi = by == tiles_y - 1 ? S : gyb + HY + TY;
  bool cout[2];  // this lane's columns lie in the output tile
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int gx = gxl + b;
    cout[b] = gx >= xlo && gx < xhi;
  }
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int gy = gy0 + i;
    if (gy < ylo || gy >= yhi) continue;  // wave-uniform
    GAS char* dp = (GAS char*)(dst + (int64_t)gy * S);
    if (cout[0] && cout[1]) {  // one 8-byte store; only the tile's edge lanes store singles
      f2 v;
      v.x = x[i][0];
      v.y = x[i][1];
      *(GAS f2*)(dp + 4u * (uint32_t)gxl) = v;
    } else {
#pragma unroll
      for (int b = 0; b < 2; ++b)
        if (cout[b]) *(GAS float*)(dp + 4u * (uint32_t)(gxl + b)) = x[i][b];
    }
  }
}

// One pass of up to three lin_solves that do not depend on each other: the
// tiles of one after those of the other.
template <int T, int NW, int R>
__global__ void __launch_bounds__(64 * NW)
    __attribute__((amdgpu_waves_per_eu((NW == 8 && R <= 10) ? 8 : (NW == 8 && R <= 14) ? 6 : (NW == 8 && R <= 18) ? 4 : 1)))
    k_rb_band(const RbScene* __restrict__ scs, BandArgs args, int nsweeps) {
  // [buffer][first / last row][column of the lane's pair][wave][lane]: one
  // float per lane and store, so a wave's 64 accesses hit 64 distinct banks
  __shared__ float edg[2][2][2][NW][64];
  int L = blockIdx.x, k = 0;
  while (L >= args.s[k].nt) L -= args.s[k++].nt;  // (the grid is the sum of the slots' tiles)
  const BandSlot& sl = args.s[k];
  if (sl.mode == M_ROW) band_tile<M_ROW, T, NW, R>(edg, scs, sl, L, nsweeps);
  else if (sl.mode == M_COL) band_tile<M_COL, T, NW, R>(edg, scs, sl, L, nsweeps);
  else band_tile<M_PASSIVE, T, NW, R>(edg, scs, sl, L, nsweeps);
}

// set_boundaries (fluid.rs:151-187) and its corners (fluid.rs:265-271) run
// inside the kernels that produce a field: a thread that has a cell's new value
// also writes the cells that take theirs from it, so nothing waits for a
// neighbour's thread.  On their own (a list of cells, then the corners) they
// were 12 of a frame's 25 launches, and the break columns of the two advections
// two more; a frame took 0.162 ms at N=30 (16 sweeps, exact), 0.297 at N=250
// (red-black) and takes 0.139 and 0.274.

// AdjustRow / AdjustColumn: a fluid cell beside a wall takes minus the wall
// cell's value.  It takes it from the wall cell's thread, or from the ring,
// which holds still.  Rule bytes mark the few wall cells of the interior that
// have such a neighbour.
__device__ __forceinline__ uint32_t row_rule(uint32_t c) { return (c >> R_ROW_SHIFT) & 3u; }
__device__ __forceinline__ uint32_t col_rule(uint32_t c) { return (c >> R_COL_SHIFT) & 3u; }
// Cell (i, j), rule byte c, of u (AdjustRow) and v (AdjustColumn) gets nu, nv
// (where `keep`, has what it holds).
__device__ __forceinline__ void put_ruled(const SceneDesc& d, uint32_t c, int i, int j, float* __restrict__ u,
                                          float* __restrict__ v, float nu, float nv, bool keep) {
  const int S = d.S, N = d.N, q = j * S + i, Sc = rm_code_stride(S);
  const uint32_t rr = row_rule(c), rc = col_rule(c);
  const uint8_t* code = d.code + j * Sc + i;
  if (rr == R_NEG_FIRST) {
    if (i == 1) u[q] = -u[q - 1];
  } else if (rr == R_NEG_SECOND) {
    if (i == N) u[q] = -u[q + 1];
  } else {
    if (!keep) u[q] = nu;
    if (rr == R_SOURCE) {
      if (keep) nu = u[q];
      if (row_rule(code[-1]) == R_NEG_SECOND) u[q - 1] = -nu;
      if (row_rule(code[1]) == R_NEG_FIRST) u[q + 1] = -nu;
    }
  }
  if (rc == R_NEG_FIRST) {
    if (j == 1) v[q] = -v[q - S];
  } else if (rc == R_NEG_SECOND) {
    if (j == N) v[q] = -v[q + S];
  } else {
    if (!keep) v[q] = nv;
    if (rc == R_SOURCE) {
      if (keep) nv = v[q];
      if (col_rule(code[-Sc]) == R_NEG_SECOND) v[q - S] = -nv;
      if (col_rule(code[Sc]) == R_NEG_FIRST) v[q + S] = -nv;
    }
  }
}
// Passive: ring cells of rows and columns that hold a NoWall cell take the
// interior neighbour's value; then, where `corner`, the corners, each by the
// thread that has the two ring cells it is the mean of.  For interior cell
// (i, j) beside the ring, of value val.
__device__ __forceinline__ void put_ring(const SceneDesc& d, int i, int j, float* __restrict__ x, float val,
                                         bool corner) {
  const int S = d.S, N = d.N, Sc = rm_code_stride(S);
  const bool all = d.ring_copies == 4 * N;
  auto on = [&](int rx, int ry) { return all || (d.code[ry * Sc + rx] >> R_PAS_SHIFT) != 0; };
  if (i == 1 && on(0, j)) x[j * S] = val;
  if (i == N && on(S - 1, j)) x[j * S + S - 1] = val;
  if (j == 1 && on(i, 0)) x[i] = val;
  if (j == N && on(i, S - 1)) x[(S - 1) * S + i] = val;
  if (!corner || (i != 1 && i != N) || (j != 1 && j != N)) return;
  for (int k = 0; k < 4; ++k) {
    const int cx = k & 1 ? S - 1 : 0, cy = k & 2 ? S - 1 : 0, nx = k & 1 ? N : 1, ny = k & 2 ? N : 1;
    if (i != nx || j != ny) continue;
    const float a = on(nx, cy) ? val : x[cy * S + nx], b = on(cx, ny) ? val : x[ny * S + cx];
    x[cy * S + cx] = 0.5f * (a + b);
  }
}
// ... for the values of a segment's cells (val[k]: cell 64 k + lane).
template <int K>
__device__ __forceinline__ void put_ring_seg(const SceneDesc& d, const Seg& g, int lane, float* __restrict__ x,
                                             const float (&val)[K], bool corner) {
  const int N = d.N;
  if (g.j == 1 || g.j == N) {
#pragma unroll
    for (int k = 0; k < K; ++k)
      if (64 * k + lane < g.n) put_ring(d, g.c0 + 64 * k + lane, g.j, x, val[k], corner);
  } else {
    if (g.c0 == 1 && lane == 0) put_ring(d, 1, g.j, x, val[0], false);
    if (N > 1 && g.c0 + g.n - 1 == N && lane == ((g.n - 1) & 63)) put_ring(d, N, g.j, x, val[K - 1], false);
  }
}
// Corners of a field whose ring holds still: corner k of it.
__device__ __forceinline__ void put_corner(int S, int k, float* __restrict__ x) {
  const int cx = k & 1 ? S - 1 : 0, cy = k & 2 ? S - 1 : 0, nx = k & 1 ? S - 2 : 1, ny = k & 2 ? S - 2 : 1;
  x[cy * S + cx] = 0.5f * (x[cy * S + nx] + x[ny * S + cx]);
}

// project, first half (fluid.rs:339-349), with Passive set_boundaries of both
// results and, where `corner`, the divergence's corners.  imap: workgroup ->
// its first wave's segment (seg_of).
template <int K>
__device__ __forceinline__ void div_seg(const SceneDesc& d, const Seg& g, int lane, const float* __restrict__ u,
                                        const float* __restrict__ v, float* __restrict__ dv, float* __restrict__ p,
                                        int corner) {
  const int S = d.S;
  float ur[K], ul[K], vd[K], vu[K];
  uint32_t q[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    q[k] = (uint32_t)(g.j * S + g.c0) + (uint32_t)(k < K - 1 ? 64 * k + lane : min(64 * k + lane, g.n - 1));
    ur[k] = ld(u + 1, q[k]);
    ul[k] = ld(u - 1, q[k]);
    vd[k] = ld(v + S, q[k]);
    vu[k] = ld(v - S, q[k]);
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    ur[k] = -0.5f * (ur[k] - ul[k] + vd[k] - vu[k]) / d.sf;
    if (64 * k + lane < g.n) {
      stg(dv, q[k], ur[k]);
      stg(p, q[k], 0.0f);
      ul[k] = 0.0f;
    }
  }
  put_ring_seg<K>(d, g, lane, dv, ur, corner != 0);
  put_ring_seg<K>(d, g, lane, p, ul, false);
}
__global__ void __launch_bounds__(256) k_div(const RbScene* __restrict__ scs, const int4* __restrict__ imap,
                                             int u_role, int v_role, int div_role, int p_role, int corner) {
  const int4 at = imap[blockIdx.x];
  const RbScene& sc = scs[at.x];
  const int lane = threadIdx.x & 63;
  const Seg g = seg_of(at, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), sc.d.N);
  const float *u = role_ptr(sc, u_role), *v = role_ptr(sc, v_role);
  float *dv = role_ptr(sc, div_role), *p = role_ptr(sc, p_role);
  if (g.n > 192) div_seg<4>(sc.d, g, lane, u, v, dv, p, corner);
  else if (g.n > 128) div_seg<3>(sc.d, g, lane, u, v, dv, p, corner);
  else if (g.n > 64) div_seg<2>(sc.d, g, lane, u, v, dv, p, corner);
  else if (g.n > 0) div_seg<1>(sc.d, g, lane, u, v, dv, p, corner);
}

// project, second half (fluid.rs:364-371), with set_boundaries of both results
// and their corners (their ring cells hold still); the corners of p too where
// `pc`, and those of the field c_role (ROLE_NONE: none) where the scene's
// diffusion has sweeps.  imap as for k_div.
template <int K>
__device__ __forceinline__ void grad_seg(const SceneDesc& d, const Seg& g, int lane, float* __restrict__ u,
                                         float* __restrict__ v, const float* __restrict__ p) {
  const int S = d.S;
  const uint8_t* code = d.code + (g.j * rm_code_stride(S) + g.c0);
  float uq[K], vq[K], pr[K], pl[K], pd[K], pu[K];
  uint32_t q[K], c[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const uint32_t o = (uint32_t)(k < K - 1 ? 64 * k + lane : min(64 * k + lane, g.n - 1));
    q[k] = (uint32_t)(g.j * S + g.c0) + o;
    uq[k] = ld(u, q[k]);
    vq[k] = ld(v, q[k]);
    pr[k] = ld(p + 1, q[k]);
    pl[k] = ld(p - 1, q[k]);
    pd[k] = ld(p + S, q[k]);
    pu[k] = ld(p - S, q[k]);
    c[k] = code[o];
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    uq[k] = uq[k] - 0.5f * (pr[k] - pl[k]) * d.sf;
    vq[k] = vq[k] - 0.5f * (pd[k] - pu[k]) * d.sf;
    const bool in = 64 * k + lane < g.n;
    if (in && c[k] == R_INTERIOR) {
      stg(u, q[k], uq[k]);
      stg(v, q[k], vq[k]);
    } else if (in) {
      put_ruled(d, c[k], g.c0 + 64 * k + lane, g.j, u, v, uq[k], vq[k], false);
    }
  }
}
__global__ void __launch_bounds__(256) k_grad(const RbScene* __restrict__ scs, const int4* __restrict__ imap,
                                              int u_role, int v_role, int p_role, int pc, int c_role) {
  const int4 at = imap[blockIdx.x];
  const RbScene& sc = scs[at.x];
  const int S = sc.d.S, lane = threadIdx.x & 63;
  const Seg g = seg_of(at, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), sc.d.N);
  float *u = role_ptr(sc, u_role), *v = role_ptr(sc, v_role);
  const float* p = role_ptr(sc, p_role);
  if (at.y == 1 && at.z == 0 && threadIdx.x >= 240) {  // 16 threads: corner k of up to four fields
    const int k = threadIdx.x & 3, f = (threadIdx.x >> 2) & 3;
    const int role = f == 0 ? u_role : f == 1 ? v_role : f == 2 ? (pc ? p_role : ROLE_NONE)
                                                                : (sc.d.diff_iters > 0 ? c_role : ROLE_NONE);
    if (role != ROLE_NONE) put_corner(S, k, role_ptr(sc, role));
  }
  if (g.n > 192) grad_seg<4>(sc.d, g, lane, u, v, p);
  else if (g.n > 128) grad_seg<3>(sc.d, g, lane, u, v, p);
  else if (g.n > 64) grad_seg<2>(sc.d, g, lane, u, v, p);
  else if (g.n > 0) grad_seg<1>(sc.d, g, lane, u, v, p);
}

struct Trace {
  int i0, i1, j0, j1;
  float s0, s1, t0, t1;
  bool trig;
};
__device__ __forceinline__ Trace back_trace(const SceneDesc& d, int c, int j, float uu, float vv) {
  Trace r;
  float x = (float)c - d.dt0 * uu;
  float y = (float)j - d.dt0 * vv;
  x = rclamp(x, 0.5f, d.sfm1);
  y = rclamp(y, 0.5f, d.sfm1);
  const float i0 = floorf(x), i1 = i0 + 1.0f, j0 = floorf(y), j1 = j0 + 1.0f;
  r.s1 = x - i0;
  r.s0 = 1.0f - r.s1;
  r.t1 = y - j0;
  r.t0 = 1.0f - r.t1;
  r.trig = (i1 >= d.sf) || (j1 >= d.sf);
  r.i0 = sat_idx(i0, d.S);
  r.i1 = sat_idx(i1, d.S);
  r.j0 = sat_idx(j0, d.S);
  r.j1 = sat_idx(j1, d.S);
  return r;
}
__device__ __forceinline__ float gather(const float* __restrict__ d0, const Trace& r, int S) {
  const uint32_t a = (uint32_t)(r.j0 * S), b = (uint32_t)(r.j1 * S);
  return r.s0 * (r.t0 * ld(d0, a + r.i0) + r.t1 * ld(d0, b + r.i0)) +
         r.s1 * (r.t0 * ld(d0, a + r.i1) + r.t1 * ld(d0, b + r.i1));
}

// advect (fluid.rs:385-434) for one field (DENSITY: Passive set_boundaries and
// the corners after it) or the two velocities (AdjustRow / AdjustColumn after
// it).  A row stops at the first column whose back-trace reaches the far edge
// (the `break` of fluid.rs:420-423): that cell copies its left neighbour's
// value, cells right of it keep the buffer's content.  So the waves of a row
// (R to a workgroup of NW; amap: its first row) first agree on the break
// column, by lanes where a wave has the row alone, else in LDS, and then gather;
// a segment's velocities stay in registers between the two, except where a row
// has more than SEG * NW cells: they are read again (from the cache).
template <bool DENSITY>
struct AdvArgs {
  const float *d0, *d1, *u, *v;
  float *o0, *o1;
};
// First column of the segment whose back-trace reaches the far edge (N + 1: none).
template <int K>
__device__ __forceinline__ int seg_break(const SceneDesc& d, const Seg& g, int lane, const float (&uu)[K],
                                         const float (&vv)[K]) {
  int tr = d.N + 1;
#pragma unroll
  for (int k = K - 1; k >= 0; --k) {
    const bool t = 64 * k + lane < g.n && back_trace(d, g.c0 + 64 * k + lane, g.j, uu[k], vv[k]).trig;
    const uint64_t m = __builtin_amdgcn_ballot_w64(t);
    tr = m ? g.c0 + 64 * k + (int)__builtin_ctzll(m) : tr;
  }
  return tr;
}
template <int K>
__device__ __forceinline__ void seg_load(const SceneDesc& d, const Seg& g, int lane, const float* __restrict__ u,
                                         const float* __restrict__ v, float (&uu)[K], float (&vv)[K]) {
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const uint32_t q = (uint32_t)(g.j * d.S + g.c0) + (uint32_t)min(64 * k + lane, g.n - 1);
    uu[k] = ld(u, q);
    vv[k] = ld(v, q);
  }
}
template <bool DENSITY, int K>
__device__ __forceinline__ void seg_gather(const SceneDesc& d, const Seg& g, int lane, int tr, const AdvArgs<DENSITY>& a,
                                           float (&uu)[K], float (&vv)[K]) {
  const int S = d.S;
  const uint8_t* code = d.code + (g.j * rm_code_stride(S) + g.c0);
  float* __restrict__ o0 = a.o0;
  float* __restrict__ o1 = a.o1;
  float r0[K], r1[K];
  uint32_t c[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int o = min(64 * k + lane, g.n - 1), i = g.c0 + o, row = g.j * S;
    int b = i;
    if (tr <= g.c0 + 64 * k + 63 && i == tr && i > 1) {  // (the first: the same for all lanes)
      b = i - 1;
      uu[k] = a.u[row + b];
      vv[k] = a.v[row + b];
    }
    const Trace t = back_trace(d, b, g.j, uu[k], vv[k]);
    r0[k] = gather(a.d0, t, S);
    if constexpr (!DENSITY) {
      r1[k] = gather(a.d1, t, S);
      c[k] = code[o];
    }
    if (tr == 1 && i == 1) {  // trigger in column 1: copies the ring cell d(0, j)
      r0[k] = o0[row];
      if constexpr (!DENSITY) r1[k] = o1[row];
    }
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int i = g.c0 + 64 * k + lane;
    const uint32_t q = (uint32_t)(g.j * S + i);
    const bool in = 64 * k + lane < g.n, keep = i > tr;
    if constexpr (DENSITY) {
      if (in && !keep) stg(o0, q, r0[k]);
      else if (in && (i == 1 || i == d.N || g.j == 1 || g.j == d.N)) r0[k] = o0[q];
    } else {
      if (in && c[k] == R_INTERIOR) {
        if (!keep) {
          stg(o0, q, r0[k]);
          stg(o1, q, r1[k]);
        }
      } else if (in) {
        put_ruled(d, c[k], i, g.j, o0, o1, r0[k], r1[k], keep);
      }
    }
  }
  if constexpr (DENSITY) put_ring_seg<K>(d, g, lane, o0, r0, true);
}
template <bool DENSITY, int K>
__device__ __forceinline__ void adv_row(const SceneDesc& d, const Seg& g, int lane, const AdvArgs<DENSITY>& a) {
  float uu[K], vv[K];
  seg_load<K>(d, g, lane, a.u, a.v, uu, vv);
  seg_gather<DENSITY, K>(d, g, lane, seg_break<K>(d, g, lane, uu, vv), a, uu, vv);
}
template <bool DENSITY, int NW>
__global__ void __launch_bounds__(64 * NW) k_adv(const RbScene* __restrict__ scs, const int4* __restrict__ amap,
                                                 int o0_role, int i0_role, int o1_role, int i1_role, int u_role,
                                                 int v_role) {
  __shared__ int brk;
  const int4 at = amap[blockIdx.x];
  const RbScene& sc = scs[at.x];
  const SceneDesc& d = sc.d;
  const int N = d.N, lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  AdvArgs<DENSITY> a;
  a.d0 = role_ptr(sc, i0_role);
  a.d1 = DENSITY ? nullptr : role_ptr(sc, i1_role);
  a.u = role_ptr(sc, u_role);
  a.v = role_ptr(sc, v_role);
  a.o0 = role_ptr(sc, o0_role);
  a.o1 = DENSITY ? nullptr : role_ptr(sc, o1_role);
  if (N <= SEG) {  // a row per wave
    const Seg g{at.y + w, 1, at.y + w <= N ? N : 0};
    if (g.n > 192) adv_row<DENSITY, 4>(d, g, lane, a);
    else if (g.n > 128) adv_row<DENSITY, 3>(d, g, lane, a);
    else if (g.n > 64) adv_row<DENSITY, 2>(d, g, lane, a);
    else if (g.n > 0) adv_row<DENSITY, 1>(d, g, lane, a);
    return;
  }
  if (threadIdx.x == 0) brk = N + 1;
  __syncthreads();
  constexpr int STEP = SEG * NW;
  float uu[SEG_K], vv[SEG_K];
  for (int c0 = 1 + w * SEG; c0 <= N; c0 += STEP) {
    const Seg g{at.y, c0, min(SEG, N + 1 - c0)};
    seg_load<SEG_K>(d, g, lane, a.u, a.v, uu, vv);
    const int tr = seg_break<SEG_K>(d, g, lane, uu, vv);
    if (tr <= N && lane == 0) atomicMin(&brk, tr);
  }
  __syncthreads();
  const int tr = __builtin_amdgcn_readfirstlane(brk);
  for (int c0 = 1 + w * SEG; c0 <= N; c0 += STEP) {
    const Seg g{at.y, c0, min(SEG, N + 1 - c0)};
    if (N > STEP) seg_load<SEG_K>(d, g, lane, a.u, a.v, uu, vv);
    if (g.n > 192) {
      seg_gather<DENSITY, SEG_K>(d, g, lane, tr, a, uu, vv);
    } else {
      float u1[3] = {uu[0], uu[1], uu[2]}, v1[3] = {vv[0], vv[1], vv[2]};
      if (g.n > 128) {
        seg_gather<DENSITY, 3>(d, g, lane, tr, a, u1, v1);
      } else {
        float u2[2] = {uu[0], uu[1]}, v2[2] = {vv[0], vv[1]}, u3[1] = {uu[0]}, v3[1] = {vv[0]};
        if (g.n > 64) seg_gather<DENSITY, 2>(d, g, lane, tr, a, u2, v2);
        else seg_gather<DENSITY, 1>(d, g, lane, tr, a, u3, v3);
      }
    }
  }
}

// Frame sources (only the fields that were set; adding 0 would turn -0 into
// +0) over every cell of every scene.  cmap: workgroup -> {scene, block of
// CELL_BLOCK cells}; each thread loads its CELL_K cells (256 apart) before
// storing any.
__device__ __forceinline__ void add_field(float* __restrict__ f, const float* __restrict__ a, int64_t e0,
                                          int64_t cells) {
  float x[CELL_K], y[CELL_K];
#pragma unroll
  for (int k = 0; k < CELL_K; ++k) {
    const int64_t e = min(e0 + k * 256, cells - 1);
    x[k] = f[e];
    y[k] = a[e];
  }
#pragma unroll
  for (int k = 0; k < CELL_K; ++k)
    if (e0 + k * 256 < cells) f[e0 + k * 256] = x[k] + y[k];
}
__global__ void __launch_bounds__(256) k_sources(const RbScene* __restrict__ scs, const int2* __restrict__ cmap) {
  const int2 cm = cmap[blockIdx.x];
  const SceneDesc& d = scs[cm.x].d;
  const int m = d.has_src;
  if (!m) return;
  const int64_t n = d.fstride, cells = (int64_t)d.S * d.S;
  const int64_t e0 = (int64_t)cm.y * CELL_BLOCK + threadIdx.x;
  if (m & 1) {
    float a[CELL_K], x[CELL_K], y[CELL_K];
#pragma unroll
    for (int k = 0; k < CELL_K; ++k) {
      const int64_t e = min(e0 + k * 256, cells - 1);
      a[k] = d.src[e];
      x[k] = d.fld[F_D * n + e];
      y[k] = d.fld[F_SC * n + e];
    }
#pragma unroll
    for (int k = 0; k < CELL_K; ++k)
      if (e0 + k * 256 < cells) {
        d.fld[F_D * n + e0 + k * 256] = x[k] + a[k];
        d.fld[F_SC * n + e0 + k * 256] = y[k] + a[k];
      }
  }
  if (m & 2) add_field(d.fld + F_U * n, d.src + n, e0, cells);
  if (m & 4) add_field(d.fld + F_V * n, d.src + 2 * n, e0, cells);
}

// dst = src over every cell of every scene (cmap as for k_sources), for up to
// three pairs of fields (ROLE_NONE: fewer).
struct CopyArgs {
  int dst[3], src[3];
};
__global__ void __launch_bounds__(256) k_copy(const RbScene* __restrict__ scs, const int2* __restrict__ cmap,
                                              CopyArgs args) {
  const int2 cm = cmap[blockIdx.x];
  const RbScene& sc = scs[cm.x];
  const int64_t cells = (int64_t)sc.d.S * sc.d.S;
  const int64_t e0 = (int64_t)cm.y * CELL_BLOCK + threadIdx.x;
  for (int f = 0; f < 3 && args.dst[f] != ROLE_NONE; ++f) {
    const float* __restrict__ src = role_ptr(sc, args.src[f]);
    float* __restrict__ dst = role_ptr(sc, args.dst[f]);
    float x[CELL_K];
#pragma unroll
    for (int k = 0; k < CELL_K; ++k) x[k] = src[min(e0 + k * 256, cells - 1)];
#pragma unroll
    for (int k = 0; k < CELL_K; ++k)
      if (e0 + k * 256 < cells) dst[e0 + k * 256] = x[k];
  }
}

// A scene's entry of the tables.
__global__ void k_put_scene(RbScene* __restrict__ at, RbScene v) { *at = v; }

}  // namespace rb

// ------------------------------------------------------------------ host --
// A launch group: its scenes and the prefix tables of their work units, in
// one device buffer written before any frame is captured.
struct RbGroup {
  std::vector<eqf_scene*> scenes;  // largest first
  hipStream_t stream = nullptr;    // null: each frame runs on scenes[0]'s stream
  void* d_tab = nullptr;
  size_t tab_bytes = 0;
  std::vector<char> h_tab;  // host image of the tables
  RbScene* d_scs = nullptr;
  // work unit -> {scene, index in it}: band tiles, cell blocks; -> {scene, row,
  // segment, segments per row}: segments of rows, rows
  int2 *d_tmap[3] = {nullptr, nullptr, nullptr}, *d_cmap = nullptr;
  int4 *d_imap = nullptr, *d_amap = nullptr;
  // exact mode: strips of the three diffusions (of one of them where a scene has
  // one slot) and of a pressure solve, in ticket order; counters; where a wait
  // reports that it gave up
  bool exact = false;
  LexTask *d_ldiff = nullptr, *d_lpress = nullptr;
  int n_ldiff = 0, n_lpress = 0, n_lflags = 0;
  // ... and by class the solves of small scenes where there are many (eqf_lex_small.hip)
  struct {
    int2 *diff, *press;
    int ndiff, npress;
  } small[LEX_SMALL_CLASSES] = {};
  uint32_t* d_ctl = nullptr;
  uint32_t* h_err = nullptr;
  uint32_t polls = 0;              // LaunchLimits::wait_polls that the graph holds
  std::atomic<bool> stale{false};  // a wait gave up: the counters have to be set up again
  int n = 0, maxN = 0, tiles[3] = {0, 0, 0}, iblocks = 0, cblocks = 0, ablocks = 0;
  bool any_src = false;
  int slots = 1;  // lin_solves that every scene has workspaces for
  int diff_iters = 0, press_iters = 0;  // red-black: the same for every scene
  int diff_rounds = 0, press_rounds = 0;  // exact: the most of any scene
  int tile = 5, tsweeps = 5;  // band shape index (kBands) and sweeps per launch (untuned default)
  int tab_tile = -1, tab_T = -1;
  hipGraphExec_t graph = nullptr;
  uint64_t key = 0;   // what the work maps and the graph were built for
  uint64_t dkey = 0;  // the descriptors that the tables hold
  int64_t key_frames = 0;  // frames launched since
};

constexpr uint32_t kAllFields = (1u << NFIELDS) - 1;

struct FrameWork {
  float* tmp[3] = {nullptr, nullptr, nullptr};  // ping-pong fields: one, or one per diffusion
  RbGroup one;           // the scene alone (eqf_step)
};

// Band shapes (waves per workgroup x rows per wave); the region is always 128
// columns wide.
struct BandCfg {
  int nw, r;
};
static const BandCfg kBands[] = {{8, 16}, {8, 32}, {16, 16}, {8, 18}, {8, 14}, {8, 10}};

// Waves per workgroup of the advection: enough for a row of the largest scene.
static int adv_waves(int maxN) { return maxN > 8 * rb::SEG ? 16 : maxN > 4 * rb::SEG ? 8 : 4; }

static int band_tiles(int S, int tile, int T, int mode) {
  const BandCfg b = kBands[tile];
  const int TX = 128 - 2 * rb::band_halo_x(mode, T), TY = b.nw * b.r - 2 * rb::band_halo_y(mode, T);
  return rb::band_span(S, 128, TX) * rb::band_span(S, b.nw * b.r, TY);
}

struct Hash {
  uint64_t key = 1469598103934665603ull;
  void mix(uint64_t v) { key = (key ^ v) * 1099511628211ull; }
};
// What the work maps and the graph are made for.
static uint64_t group_key(const RbGroup& g) {
  Hash h;
  for (const eqf_scene* s : g.scenes) {
    h.mix(s->uid);
    h.mix((uint64_t)s->desc.diff_iters << 32 | (uint32_t)s->desc.press_iters);
    h.mix(s->desc.has_src != 0);
  }
  h.mix((uint64_t)g.tile * 16 + (uint64_t)g.tsweeps);
  h.mix(g.polls);
  return h.key;
}
// What the tables' copies of the descriptors hold: every byte counts (dt0
// included: with zero viscosity and diffusion a new delta_t changes only dt0).
// A descriptor is value-initialised, so its padding bytes are zero.
static uint64_t desc_key(const RbGroup& g) {
  Hash h;
  for (const eqf_scene* s : g.scenes) {
    uint64_t words[(sizeof(SceneDesc) + 7) / 8] = {};
    std::memcpy(words, &s->desc, sizeof(SceneDesc));
    for (uint64_t w : words) h.mix(w);
  }
  return h.key;
}
static RbScene scene_entry(const eqf_scene* s) {
  const auto* w = static_cast<const FrameWork*>(s->work);
  return RbScene{s->desc, {w->tmp[0], w->tmp[1], w->tmp[2]}};
}

// The strips of `nslots` lin_solves of scene i, `iters` sweeps each.
static void lex_tasks(int i, const eqf_scene* s, int iters, int nslots, std::vector<LexTask>& v, int& nflags) {
  const int S = s->S;
  const int K = lex_round_sweeps(iters, 0);  // the longest round
  if (K == 0) return;
  const int n = lex_strips(S, K);
  for (int slot = 0; slot < nslots; ++slot)
    for (int strip = 0; strip < n; ++strip)
      v.push_back(LexTask{i, slot, strip, n, nflags++, 0, s->d_hand + slot * lex_solve_floats(S) + strip * lex_handoff_floats(S)});
}
// Solves of small scenes: by class, kinds apart, whole waves.
static void small_tasks(const std::vector<int>& scenes, int cls, int nslots, std::vector<int2>& v) {
  const size_t w = (size_t)lex_small_group(cls);
  for (int slot = 0; slot < nslots; ++slot) {
    for (int i : scenes) v.push_back(make_int2(i, slot));
    while (v.size() % w) v.push_back(make_int2(-1, slot));
  }
}
// From how many small scenes on they are solved by waves of their own: a lone solve
// takes a wave longer than a strip's eight (N=62 266 us per frame of 20 sweeps instead
// of 180, N=8 97 instead of 105), the strips fill the CUs much sooner.  us by strips and
// by waves, 20 sweeps (4 sweeps): 128 scenes of N=30 175 and 157 (101 and 93), N=48 256
// and 280 (123 and 148), N=64 344 and 411 (231 and 205); 192 scenes 212 and 162, 356 and
// 293 (155 and 162), 413 and 433; 256 scenes 224 and 169 (137 and 105), 412 and 305
// (175 and 173), 483 and 445 (322 and 239); 512 scenes 370 and 195, 643 and 363, 751
// and 539.
static constexpr int SMALL_MIN = 256;
static size_t lex_ctl_bytes(int nflags) { return (sizeof(uint32_t) * (size_t)(nflags + 2) + 255) & ~(size_t)255; }
int64_t frame_table_bytes(int S, bool exact) {
  const int64_t N = S - 2, nseg = (N + rb::SEG - 1) / rb::SEG;
  int64_t b = sizeof(RbScene) + sizeof(int4) * ((N * nseg + 3) / 4 + (nseg > 1 ? N : (N + 3) / 4)) +
              sizeof(int2) * (((int64_t)S * S + rb::CELL_BLOCK - 1) / rb::CELL_BLOCK);
  if (exact) b += 4 * lex_strips(S, LEX_KMAX) * (int64_t)(sizeof(LexTask) + sizeof(uint32_t));
  else for (int mode = 0; mode < 3; ++mode) b += sizeof(int2) * (int64_t)band_tiles(S, 5, 5, mode);
  return 2 * b;  // with the headroom of group_tables
}

// Ticket order: the longest remaining chain of a scene first (a strip waits
// about 100 steps for the one above it), which puts every strip after the one
// above it and, in a batch, fills the chip with strips that need not wait.
static void lex_order(std::vector<LexTask>& v, const std::vector<eqf_scene*>& scenes) {
  std::stable_sort(v.begin(), v.end(), [&scenes](const LexTask& a, const LexTask& b) {
    const int ka = (a.nstrips - 1 - a.strip) * 100 + scenes[a.scene]->S;
    const int kb = (b.nstrips - 1 - b.strip) * 100 + scenes[b.scene]->S;
    return ka > kb;
  });
}

// (Re)writes the group's tables from its scenes' descriptors, on `st`.
static int group_tables(RbGroup& g, hipStream_t st, std::string& err) {
  const int n = (int)g.scenes.size();
  std::vector<RbScene> scs(n);
  std::vector<int2> tmap[3], cmap;
  std::vector<int4> imap, amap;
  std::vector<LexTask> ldiff, lpress;
  int fd = 0, fp = 0;
  g.any_src = false;
  g.slots = 3;
  g.maxN = 0;
  for (const eqf_scene* s : g.scenes) {
    g.maxN = std::max(g.maxN, s->N);
    if (s->slots < 3) g.slots = 1;
  }
  std::vector<int2> sdiff[LEX_SMALL_CLASSES], spress[LEX_SMALL_CLASSES];
  std::vector<int> sd[LEX_SMALL_CLASSES], spr[LEX_SMALL_CLASSES];
  int nsmall = 0;
  for (const eqf_scene* s : g.scenes) nsmall += lex_small_class(s->S) >= 0;
  const bool small = g.exact && nsmall >= SMALL_MIN;
  g.diff_rounds = g.press_rounds = 0;
  for (int i = 0; i < n; ++i) {
    eqf_scene* s = g.scenes[i];
    scs[i] = scene_entry(s);
    const int cls = small ? lex_small_class(s->S) : -1;
    if (cls >= 0) {
      if (s->desc.diff_iters > 0) sd[cls].push_back(i);
      if (s->desc.press_iters > 0) spr[cls].push_back(i);
    } else {
      g.diff_rounds = std::max(g.diff_rounds, lex_rounds(s->desc.diff_iters));
      g.press_rounds = std::max(g.press_rounds, lex_rounds(s->desc.press_iters));
    }
    if (g.exact && cls < 0) {
      lex_tasks(i, s, s->desc.diff_iters, g.slots, ldiff, fd);
      lex_tasks(i, s, s->desc.press_iters, 1, lpress, fp);
    } else if (!g.exact) {
      for (int mode = 0; mode < 3; ++mode) {
        const int nt = band_tiles(s->S, g.tile, g.tsweeps, mode);
        for (int t = 0; t < nt; ++t) tmap[mode].push_back(make_int2(i, t));
      }
    }
    const int nseg = (s->N + rb::SEG - 1) / rb::SEG;
    for (int64_t k = 0; k < (int64_t)s->N * nseg; k += 4)
      imap.push_back(make_int4(i, 1 + (int)(k / nseg), (int)(k % nseg), nseg));
    const int64_t nb = ((int64_t)s->S * s->S + rb::CELL_BLOCK - 1) / rb::CELL_BLOCK;
    for (int64_t k = 0; k < nb; ++k) cmap.push_back(make_int2(i, (int)k));
    for (int j = 1; j <= s->N; j += nseg > 1 ? 1 : adv_waves(g.maxN)) amap.push_back(make_int4(i, j, 0, nseg));
    g.any_src = g.any_src || s->desc.has_src;
  }
  if (tmap[M_ROW].size() > INT32_MAX / 2 || tmap[M_COL].size() > INT32_MAX / 2 || cmap.size() > INT32_MAX / 2 || imap.size() > INT32_MAX / 2) {  // amap <= imap * 4
    err = "launch group too large for one launch";
    return EQF_EINVAL;
  }
  g.n = n;
  for (int m = 0; m < 3; ++m) g.tiles[m] = (int)tmap[m].size();
  g.iblocks = (int)imap.size();
  g.cblocks = (int)cmap.size();
  g.ablocks = (int)amap.size();
  auto up = [](size_t v) { return (v + 255) & ~(size_t)255; };
  const size_t b_scs = up(sizeof(RbScene) * n);
  size_t b_t[3];
  for (int m = 0; m < 3; ++m) b_t[m] = up(sizeof(int2) * tmap[m].size());
  const size_t b_m = up(sizeof(int4) * imap.size()), b_c = up(sizeof(int2) * cmap.size());
  const size_t b_a = up(sizeof(int4) * amap.size());
  lex_order(ldiff, g.scenes);
  lex_order(lpress, g.scenes);
  const size_t b_ld = up(sizeof(LexTask) * ldiff.size()), b_lp = up(sizeof(LexTask) * lpress.size());
  size_t b_small = 0;
  for (int c = 0; c < LEX_SMALL_CLASSES; ++c) {
    small_tasks(sd[c], c, g.slots, sdiff[c]);
    small_tasks(spr[c], c, 1, spress[c]);
    b_small += up(sizeof(int2) * sdiff[c].size()) + up(sizeof(int2) * spress[c].size());
  }
  g.n_lflags = std::max(fd, fp);
  const size_t b_ctl = lex_ctl_bytes(g.n_lflags);  // zero at first; every launch leaves it so
  const size_t bytes = b_ctl + b_scs + b_t[0] + b_t[1] + b_t[2] + b_m + b_c + b_a + b_ld + b_lp + b_small;
  if (bytes > g.tab_bytes) {  // with headroom: a server's group changes size often
    (void)hipFree(g.d_tab);
    g.d_tab = nullptr;
    g.tab_bytes = 0;
    const size_t cap = std::max(bytes, (size_t)4096) * 2;
    hipError_t e = hipMalloc(&g.d_tab, cap);
    if (e != hipSuccess) {
      err = std::string("frame tables: ") + hipGetErrorString(e);
      return EQF_ENOMEM;
    }
    g.tab_bytes = cap;
  }
  g.h_tab.assign(bytes, 0);
  char* base = g.h_tab.data();
  size_t off = b_ctl;
  auto put = [&](const void* src, size_t len, size_t slot) {
    if (len) std::memcpy(base + off, src, len);
    const size_t at = off;
    off += slot;
    return at;
  };
  const size_t o_scs = put(scs.data(), sizeof(RbScene) * n, b_scs);
  size_t o_t[3];
  for (int m = 0; m < 3; ++m) o_t[m] = put(tmap[m].data(), sizeof(int2) * tmap[m].size(), b_t[m]);
  const size_t o_m = put(imap.data(), sizeof(int4) * imap.size(), b_m);
  const size_t o_c = put(cmap.data(), sizeof(int2) * cmap.size(), b_c);
  const size_t o_a = put(amap.data(), sizeof(int4) * amap.size(), b_a);
  const size_t o_ld = put(ldiff.data(), sizeof(LexTask) * ldiff.size(), b_ld);
  const size_t o_lp = put(lpress.data(), sizeof(LexTask) * lpress.size(), b_lp);
  char* d = (char*)g.d_tab;
  g.d_ctl = (uint32_t*)d;
  g.d_scs = (RbScene*)(d + o_scs);
  for (int m = 0; m < 3; ++m) g.d_tmap[m] = (int2*)(d + o_t[m]);
  g.d_imap = (int4*)(d + o_m);
  g.d_cmap = (int2*)(d + o_c);
  g.d_amap = (int4*)(d + o_a);
  g.d_ldiff = (LexTask*)(d + o_ld);
  g.d_lpress = (LexTask*)(d + o_lp);
  for (int c = 0; c < LEX_SMALL_CLASSES; ++c) {
    auto& sm = g.small[c];
    sm.diff = (int2*)(d + put(sdiff[c].data(), sizeof(int2) * sdiff[c].size(), up(sizeof(int2) * sdiff[c].size())));
    sm.press = (int2*)(d + put(spress[c].data(), sizeof(int2) * spress[c].size(), up(sizeof(int2) * spress[c].size())));
    sm.ndiff = (int)sdiff[c].size();
    sm.npress = (int)spress[c].size();
  }
  g.n_ldiff = (int)ldiff.size();
  g.n_lpress = (int)lpress.size();
  if (g.exact && !g.h_err) {
    hipError_t e = hipHostMalloc((void**)&g.h_err, sizeof(uint32_t), hipHostMallocDefault);
    if (e != hipSuccess) {
      err = std::string("lin_solve status: ") + hipGetErrorString(e);
      return EQF_ENOMEM;
    }
    *g.h_err = 0;
  }
  // behind the frames already queued on `st` (they read the old tables)
  hipError_t e = hipMemcpyAsync(g.d_tab, base, bytes, hipMemcpyHostToDevice, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  if (e != hipSuccess) {
    err = std::string("frame tables: ") + hipGetErrorString(e);
    return EQF_EDEVICE;
  }
  g.tab_tile = g.tile;
  g.tab_T = g.tsweeps;
  return EQF_OK;
}

template <int T, int NW, int R>
static void launch_band(hipStream_t st, const RbGroup& g, const rb::BandArgs& a, int nsw) {
  hipLaunchKernelGGL((rb::k_rb_band<T, NW, R>), dim3((unsigned)(a.s[0].nt + a.s[1].nt + a.s[2].nt)), dim3(64 * NW), 0, st,
                     g.d_scs, a, nsw);
}

template <int NW, int R>
static void launch_band_t(hipStream_t st, const RbGroup& g, const rb::BandArgs& a, int nsw) {
  const int T = g.tsweeps;
  if (T == 1) launch_band<1, NW, R>(st, g, a, nsw);
  else if (T == 2) launch_band<2, NW, R>(st, g, a, nsw);
  else if (T == 4) launch_band<4, NW, R>(st, g, a, nsw);
  else if (T == 5) launch_band<5, NW, R>(st, g, a, nsw);
  else if (T == 6) launch_band<6, NW, R>(st, g, a, nsw);
  else launch_band<8, NW, R>(st, g, a, nsw);
}

static void launch_bands(hipStream_t st, const RbGroup& g, const rb::BandArgs& a, int nsw) {
  if (g.tile == 1) launch_band_t<8, 32>(st, g, a, nsw);
  else if (g.tile == 2) launch_band_t<16, 16>(st, g, a, nsw);
  else if (g.tile == 3) launch_band_t<8, 18>(st, g, a, nsw);
  else if (g.tile == 4) launch_band_t<8, 14>(st, g, a, nsw);
  else if (g.tile == 5) launch_band_t<8, 10>(st, g, a, nsw);
  else launch_band_t<8, 16>(st, g, a, nsw);
}

static void g_copy(hipStream_t st, const RbGroup& g, const rb::CopyArgs& a) {
  hipLaunchKernelGGL(rb::k_copy, dim3((unsigned)g.cblocks), dim3(256), 0, st, g.d_scs, g.d_cmap, a);
}

// A lin_solve: set_boundaries mode, fields and coefficients.
struct Solve {
  int mode, x, x0, coef;
};
// Up to three lin_solves in red-black order on every scene of the group (one
// iteration count): ceil(iters/T) tile passes ping-ponging between x and a
// scratch field; an odd pass count ends with a copy back.
static void g_lin_solve(hipStream_t st, const RbGroup& g, const Solve* sv, int n, int iters) {
  if (iters <= 0) return;
  rb::BandArgs a{};
  for (int k = 0; k < n; ++k)
    a.s[k] = rb::BandSlot{g.d_tmap[sv[k].mode], g.tiles[sv[k].mode], sv[k].mode, sv[k].x, rb::ROLE_TMP + k, sv[k].x0, sv[k].coef};
  int passes = 0;
  for (int done = 0; done < iters; ++passes) {
    const int nsw = std::min(g.tsweeps, iters - done);
    launch_bands(st, g, a, nsw);
    for (int k = 0; k < n; ++k) std::swap(a.s[k].src, a.s[k].dst);
    done += nsw;
  }
  if (passes & 1) {
    rb::CopyArgs c;
    for (int k = 0; k < 3; ++k) {
      c.dst[k] = k < n ? sv[k].x : rb::ROLE_NONE;
      c.src[k] = rb::ROLE_TMP + k;
    }
    g_copy(st, g, c);
  }
}
// Lexicographic lin_solves: the three diffusions of a frame in one launch per
// round (they read and write different fields: u and v from the last frame's
// velocity, density from the last frame's density), or a pressure solve.
static void g_lex(hipStream_t st, const RbGroup& g, bool press, const LexSpec& s0, const LexSpec& s1,
                  const LexSpec& s2) {
  for (int r = 0; r < (press ? g.press_rounds : g.diff_rounds); ++r) {
    const LexArgs a{{s0, s1, s2}, r, press ? 1 : 0, g.polls};
    lex_launch(st, g.d_scs, press ? g.d_lpress : g.d_ldiff, press ? g.n_lpress : g.n_ldiff, a, g.d_ctl, g.n_lflags,
               g.h_err, g.maxN, g.scenes[0]->limits->cus);
  }
  const LexArgs a{{s0, s1, s2}, 0, press ? 1 : 0, 0};
  for (int c = 0; c < LEX_SMALL_CLASSES; ++c)
    lex_small_launch(st, g.d_scs, press ? g.small[c].press : g.small[c].diff, c, press ? g.small[c].npress : g.small[c].ndiff, a);
}
static void g_pressure(hipStream_t st, const RbGroup& g, int p, int div) {
  if (g.exact) g_lex(st, g, true, LexSpec{M_PASSIVE, p, div, 2}, LexSpec{}, LexSpec{});
  else {
    const Solve s{M_PASSIVE, p, div, 2};
    g_lin_solve(st, g, &s, 1, g.press_iters);
  }
}

template <bool DENSITY>
static void g_adv(hipStream_t st, const RbGroup& g, int o0, int i0, int o1, int i1, int u, int v) {
  const dim3 rows((unsigned)g.ablocks);
  const int nw = adv_waves(g.maxN);
  if (nw == 4) hipLaunchKernelGGL((rb::k_adv<DENSITY, 4>), rows, dim3(256), 0, st, g.d_scs, g.d_amap, o0, i0, o1, i1, u, v);
  else if (nw == 8) hipLaunchKernelGGL((rb::k_adv<DENSITY, 8>), rows, dim3(512), 0, st, g.d_scs, g.d_amap, o0, i0, o1, i1, u, v);
  else hipLaunchKernelGGL((rb::k_adv<DENSITY, 16>), rows, dim3(1024), 0, st, g.d_scs, g.d_amap, o0, i0, o1, i1, u, v);
}

// One frame (fluid.rs:437-524) of every scene of the group.  Red-black scenes share
// the iteration counts; exact ones need not: the launches are those of the scene
// with the most rounds of sweeps, the others have no work in the last of them.
//
// Corners (fluid.rs:265-271) are read only by advect's bilinear gathers and
// are part of the frame's final state; no sweep, divergence or gradient reads
// them.  So a field's corners are computed only where a gather or the end of
// the frame reads them before the field's next set_boundaries rewrites them:
// U0 and V0 with the first gradient (advected from), V0 with the second
// divergence, U0 and the density scratch with the second gradient (their solves
// are done), U and V too, the density with its advection.
static void g_frame(hipStream_t st, const RbGroup& g) {
  using rb::ROLE_NONE;
  const dim3 cells((unsigned)g.iblocks);  // interior cell blocks
  if (g.any_src)
    hipLaunchKernelGGL(rb::k_sources, dim3((unsigned)g.cblocks), dim3(256), 0, st, g.d_scs, g.d_cmap);
  // the three diffusions, fluid.rs:438, 448, 501 (the density's reads no velocity)
  // together, or each of them alone where a scene has one slot
  if (g.exact) {
    const LexSpec s[3] = {{M_ROW, F_U0, F_U, 0}, {M_COL, F_V0, F_V, 0}, {M_PASSIVE, F_SC, F_D, 1}};
    if (g.slots == 3) g_lex(st, g, false, s[0], s[1], s[2]);
    else for (int k = 0; k < 3; ++k) g_lex(st, g, false, s[k], LexSpec{}, LexSpec{});
  } else {
    const Solve s[3] = {{M_ROW, F_U0, F_U, 0}, {M_COL, F_V0, F_V, 0}, {M_PASSIVE, F_SC, F_D, 1}};
    for (int k = 0; k < 3; k += g.slots) g_lin_solve(st, g, s + k, g.slots, g.diff_iters);
  }
  // project(U0, V0, p=U, div=V), fluid.rs:459
  hipLaunchKernelGGL(rb::k_div, cells, dim3(256), 0, st, g.d_scs, g.d_imap, F_U0, F_V0, F_V, F_U, 0);
  g_pressure(st, g, F_U, F_V);
  hipLaunchKernelGGL(rb::k_grad, cells, dim3(256), 0, st, g.d_scs, g.d_imap, F_U0, F_V0, F_U, 0, ROLE_NONE);
  // advect U from U0 and V from V0 with (U0, V0), fluid.rs:469-489
  g_adv<false>(st, g, F_U, F_U0, F_V, F_V0, F_U0, F_V0);
  // project(U, V, p=U0, div=V0), fluid.rs:491
  hipLaunchKernelGGL(rb::k_div, cells, dim3(256), 0, st, g.d_scs, g.d_imap, F_U, F_V, F_V0, F_U0, 1);
  g_pressure(st, g, F_U0, F_V0);
  hipLaunchKernelGGL(rb::k_grad, cells, dim3(256), 0, st, g.d_scs, g.d_imap, F_U, F_V, F_U0, 1, F_SC);
  // fluid.rs:511-523
  g_adv<true>(st, g, F_D, F_SC, ROLE_NONE, ROLE_NONE, F_U, F_V);
  g_copy(st, g, rb::CopyArgs{{F_SC, ROLE_NONE, ROLE_NONE}, {F_D, 0, 0}});
}

static void group_release(RbGroup& g) {
  if (g.graph) (void)hipGraphExecDestroy(g.graph);
  g.graph = nullptr;
  if (g.d_tab) (void)hipFree(g.d_tab);
  g.d_tab = nullptr;
  g.tab_bytes = 0;
  if (g.h_err) (void)hipHostFree(g.h_err);
  g.h_err = nullptr;
}

// One frame as a graph on `st`.
static int group_capture(RbGroup& g, hipStream_t st, std::string& err) {
  hipGraph_t gr = nullptr;
  hipError_t e = hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal);
  if (e != hipSuccess) {
    err = std::string("capture: ") + hipGetErrorString(e);
    return EQF_EDEVICE;
  }
  g_frame(st, g);
  hipError_t le = hipGetLastError();
  e = hipStreamEndCapture(st, &gr);
  if (le != hipSuccess || e != hipSuccess) {
    err = std::string("frame capture: ") + hipGetErrorString(le != hipSuccess ? le : e);
    if (gr) (void)hipGraphDestroy(gr);
    return EQF_EDEVICE;
  }
  e = hipGraphInstantiate(&g.graph, gr, nullptr, nullptr, 0);
  (void)hipGraphDestroy(gr);
  if (e != hipSuccess) {
    err = std::string("graph instantiate: ") + hipGetErrorString(e);
    return EQF_EDEVICE;
  }
  return EQF_OK;
}

// Kernels of a frame, and up to how many of them it is worth a graph: the sweep
// counts have no bound that would keep a graph's size reasonable (2^24 sweeps are
// 2.5 million launches), and a frame this long hides its launches.
static constexpr int64_t GRAPH_MAX = 4096;
static int64_t frame_launches(const RbGroup& g) {
  auto solve = [&g](int iters) { return (int64_t)(iters + g.tsweeps - 1) / g.tsweeps + 1; };
  const int64_t d = g.exact ? g.diff_rounds : solve(g.diff_iters), p = g.exact ? g.press_rounds : solve(g.press_iters);
  return 8 + d * (3 / g.slots) + 2 * p;
}

// Advances every scene of the group by nframes on `st`.  The tables are
// rebuilt when the scenes, their iteration counts or the tiling change.  The first
// frame after that is launched kernel by kernel; further ones replay a graph
// captured once (a server's groups change membership often, and one frame's
// launches cost less than a capture).
static int group_step_all(RbGroup& g, hipStream_t st, int64_t nframes, std::string& err) {
  if (nframes <= 0 || g.scenes.empty()) return EQF_OK;
  g.diff_iters = g.scenes[0]->desc.diff_iters;
  g.press_iters = g.scenes[0]->desc.press_iters;
  g.exact = g.scenes[0]->p.gs_mode == EQF_GS_WAVEFRONT;
  if (!g.exact)
    for (const eqf_scene* s : g.scenes)
      if (s->desc.diff_iters != g.diff_iters || s->desc.press_iters != g.press_iters) {
        err = "red-black scenes of one batch need the same iteration counts";
        return EQF_EINVAL;
      }
  for (eqf_scene* s : g.scenes)
    if (s->invalid.load()) s->invalid.store(kAllFields);  // a frame mixes the fields
  g.polls = g.scenes[0]->limits->wait_polls.load();
  const uint64_t key = group_key(g), dkey = desc_key(g);
  const bool descs = dkey != g.dkey;
  if (g.stale.exchange(false) || !g.d_tab || key != g.key || g.tab_tile != g.tile || g.tab_T != g.tsweeps ||
      (descs && g.n > 1)) {
    int rc = group_tables(g, st, err);
    if (rc) {
      g.tab_tile = -1;  // not usable
      return rc;
    }
    if (g.graph) (void)hipGraphExecDestroy(g.graph);
    g.graph = nullptr;
    g.key = key;
    g.dkey = dkey;
    g.key_frames = 0;
  } else if (descs) {
    // A lone scene's parameters (the scenes of a group keep theirs): behind the
    // queued frames, without a wait, and the graph stays.  Tables made anew wait for
    // the frames before them.
    hipLaunchKernelGGL(rb::k_put_scene, dim3(1), dim3(1), 0, st, g.d_scs, scene_entry(g.scenes[0]));
    g.dkey = dkey;
  }
  const bool graph = frame_launches(g) <= GRAPH_MAX;
  for (int64_t f = 0; f < nframes; ++f) {
    if (g.key_frames++ == 0 || !graph) {
      g_frame(st, g);
      hipError_t e = hipGetLastError();
      if (e != hipSuccess) {
        err = std::string("frame launch: ") + hipGetErrorString(e);
        return EQF_EDEVICE;
      }
      continue;
    }
    if (!g.graph) {
      int rc = group_capture(g, st, err);
      if (rc) return rc;
    }
    hipError_t e = hipGraphLaunch(g.graph, st);
    if (e != hipSuccess) {
      err = std::string("graph launch: ") + hipGetErrorString(e);
      return EQF_EDEVICE;
    }
  }
  return EQF_OK;
}

static int group_step(RbGroup& g, hipStream_t st, int64_t nframes, std::string& err) {
  try {
    return group_step_all(g, st, nframes, err);
  } catch (...) {  // std::bad_alloc of the tables' host image
    g.tab_tile = -1;
    err = "out of memory";
    return EQF_ENOMEM;
  }
}

void* frame_create(eqf_scene* s, std::string& err) {
  auto* w = new FrameWork;
  const size_t n = (size_t)s->S * s->S;
  hipError_t e = hipSuccess;
  if (s->p.gs_mode == EQF_GS_REDBLACK) {
    const size_t fs = (size_t)rm_field_floats(s->S);
    auto alloc = [&] { return eqf_scene_malloc(s, (void**)&w->tmp[0], sizeof(float) * (s->slots > 1 ? s->slots * fs : n)); };
    e = alloc();
    if (e == hipErrorOutOfMemory && s->slots > 1) {  // the diffusions one after the other then
      (void)hipGetLastError();
      w->tmp[0] = nullptr;
      s->slots = 1;
      e = alloc();
    }
    for (int i = 1; i < s->slots && e == hipSuccess; ++i) w->tmp[i] = w->tmp[0] + i * fs;
  }
  if (e != hipSuccess) {
    err = std::string("frame workspace: ") + hipGetErrorString(e);
    eqf_scene_mfree(s, w->tmp[0]);
    delete w;
    return nullptr;
  }
  w->one.scenes = {s};
  w->one.tile = 5;  // the autotuner (equilibrium_amd/tune.py) may override these
  w->one.tsweeps = 5;
  return w;
}

void frame_destroy(eqf_scene* s) {
  auto* w = static_cast<FrameWork*>(s->work);
  if (!w) return;
  group_release(w->one);
  eqf_scene_mfree(s, w->tmp[0]);
  delete w;
  s->work = nullptr;
}

static bool tiling_ok(int tile, int tsweeps) {
  return tile >= 0 && tile <= 5 && tsweeps >= 1 && tsweeps <= 8 && tsweeps != 3 && tsweeps != 7;
}

int frame_set_tiling(eqf_scene* s, int tile, int tsweeps) {
  auto* w = static_cast<FrameWork*>(s->work);
  if (!w || !tiling_ok(tile, tsweeps)) return EQF_EINVAL;
  w->one.tile = tile;
  w->one.tsweeps = tsweeps;
  return EQF_OK;
}

int frame_step(eqf_scene* s, int64_t nframes, std::string& err) {
  auto* w = static_cast<FrameWork*>(s->work);
  return group_step(w->one, s->stream, nframes, err);
}

bool frame_collect(const eqf_scene* s) {
  auto* w = static_cast<FrameWork*>(s->work);
  return w && group_collect(&w->one);
}

// Batches (eqf_runtime.hip) and server lanes: one group over all scenes.
void* group_create(const std::vector<eqf_scene*>& scenes, hipStream_t st, std::string& err) {
  if (scenes[0]->p.gs_mode == EQF_GS_REDBLACK)
    for (const eqf_scene* s : scenes)
      if (s->desc.diff_iters != scenes[0]->desc.diff_iters || s->desc.press_iters != scenes[0]->desc.press_iters) {
        err = "red-black scenes of one batch need the same iteration counts";
        return nullptr;
      }
  auto* g = new RbGroup;
  g->scenes = scenes;
  g->stream = st;
  return g;
}
void group_destroy(void* p) {
  auto* g = static_cast<RbGroup*>(p);
  if (!g) return;
  group_release(*g);
  delete g;
}
int group_set_tiling(void* p, int tile, int tsweeps) {
  auto* g = static_cast<RbGroup*>(p);
  if (!g || !tiling_ok(tile, tsweeps)) return EQF_EINVAL;
  g->tile = tile;
  g->tsweeps = tsweeps;
  return EQF_OK;
}
int group_step_frames(void* p, int64_t nframes, std::string& err) {
  auto* g = static_cast<RbGroup*>(p);
  return group_step(*g, g->stream, nframes, err);
}
void group_set_scenes(void* p, const std::vector<eqf_scene*>& scenes) {
  auto* g = static_cast<RbGroup*>(p);
  g->scenes = scenes;  // a new membership changes the key: tables and graph are rebuilt
}
bool group_collect(void* p) {
  auto* g = static_cast<RbGroup*>(p);
  if (!g || !g->h_err || __atomic_load_n(g->h_err, __ATOMIC_ACQUIRE) == 0) return false;
  // cleared last: a thread that has another of the scenes and finds the status clear
  // finds its scene marked (two threads that see it set both mark, which does no harm)
  for (eqf_scene* s : g->scenes) {
    s->invalid.store(kAllFields);
    s->failures.fetch_add(1);
  }
  g->stale.store(true);
  __atomic_store_n(g->h_err, 0u, __ATOMIC_RELEASE);
  return true;
}

}  // namespace eqf
