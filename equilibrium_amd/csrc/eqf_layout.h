// eqf_layout.h -- scene layout shared by the host runtime and the kernels.
//
// A scene of `size` S = N + 2 (N interior rows/columns plus the 1-cell wall
// ring of the reference, fluid.rs:552-570) keeps its six fields resident in
// HBM, row-major `x + y*S` like the reference (fluid.rs:31-35), ring included.
//
// Field order follows the Fluid struct (fluid.rs:59-77).
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#define EQF_HD __host__ __device__
#else
#define EQF_HD
#endif

namespace eqf {

enum Field { F_D = 0, F_SC = 1, F_U = 2, F_V = 3, F_U0 = 4, F_V0 = 5, NFIELDS = 6 };
enum Mode { M_ROW = 0, M_COL = 1, M_PASSIVE = 2 };  // Orientation, fluid.rs:22-29

// Per-cell rule byte (one byte per cell, ring included, cell (x, y) at
// y * rm_code_stride(S) + x), read by the lin_solve kernels:
//   bit 0     interior cell (updated by the sweeps)
//   bits 1-2  AdjustRow: 0 keep, 1 -(left), 2 -(right)  (right wins, fluid.rs:151-164)
//   bits 3-4  AdjustColumn: 0 keep, 1 -(up), 2 -(down)  (up wins, fluid.rs:165-177)
//             (either: 3 an interior wall cell, kept, that a fluid cell takes its value from)
//   bits 5-7  Passive, ring cells whose row / column holds a NoWall cell
//             (fluid.rs:179-187): 0 none, 1 copy the left, 2 the right, 3 the
//             upper, 4 the lower neighbour
// The lexicographic kernel runs AdjustColumn with rows and columns exchanged
// and reads a second, transposed array (cell (x, y) at x * rm_code_stride(S) +
// y), rm_code_bytes(S) after the first.
enum RuleBits : uint32_t {
  R_INTERIOR = 1u,
  R_ROW_SHIFT = 1, R_COL_SHIFT = 3, R_PAS_SHIFT = 5,
  R_NEG_FIRST = 1u, R_NEG_SECOND = 2u,  // left / up, right / down
  R_SOURCE = 3u,
  R_COPY_LEFT = 1u, R_COPY_RIGHT = 2u, R_COPY_UP = 3u, R_COPY_DOWN = 4u,
};

struct SceneDesc {
  float* fld;            // NFIELDS fields, `fstride` floats apart
  const float* src;      // per-frame sources (density, vx, vy) or nullptr
  const uint8_t* code;   // RuleBits at x + y*rm_code_stride(S), then the transposed array
  int64_t fstride;       // floats per field
  int S, N;              // size, interior size
  int ring_copies;       // Passive ring cells that copy their neighbour (4 N: all but the corners)
  int diff_iters, press_iters;
  float a_visc, cr_visc; // diffuse coefficients for velocity (fluid.rs:286-294, 311)
  float a_diff, cr_diff; // diffuse coefficients for density
  float dt0;             // dt * (S-2)         (fluid.rs:390)
  float sf;              // (float)S           (fluid.rs:345, 396)
  float sfm1;            // (float)S - 1.0f    (fluid.rs:403)
  int has_src;           // frame sources to add: bit 0 density (and scratch), 1 vx, 2 vy
};

EQF_HD inline int64_t rm_field_floats(int S) {
  int64_t n = (int64_t)S * S;
  return (n + 63) & ~(int64_t)63;
}
// Floats allocated before field 0, and bytes before the rule bytes (the end of
// the last field) that a 4-element access beginning left of a row may touch.
constexpr int FLD_PAD = 64;
constexpr int CODE_PAD = 16;

// Rule bytes: rows padded to an even length, so that a lane's column pair
// (even first column) is one 2-byte-aligned load for any S; the array padded
// so that the transposed one is aligned too.
EQF_HD inline int rm_code_stride(int S) { return S + (S & 1); }
EQF_HD inline int64_t rm_code_used(int S) { return (int64_t)S * rm_code_stride(S); }
EQF_HD inline int64_t rm_code_bytes(int S) { return (rm_code_used(S) + 63) & ~(int64_t)63; }
EQF_HD inline int rm_code_arrays(bool exact) { return exact ? 2 : 1; }

// Lin_solves that a scene has workspaces for at once (red-black: ping-pong fields;
// exact: hand-off values): the three diffusions, which then share their launches, or
// one (a server's scene whose budget does not hold more).  Red-black scenes have one
// from the size where one diffusion fills the device and the caches hold
// more of one than of three.  ms per frame of 20 sweeps apart and together: N=250
// 0.274 and 0.183, N=1501 0.436 and 0.346, N=2046 0.574 and 0.469, N=3000 0.948
// and 0.909, N=4096 1.510 and 1.543.
EQF_HD inline int scene_slots(bool exact, int S) { return exact || S <= 3072 ? 3 : 1; }

// ---- lexicographic lin_solve (eqf_lex.hip) ----
// Sweeps per round, steps per block.
constexpr int LEX_KMAX = 20, LEX_B = 8;
// Rounds of a lin_solve of `iters` sweeps, and the sweeps of each: as even as possible.
EQF_HD inline int lex_rounds(int iters) { return iters > 0 ? (iters + LEX_KMAX - 1) / LEX_KMAX : 0; }
EQF_HD inline int lex_round_sweeps(int iters, int round) {
  const int n = lex_rounds(iters);
  return round < n ? iters / n + (round < iters % n ? 1 : 0) : 0;
}
// Rows of a strip: 64 lanes, the first of which repeats the last row of the strip above.
constexpr int LEX_ROWS = 63;
// Strips that K sweeps of S rows take, each sweep one row further up.
EQF_HD inline int lex_strips(int S, int K) { return (S + K - 1 + LEX_ROWS - 1) / LEX_ROWS; }
// Blocks of LEX_B steps of a strip: column S-1 of lane 63 in the last sweep, and its final value a step later.
EQF_HD inline int lex_blocks(int S, int K) { return ((S + 63 + 2 * (K - 1)) >> 3) + 1; }
// Hand-off values a strip leaves for the next one: one per sweep and step.
EQF_HD inline int64_t lex_handoff_floats(int S) { return (int64_t)LEX_KMAX * lex_blocks(S, LEX_KMAX) * LEX_B; }
// ... of a lin_solve of any number of sweeps.
EQF_HD inline int64_t lex_solve_floats(int S) { return (lex_strips(S, LEX_KMAX) - 1) * lex_handoff_floats(S); }

}  // namespace eqf
