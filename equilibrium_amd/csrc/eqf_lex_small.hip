// eqf_lex_small.hip -- lexicographic Gauss-Seidel (lin_solve, fluid.rs:301-325) of
// many small scenes, bit for bit: a wave takes whole solves of grids of up to 66 x
// 66 cells (ring included) through all their sweeps in registers.
//
// Work split.  A lane owns a row; grids of up to 16 or 32 rows share a wave by
// four or two.  At step t lane r works on column c = (t - r) mod P, sweep
// floor((t - r) / P), so sweeps follow each other without a gap: of the strips of
// eqf_lex.hip 40% of a lane's steps lie outside an N=64 grid and a third of its
// lanes, and a strip takes half a CU.  The cell of step t is in register t mod P of
// its lane; then everything an update reads is in a register of a fixed number:
//   left   x_k(c-1, j)      the lane's value of the step before
//   up     x_k(c, j-1)      the lane before it, the step before
//   right  x_{k-1}(c+1, j)  register (t + 1) mod P
//   down   x_{k-1}(c, j+1)  the same register of the next lane
// x, x0 and the rules of P cells are 2 P + P / 8 registers: no memory is touched
// between the first load and the last store.  Ring cells are cells like the others
// whose update is their value; in Passive they take the interior neighbour's value
// when it is known (a step before or after).  AdjustRow's final values are formed
// a step later too, and AdjustColumn runs with rows and columns exchanged
// (eqf_lex.hip).  A grid of 65 or 66 rows has its first (and last) ring row in the lanes
// of registers of their own, which turn by a lane per step.
//
// Bound: instruction issue, about 15 (Passive 22) vector instructions a step, which
// two (P = 66) to eight (P = 16) waves per SIMD share; a lone wave waits for its chain
// of eight dependent ones.  us per frame of 20 sweeps by strips and by waves (the other
// phases of a frame included): 2048 scenes of N=8 782 and 149, of N=30 1261 and 413,
// of N=48 2291 and 880, of N=64 2748 and 1099.
//
// The registers hold because no phase of a solve keeps addresses or lane masks for
// the next (anew), x0 comes in parts while x has its registers, and what is not a cell
// of a sweep (the skew at the start and the end) is one by its code (3), so that there
// is one body of P steps.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "eqf_internal.h"

namespace eqf {
namespace small {

__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ int as_i(float v) { return __builtin_bit_cast(int, v); }
__device__ __forceinline__ float as_f(int v) { return __builtin_bit_cast(float, v); }
// v, computed anew: keeps the phases of a solve from sharing addresses and lane
// masks, which would stay in registers through the sweeps.
__device__ __forceinline__ int anew(int v) {
  asm volatile("" : "+v"(v));
  return v;
}
// Lane shifts (DPP wave_shr:1 / wave_shl:1): the lane without a source gets `edge`
// where EDGE, else 0.
template <bool EDGE>
__device__ __forceinline__ float from_prev_lane(float v, float edge) {
  return as_f(__builtin_amdgcn_update_dpp(EDGE ? as_i(edge) : 0, as_i(v), 0x138, 0xf, 0xf, !EDGE));
}
template <bool EDGE>
__device__ __forceinline__ float from_next_lane(float v, float edge) {
  return as_f(__builtin_amdgcn_update_dpp(EDGE ? as_i(edge) : 0, as_i(v), 0x130, 0xf, 0xf, !EDGE));
}

// Code of a cell.  ROW / COL (logical): 0 plain, 1 -(left), 2 -(right), 3 keeps its
// value.  PASSIVE: 0 plain, 1 the left, 2 the upper neighbour's value, 3 keeps its
// value, 4 and 5 keep it and then take the right / lower neighbour's; bit 3: the ring
// cell beyond (row 0 or 65, which have no lane) takes the cell's.
template <int MODE>
__device__ __forceinline__ uint32_t code_of(uint32_t rule) {
  if constexpr (MODE == M_PASSIVE) {
    const uint32_t r = rule >> R_PAS_SHIFT;
    return (rule & R_INTERIOR) ? 0u : r == R_COPY_LEFT ? 1u : r == R_COPY_UP ? 2u : r == R_COPY_RIGHT ? 4u : r == R_COPY_DOWN ? 5u : 3u;
  } else {
    const uint32_t r = (rule >> (MODE == M_COL ? R_COL_SHIFT : R_ROW_SHIFT)) & 3u;
    return !(rule & R_INTERIOR) ? 3u : r == R_SOURCE ? 0u : r;
  }
}

// Columns of P registers, groups of LG lanes; EDGE: rows 1 .. 64 have lanes, else rows
// 0 .. LG-1.
template <int MODE, int P, int LG, bool EDGE>
struct Solve {
  static constexpr int NG = 64 / LG, BITS = MODE == M_PASSIVE ? 4 : 2, PER = 32 / BITS, NC = (P + PER - 1) / PER;
  static_assert(P >= LG || P == 48, "a row has a lane");
  static_assert(P % 2 == 0, "P - 1 is odd: the skewed accesses to LDS lie in distinct banks");
  float X[P], X0[P];
  uint32_t cd[NC];
  float r1, r2;   // the lane's values of the last step and the one before it
  uint32_t selp;  // code of the last step's cell
  // EDGE: the first (last) ring row's cells.  T[0], B[0] turn by a lane per step: lane
  // 0 / 63 has the cell of step s < 64; [s - 63] those of the steps 64 and 65.
  float T[3], B[3];

  // P steps: lane r runs sweep k from step r on, sweep k - 1 before.  Cells of sweeps
  // that are none of its K keep their values: code 3.
  __device__ __forceinline__ void sweep(int k, int kmin, int r, int K, float a, float cr) {
    uint32_t c[NC];
    const bool some = k == 0 || k >= kmin;  // (uniform)
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      c[i] = cd[i];
      if (some) {
        const int n = min(max(r - i * PER, 0), PER);  // steps of the register before r
        const uint32_t before = n == PER ? ~0u : (1u << (BITS * n)) - 1u;
        const uint32_t keep = ((uint32_t)k < (uint32_t)K ? 0u : ~before) | ((uint32_t)(k - 1) < (uint32_t)K ? 0u : before);
        c[i] = (c[i] & ~keep) | (keep & (MODE == M_PASSIVE ? 0x33333333u : ~0u));
      }
      // keeps the compiler from hoisting every lane mask out of the loop over sweeps
      // (into scalar registers)
      asm volatile("" : "+v"(c[i]));
    }
    const int lane = anew(threadIdx.x);
#pragma unroll
    for (int s = 0; s < P; ++s) {
      const int s1 = (s + 1) % P, sm = (s + P - 1) % P;
      const float rt = X[s1], lt = r1;
      const int es = EDGE && s >= 64 ? s - 63 : 0;
      const float dn = from_next_lane<EDGE>(X[s1], B[es]), up = from_prev_lane<EDGE>(r1, T[es]);
      // fluid.rs:315-320; AdjustColumn: logical right / left are down / up
      float nv = MODE == M_COL ? ((up + dn) + rt) + lt : ((rt + lt) + dn) + up;
      nv = (X0[s] + a * nv) * cr;
      asm volatile("" : "+v"(nv));  // selects, not a branch around the update
      const uint32_t sel = (c[s / PER] >> (BITS * (s % PER))) & (MODE == M_PASSIVE ? 7u : 3u);
      if constexpr (MODE == M_PASSIVE) {
        nv = sel == 1u ? lt : nv;
        nv = sel == 2u ? up : nv;
      }
      nv = sel >= 3u ? X[s] : nv;
      // the last step's cell
      float f = r1;
      if constexpr (MODE == M_PASSIVE) {
        const float below = from_next_lane<false>(nv, 0.0f);
        f = selp == 4u ? nv : f;
        f = selp == 5u ? below : f;
      } else {
        f = selp == 1u ? -r2 : f;
        f = selp == 2u ? -nv : f;
      }
      asm volatile("" : "+v"(f));  // here, not where it is read: nv need not be kept
      X[sm] = f;
      r2 = r1;
      r1 = nv;
      selp = sel;
      if constexpr (EDGE) {
        if constexpr (MODE == M_PASSIVE) {
          const bool on = (c[s / PER] >> (BITS * (s % PER))) & 8u;
          T[es] = on && lane == 0 ? nv : T[es];
          B[es] = on && lane == 63 ? nv : B[es];
        }
        if (s < 64) {
          T[0] = as_f(__builtin_amdgcn_update_dpp(0, as_i(T[0]), 0x134, 0xf, 0xf, true));  // wave_rol:1
          B[0] = as_f(__builtin_amdgcn_update_dpp(0, as_i(B[0]), 0x13c, 0xf, 0xf, true));  // wave_ror:1
        }
      }
      if (s % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_sched_barrier(0);
    X[P - 1] = r1;  // (its final value comes with the next step)
  }
};

typedef __amdgpu_buffer_rsrc_t rsrc_t;
// A scene's array of `bytes` bytes (uniform): reads beyond it give 0, writes nothing.
__device__ __forceinline__ rsrc_t view(const void* base, int bytes) {
  const uint64_t p = (uint64_t)(uintptr_t)base;
  const uint64_t pu = (uint64_t)(uint32_t)uni((int)(uint32_t)p) | ((uint64_t)(uint32_t)uni((int)(p >> 32)) << 32);
  return __builtin_amdgcn_make_buffer_rsrc((void*)(uintptr_t)pu, (short)0, bytes, 0x00020000);
}

// The fields of the NG scenes of a wave between memory and LDS (P x P cells per
// scene): access i of scene g takes NG rows from NG i on, a lane LG columns of one
// of them; cells beyond the grid's columns hold whatever follows (nobody reads
// them).  EDGE: columns 64 and 65 too, 32 rows at a time.
template <int P, int LG, bool EDGE>
struct Fields {
  static constexpr int NG = 64 / LG, N = P / NG;  // P accesses, 16 to a part
  static constexpr int PARTS = (P + 15) / 16;
  float e[3];
  // part c
  static __device__ __forceinline__ void load(float (&v)[16], int c, const rsrc_t (&x)[NG], const int (&S)[NG], int lane) {
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const int g = (16 * c + k) / N, i = (16 * c + k) % N;
      if (g < NG) v[k] = as_f(__builtin_amdgcn_raw_buffer_load_b32(x[g], ((NG * i + lane / LG) * S[g] + lane % LG) * 4, 0, 0));
    }
  }
  static __device__ __forceinline__ void put(const float (&v)[16], int c, float* __restrict__ lds, int lane) {
    if (lane % LG < P)
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        const int g = (16 * c + k) / N, i = (16 * c + k) % N;
        if (g < NG) lds[g * P * P + (NG * i + lane / LG) * P + lane % LG] = v[k];
      }
  }
  __device__ __forceinline__ void load_edge(const rsrc_t (&x)[NG], const int (&S)[NG], int lane) {
    if constexpr (EDGE) {
#pragma unroll
      for (int i = 0; i < 3; ++i)
        e[i] = as_f(__builtin_amdgcn_raw_buffer_load_b32(x[0], ((32 * i + (lane >> 1)) * S[0] + 64 + (lane & 1)) * 4, 0, 0));
    }
  }
  __device__ __forceinline__ void put_edge(float* __restrict__ lds, int lane) const {
    if constexpr (EDGE) {
#pragma unroll
      for (int i = 0; i < 3; ++i)
        if (32 * i + (lane >> 1) < P) lds[(32 * i + (lane >> 1)) * P + 64 + (lane & 1)] = e[i];
    }
  }
};

template <int MODE, int P, int LG, bool EDGE>
__device__ __forceinline__ void solve(float* __restrict__ lds, const RbScene* __restrict__ scs, int scene, const LexSpec& sp,
                                      bool press) {
  typedef Solve<MODE, P, LG, EDGE> V;
  constexpr int NG = V::NG;
  const int lane = threadIdx.x & 63, g = lane / LG, r = lane % LG;
  // of the wave's scenes; of the lane's
  const SceneDesc* ds[NG];
  int Ss[NG], Ks[NG], S = 0, K = 0, kmax = 0, kmin = 1 << 30;
  rsrc_t xs[NG], x0s[NG];
  float a = 0.0f, cr = 0.0f;
#pragma unroll
  for (int i = 0; i < NG; ++i) {
    const int sc = __builtin_amdgcn_readlane(scene, i * LG);
    const SceneDesc& d = scs[sc < 0 ? 0 : sc].d;
    ds[i] = &d;
    Ss[i] = sc < 0 ? 0 : d.S;
    Ks[i] = sc < 0 ? 0 : press ? d.press_iters : d.diff_iters;
    xs[i] = view(d.fld + (int64_t)sp.x_role * d.fstride, Ss[i] * Ss[i] * 4);
    x0s[i] = view(d.fld + (int64_t)sp.x0_role * d.fstride, Ss[i] * Ss[i] * 4);
    kmax = max(kmax, Ks[i]);
    kmin = Ks[i] > 0 ? min(kmin, Ks[i]) : kmin;
    if (g == i) {
      S = Ss[i];
      K = Ks[i];
      a = sp.coef == 0 ? d.a_visc : sp.coef == 1 ? d.a_diff : 1.0f;
      cr = sp.coef == 0 ? d.cr_visc : sp.coef == 1 ? d.cr_diff : 0.25f;
    }
  }
  float* L = lds + g * P * P;
  // the lane's logical row, its column at step s, where a cell is in L
  const int rr = min(r, P - 1);
  auto row_of = [](int q) { return min(EDGE ? q + 1 : q, P - 1); };
  auto col = [](int q, int s) { return s >= q ? s - q : s - q + P; };
  auto at = [](int c, int row) { return MODE == M_COL ? c * P + row : row * P + c; };
  // (as one of two lane constants and a multiple of the step)
  auto cell = [&](int q, int s) {
    constexpr int C = MODE == M_COL ? P : 1;
    const int b = at(0, row_of(q)) - q * C;
    return (s >= q ? b : b + P * C) + s * C;
  };
  V v;
  {
    typedef Fields<P, LG, EDGE> F;
    F f;
    {
      float w[F::PARTS][16];  // on its way while the rules are read
#pragma unroll
      for (int c = 0; c < F::PARTS; ++c) F::load(w[c], c, xs, Ss, lane);
      f.load_edge(xs, Ss, lane);
      {  // the rules: the arrays of bytes through LDS
#pragma unroll
        for (int i = 0; i < NG; ++i) {
          const uint32_t* code = (const uint32_t*)(ds[i]->code + (MODE == M_COL ? rm_code_bytes(Ss[i]) : 0));
          const int n = (int)((rm_code_used(Ss[i]) + 3) / 4);
          for (int k = lane; k < n; k += 64) ((uint32_t*)lds)[i * P * P + k] = code[k];
        }
        __syncthreads();
        const uint8_t* cb = (const uint8_t*)L;
        const int q2 = anew(rr), j = row_of(q2), Sc = rm_code_stride(S);
#pragma unroll
        for (int i = 0; i < V::NC; ++i) v.cd[i] = 0;
#pragma unroll
        for (int s = 0; s < P; ++s) {
          const int c = col(q2, s);
          const bool in = c < S && j < S && r < P;
          uint32_t k = in ? code_of<MODE>(cb[in ? j * Sc + c : 0]) : 3u;
          if constexpr (EDGE && MODE == M_PASSIVE) {
            if (in && r == 0 && (cb[c] >> R_PAS_SHIFT)) k |= 8u;
            if (in && j == S - 2 && r == 63 && (cb[(S - 1) * Sc + c] >> R_PAS_SHIFT)) k |= 8u;
          }
          v.cd[s / V::PER] |= k << (V::BITS * (s % V::PER));
          if (s % 8 == 7) __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
      }
#pragma unroll
      for (int c = 0; c < F::PARTS; ++c) F::put(w[c], c, lds, lane);
      f.put_edge(lds, lane);
    }
    asm volatile("" ::: "memory");
    // x0: two parts in flight (x has its registers by then)
    float w[2][16];
    const int l0 = anew(lane);
    F::load(w[0], 0, x0s, Ss, l0);
    if (F::PARTS > 1) F::load(w[1], 1, x0s, Ss, l0);
    f.load_edge(x0s, Ss, l0);
    __syncthreads();
    const int q1 = anew(rr);
#pragma unroll
    for (int s = 0; s < P; ++s) {
      v.X[s] = L[cell(q1, s)];
      if (s % 8 == 7) __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (EDGE) {
      v.T[0] = L[at(lane, 0)];
      v.B[0] = L[at((63 - lane + 3) % P, P - 1)];  // lane 63's column at step s: s + 3
#pragma unroll
      for (int i = 1; i < 3; ++i) {
        v.T[i] = L[at(63 + i, 0)];
        v.B[i] = L[at((63 + i + 3) % P, P - 1)];
      }
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < F::PARTS; ++c) {
      F::put(w[c & 1], c, lds, lane);
      if (c + 2 < F::PARTS) F::load(w[c & 1], c + 2, x0s, Ss, l0);
      __builtin_amdgcn_sched_barrier(0);
    }
    f.put_edge(lds, lane);
    __syncthreads();
    const int q0 = anew(rr);
#pragma unroll
    for (int s = 0; s < P; ++s) {
      v.X0[s] = L[cell(q0, s)];
      if (s % 8 == 7) __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
  }
  v.r2 = 0.0f;
  v.selp = 3;
  v.r1 = v.X[P - 1];
  for (int k = 0; k <= kmax; ++k) v.sweep(k, kmin, rr, K, a, cr);
  const int q3 = anew(rr);
  if (r < P)
#pragma unroll
    for (int s = 0; s < P; ++s) L[cell(q3, s)] = v.X[s];
  if constexpr (EDGE && MODE == M_PASSIVE) {
    __syncthreads();
    // (of lanes 0 and 63 where it is one value; a grid of 65 rows has the last in a lane)
    L[at(lane, 0)] = v.T[0];
    if (S == P) L[at((63 - lane + 3) % P, P - 1)] = v.B[0];
#pragma unroll
    for (int i = 1; i < 3; ++i) {
      if (lane == 0) L[at(63 + i, 0)] = v.T[i];
      if (lane == 63 && S == P) L[at((63 + i + 3) % P, P - 1)] = v.B[i];
    }
  }
  __syncthreads();
  const int le = anew(lane);
  // everything but the corners (and the ring rows without a lane, where they hold still)
#pragma unroll
  for (int i = 0; i < NG; ++i) {
    if (Ks[i] == 0) continue;
    const int Se = Ss[i];
    auto out = [&](int q, int c) {
      const bool corner = (q == 0 || q == Se - 1) && (c == 0 || c == Se - 1);
      const int row = MODE == M_COL ? c : q;  // logical
      const bool mine = c < Se && !corner && (!EDGE || MODE == M_PASSIVE || (row > 0 && row <= 64));
      __builtin_amdgcn_raw_buffer_store_b32(as_i(lds[i * P * P + min(q, P - 1) * P + min(c, P - 1)]), xs[i],
                                            mine ? (q * Se + c) * 4 : -4, 0, 0);
    };
#pragma unroll
    for (int k = 0; k < P / NG; ++k) out(NG * k + le / LG, le % LG);
    if constexpr (EDGE) {
#pragma unroll
      for (int k = 0; k < 3; ++k) out(32 * k + (le >> 1), 64 + (le & 1));
    }
  }
}

template <int P, int LG, bool EDGE>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(P <= 16 ? 8 : P <= 32 ? 4 : P <= 64 ? 3 : 2)))
    k_lex_small(const RbScene* __restrict__ scs, const int2* __restrict__ tasks, LexArgs args) {
  constexpr int NG = 64 / LG;
  __shared__ float lds[NG * P * P];
  const int2 tk = tasks[blockIdx.x * NG + (threadIdx.x & 63) / LG];
  const LexSpec sp = args.sp[uni(tk.y)];  // the solves of a wave are of one kind (a slot without a scene has it too)
  if (sp.mode == M_ROW) solve<M_ROW, P, LG, EDGE>(lds, scs, tk.x, sp, args.press != 0);
  else if (sp.mode == M_COL) solve<M_COL, P, LG, EDGE>(lds, scs, tk.x, sp, args.press != 0);
  else solve<M_PASSIVE, P, LG, EDGE>(lds, scs, tk.x, sp, args.press != 0);
}

}  // namespace small

int lex_small_class(int S) { return S <= 16 ? 0 : S <= 32 ? 1 : S <= 48 ? 2 : S <= 64 ? 3 : S <= 66 ? 4 : -1; }
int lex_small_group(int cls) { return cls == 0 ? 4 : cls == 1 ? 2 : 1; }

void lex_small_launch(hipStream_t st, const RbScene* scs, const int2* tasks, int cls, int ntasks, const LexArgs& args) {
  if (ntasks <= 0) return;
  const dim3 n((unsigned)(ntasks / lex_small_group(cls))), t(64);
  if (cls == 0) hipLaunchKernelGGL((small::k_lex_small<16, 16, false>), n, t, 0, st, scs, tasks, args);
  else if (cls == 1) hipLaunchKernelGGL((small::k_lex_small<32, 32, false>), n, t, 0, st, scs, tasks, args);
  else if (cls == 2) hipLaunchKernelGGL((small::k_lex_small<48, 64, false>), n, t, 0, st, scs, tasks, args);
  else if (cls == 3) hipLaunchKernelGGL((small::k_lex_small<64, 64, false>), n, t, 0, st, scs, tasks, args);
  else hipLaunchKernelGGL((small::k_lex_small<66, 64, true>), n, t, 0, st, scs, tasks, args);
}

}  // namespace eqf
