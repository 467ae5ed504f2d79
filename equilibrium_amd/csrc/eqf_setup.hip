// eqf_setup.hip -- device-side scene setup: initial state, uploads, downloads
// and adds of whole fields, and the boundary rules derived from the obstacle mask.  Keeping these on the device makes
// admitting a scene cost a few small launches instead of host loops over
// every cell, which matters when the server admits hundreds of scenes/s.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <new>
#include <string>
#include <vector>

#include "eqf_internal.h"

using namespace eqf;

namespace {

struct Geo {
  int S, N;
};

__device__ __forceinline__ int off_of(const Geo& g, int x, int y) { return x + y * g.S; }

// Fluid::new / Fluid::default state (fluid.rs:93-110, 527-570) for sizes
// where the density block needs no index clamping (S >= 22): U = V = `times`
// additions of 1.0, D = S = `times` additions of 0.9 on [S/2-10, S/2+10]^2.
__global__ void k_init(Geo g, float* __restrict__ f, int64_t fs, int times) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (int64_t)g.S * g.S) return;
  const int x = (int)(e % g.S), y = (int)(e / g.S);
  const int64_t o = off_of(g, x, y);
  float vel = 0.0f, den = 0.0f;
  const int lo = g.S / 2 - 10, hi = g.S / 2 + 10;
  const bool blk = x >= lo && x <= hi && y >= lo && y <= hi;
  for (int t = 0; t < times; ++t) {
    vel += 1.0f;
    den += blk ? 0.9f : 0.0f;
  }
  f[F_D * fs + o] = den;
  f[F_SC * fs + o] = den;
  f[F_U * fs + o] = vel;
  f[F_V * fs + o] = vel;
  f[F_U0 * fs + o] = 0.0f;
  f[F_V0 * fs + o] = 0.0f;
}

// dst += src (and dst2 += src when dst2 is set: add_density writes density and scratch).
__global__ void k_add(int64_t n, const float* __restrict__ src, float* __restrict__ dst, float* __restrict__ dst2) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const float v = src[e];
  dst[e] += v;
  if (dst2) dst2[e] += v;
}

// rowf[j] / colf[i]: row / column holds a NoWall cell (Passive copy rule of
// fluid.rs:179-187).  A 2D grid of 256-column x 64-row tiles: each thread ORs
// its column over the tile's rows (coalesced row reads), each wave ORs every
// row over its 64 columns with a wave vote, and tiles combine through atomic
// ORs into zeroed 32-bit flags; k_rowcol_bytes turns them into the byte arrays.
__global__ void __launch_bounds__(256) k_rowcol_or(Geo g, const uint8_t* __restrict__ m, uint32_t* __restrict__ rowf32,
                                                   uint32_t* __restrict__ colf32) {
  const int S = g.S;
  const int x = blockIdx.x * 256 + threadIdx.x;
  const int y0 = blockIdx.y * 64;
  const int y1 = min(y0 + 64, S);
  uint32_t c = 0;
  for (int y = y0; y < y1; ++y) {  // uniform bounds: every lane takes part in the vote
    const bool f = x < S && m[(int64_t)y * S + x] != EQF_DEFAULT_WALL;
    c |= f ? 1u : 0u;
    if (__any(f) && (threadIdx.x & 63) == 0) atomicOr(&rowf32[y], 1u);
  }
  if (c) atomicOr(&colf32[x], 1u);
}

__global__ void k_rowcol_bytes(int S, const uint32_t* __restrict__ rowf32, const uint32_t* __restrict__ colf32,
                               uint8_t* __restrict__ rowf, uint8_t* __restrict__ colf) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= S) return;
  rowf[k] = rowf32[k] != 0;
  colf[k] = colf32[k] != 0;
}

// Per-cell rule bytes (eqf_layout.h RuleBits): AdjustRow (right wall wins over
// left, fluid.rs:151-164), AdjustColumn (up wins over down, fluid.rs:165-177),
// Passive ring copies (counted).
__global__ void k_codes(Geo g, const uint8_t* __restrict__ m, const uint8_t* __restrict__ rowf,
                        const uint8_t* __restrict__ colf, uint8_t* __restrict__ code, int arrays, int* __restrict__ copies) {
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int S = g.S, N = g.N;
  if (e >= (int64_t)S * S) return;
  const int x = (int)(e % S), y = (int)(e / S);
  auto wall = [&](int i, int j) { return m[(int64_t)j * S + i] == EQF_DEFAULT_WALL; };
  auto put = [&](int i, int j, uint32_t r) {
    code[(int64_t)j * rm_code_stride(S) + i] = (uint8_t)r;
    if (arrays > 1) code[rm_code_bytes(S) + (int64_t)i * rm_code_stride(S) + j] = (uint8_t)r;
  };
  if (x >= 1 && x <= N && y >= 1 && y <= N) {
    uint32_t r = R_INTERIOR;
    if (!wall(x, y)) {
      r |= (wall(x + 1, y) ? R_NEG_SECOND : wall(x - 1, y) ? R_NEG_FIRST : 0u) << R_ROW_SHIFT;
      r |= (wall(x, y - 1) ? R_NEG_FIRST : wall(x, y + 1) ? R_NEG_SECOND : 0u) << R_COL_SHIFT;
    } else {
      if (!wall(x - 1, y) || (!wall(x + 1, y) && !wall(x + 2, y))) r |= R_SOURCE << R_ROW_SHIFT;
      if (!wall(x, y + 1) || (!wall(x, y - 1) && !wall(x, y - 2))) r |= R_SOURCE << R_COL_SHIFT;
    }
    put(x, y, r);
  } else if (!((x == 0 || x == S - 1) && (y == 0 || y == S - 1))) {  // non-corner ring cell
    if ((y == 0 || y == S - 1) ? colf[x] : rowf[y]) {
      atomicAdd(copies, 1);
      put(x, y, (y == 0 ? R_COPY_DOWN : y == S - 1 ? R_COPY_UP : x == 0 ? R_COPY_RIGHT : R_COPY_LEFT) << R_PAS_SHIFT);
    }
  }
}

Geo geo_of(const eqf_scene* s) { return Geo{s->S, s->N}; }

unsigned blocks_for(int64_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace

int eqf_dev_init_fields(eqf_scene* s, int times) {
  const int64_t n = (int64_t)s->S * s->S;
  hipLaunchKernelGGL(k_init, dim3(blocks_for(n)), dim3(256), 0, s->stream, geo_of(s), s->d_fld, s->fstride, times);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? EQF_OK : eqf_internal_error(EQF_EDEVICE, std::string("init: ") + hipGetErrorString(e));
}

static int ensure_stage(eqf_scene* s) {
  if (s->d_stage) return EQF_OK;
  hipError_t e = eqf_scene_malloc(s, (void**)&s->d_stage, sizeof(float) * (size_t)s->S * s->S + 256);
  return e == hipSuccess ? EQF_OK
                         : eqf_internal_error(EQF_ENOMEM, std::string("staging buffer: ") + hipGetErrorString(e));
}

int eqf_dev_upload(eqf_scene* s, float* dst, float* dst2, const float* host, int add) {
  const size_t n = (size_t)s->S * s->S;
  float* to = dst;
  if (add) {
    int rc = ensure_stage(s);
    if (rc) return rc;
    to = s->d_stage;
  }
  hipError_t e = hipMemcpyAsync(to, host, sizeof(float) * n, hipMemcpyHostToDevice, s->stream);
  if (e == hipSuccess && add) {
    hipLaunchKernelGGL(k_add, dim3(blocks_for((int64_t)n)), dim3(256), 0, s->stream, (int64_t)n, s->d_stage, dst, dst2);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipStreamSynchronize(s->stream);
  return e == hipSuccess ? EQF_OK : eqf_internal_error(EQF_EDEVICE, std::string("upload: ") + hipGetErrorString(e));
}

int eqf_dev_copy_async(eqf_scene* s, const float* src, float* dst) {
  const hipError_t e =
      hipMemcpyAsync(dst, src, sizeof(float) * (size_t)s->S * s->S, hipMemcpyDeviceToDevice, s->stream);
  return e == hipSuccess ? EQF_OK : eqf_internal_error(EQF_EDEVICE, std::string("field copy: ") + hipGetErrorString(e));
}

HostStaging::~HostStaging() {
  while (free_) {
    Buf* b = free_;
    free_ = b->next;
    drop(b);
  }
}

void HostStaging::drop(Buf* b) {
  for (hipEvent_t e : b->ev)
    if (e) (void)hipEventDestroy(e);
  if (b->host) (void)hipHostFree(b->host);
  delete b;
}

HostStaging::Buf* HostStaging::take() {
  {
    std::lock_guard<std::mutex> lk(m_);
    if (Buf* b = free_) {
      free_ = b->next;
      --nfree_;
      return b;
    }
  }
  Buf* b = new (std::nothrow) Buf;
  if (!b) return nullptr;
  int cur = device_;  // events belong to a device; the caller's current one stays
  hipError_t e = hipGetDevice(&cur);
  if (e == hipSuccess && cur != device_) e = hipSetDevice(device_);
  if (e == hipSuccess) {
    e = hipHostMalloc((void**)&b->host, 2 * CHUNK, hipHostMallocDefault);
    for (hipEvent_t& ev : b->ev)
      if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
    if (cur != device_) (void)hipSetDevice(cur);
  }
  if (e == hipSuccess) return b;
  (void)hipGetLastError();  // the caller does without
  drop(b);
  return nullptr;
}

void HostStaging::give(Buf* b) {
  if (!b) return;
  {
    std::lock_guard<std::mutex> lk(m_);
    if (nfree_ < KEEP) {
      b->next = free_;
      free_ = b;
      ++nfree_;
      return;
    }
  }
  drop(b);
}

// Memory that the device writes by itself: pinned, managed or its own.
static bool device_writes(const void* p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return a.type != hipMemoryTypeUnregistered;
}

// Field -> the caller's memory, through pinned chunks: one is copied out while
// the next arrives.  The runtime's own copy to memory that is not pinned pins
// it for the time, or goes through small chunks: 512 fields of S 66..514 (178
// MB) took it 35 to 88 ms depending on where the memory lies, one of S = 1026
// 238 us; this takes 14 ms and 180 us, about 40 us per MB of which is the host
// reading what just arrived, on top of 10 us for the first copy.  Chunks of 1
// MB took 15 ms and 185 us, of 512 KB 16 ms and 225 us: each costs the wait for
// its event.  Where the device writes the caller's memory by itself the copy goes
// straight there: 67 MB into pinned memory 1.19 ms, through the chunks 2.51.
int eqf_dev_download(eqf_scene* s, const float* src, float* host) {
  const size_t bytes = sizeof(float) * (size_t)s->S * s->S;
  const bool direct = device_writes(host) && device_writes((const char*)host + bytes - 1);
  HostStaging::Buf* b = s->staging && !direct ? s->staging->take() : nullptr;
  hipError_t e = hipSuccess;
  if (!b) {
    e = hipMemcpyAsync(host, src, bytes, hipMemcpyDeviceToHost, s->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(s->stream);
  } else {
    const size_t n = (bytes + HostStaging::CHUNK - 1) / HostStaging::CHUNK;
    const size_t C = ((bytes + n - 1) / n + 63) & ~(size_t)63;  // equal chunks
    auto len = [&](size_t i) { return std::min(C, bytes - i * C); };
    auto fetch = [&](size_t i) {
      hipError_t r = hipMemcpyAsync(b->host + (i & 1) * C, (const char*)src + i * C, len(i), hipMemcpyDeviceToHost, s->stream);
      if (r == hipSuccess && i + 1 < n) r = hipEventRecord(b->ev[i & 1], s->stream);
      return r;
    };
    e = fetch(0);
    for (size_t i = 0; i < n && e == hipSuccess; ++i) {
      if (i + 1 < n) e = fetch(i + 1);
      if (e == hipSuccess) e = i + 1 < n ? hipEventSynchronize(b->ev[i & 1]) : hipStreamSynchronize(s->stream);
      if (e == hipSuccess) std::memcpy((char*)host + i * C, b->host + (i & 1) * C, len(i));
    }
    if (e != hipSuccess) (void)hipStreamSynchronize(s->stream);  // no copy into the buffer is left
    s->staging->give(b);
  }
  return e == hipSuccess ? EQF_OK : eqf_internal_error(EQF_EDEVICE, std::string("download: ") + hipGetErrorString(e));
}

void eqf_dev_trim(eqf_scene* s) {
  eqf_scene_mfree(s, s->d_stage);
  s->d_stage = nullptr;
  eqf_scene_mfree(s, s->d_mask);
  s->d_mask = nullptr;
}

// Layout of the scene's d_mask buffer: the mask (S*S bytes), colf (S bytes),
// then the 32-bit row/column flags (2*S) and k_codes' counter, zeroed by one
// memset.
struct MaskBuf {
  size_t colf, flags, cnt, bytes;
};
static MaskBuf mask_buf(int S) {
  const size_t n = (size_t)S * S;
  auto up = [](size_t v) { return (v + 15) & ~(size_t)15; };
  MaskBuf b;
  b.colf = up(n);
  b.flags = up(b.colf + (size_t)S);
  b.cnt = b.flags + 8 * (size_t)S;
  b.bytes = b.cnt + sizeof(int);
  return b;
}

size_t eqf_dev_mask_bytes(int S) { return mask_buf(S).bytes; }

int eqf_dev_rebuild_bnd(eqf_scene* s) {
  const int S = s->S, arrays = rm_code_arrays(s->p.gs_mode == EQF_GS_WAVEFRONT);
  const int64_t n = (int64_t)S * S;
  const MaskBuf mb = mask_buf(S);
  hipError_t e = hipSuccess;
  if (!s->d_mask) e = eqf_scene_malloc(s, (void**)&s->d_mask, mb.bytes);
  if (e != hipSuccess) return eqf_internal_error(EQF_ENOMEM, std::string("mask buffer: ") + hipGetErrorString(e));
  uint8_t* d_colf = s->d_mask + mb.colf;
  uint32_t* d_flags = (uint32_t*)(s->d_mask + mb.flags);
  int* d_cnt = (int*)(s->d_mask + mb.cnt);
  const Geo g = geo_of(s);
  e = hipMemcpyAsync(s->d_mask, s->mask.data(), (size_t)n, hipMemcpyHostToDevice, s->stream);
  if (e == hipSuccess) e = hipMemsetAsync(d_flags, 0, mb.bytes - mb.flags, s->stream);
  if (e == hipSuccess) e = hipMemsetAsync(s->d_code, 0, arrays * (size_t)rm_code_bytes(S), s->stream);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_rowcol_or, dim3((unsigned)((S + 255) / 256), (unsigned)((S + 63) / 64)), dim3(256), 0,
                       s->stream, g, s->d_mask, d_flags, d_flags + S);
    hipLaunchKernelGGL(k_rowcol_bytes, dim3(blocks_for(S)), dim3(256), 0, s->stream, S, d_flags, d_flags + S,
                       s->d_rowf, d_colf);
    hipLaunchKernelGGL(k_codes, dim3(blocks_for(n)), dim3(256), 0, s->stream, g, s->d_mask, s->d_rowf, d_colf,
                       s->d_code, arrays, d_cnt);
    e = hipGetLastError();
  }
  int copies = 0;
  if (e == hipSuccess) e = hipMemcpyAsync(&copies, d_cnt, sizeof(copies), hipMemcpyDeviceToHost, s->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(s->stream);
  if (e != hipSuccess) return eqf_internal_error(EQF_EDEVICE, std::string("boundary codes: ") + hipGetErrorString(e));
  s->ring_copies = copies;
  s->bnd_dirty = false;
  return EQF_OK;
}
