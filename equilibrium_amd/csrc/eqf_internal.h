// eqf_internal.h -- host-side objects of libeqfluid.so shared by the
// runtime (eqf_runtime.hip) and the kernels' drivers (eqf_frame.hip, eqf_lex.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/eqfluid.h"
#include "eqf_layout.h"

// Pinned host memory that downloads of a context's scenes pass through, two
// chunks per download in progress (eqf_setup.hip).  Held by the context and by
// its scenes, whichever lives longest; at most KEEP buffers wait for reuse.
class HostStaging {
 public:
  static constexpr size_t CHUNK = (size_t)1 << 21;
  static constexpr int KEEP = 4;
  struct Buf {
    char* host = nullptr;  // 2 * CHUNK bytes
    hipEvent_t ev[2] = {nullptr, nullptr};
    Buf* next = nullptr;
  };
  explicit HostStaging(int device) : device_(device) {}
  ~HostStaging();
  HostStaging(const HostStaging&) = delete;
  HostStaging& operator=(const HostStaging&) = delete;
  Buf* take();  // nullptr: none to be had
  void give(Buf* b);

 private:
  static void drop(Buf* b);
  const int device_;
  std::mutex m_;
  Buf* free_ = nullptr;
  int nfree_ = 0;
};

// Polls of about a microsecond that a strip of a lexicographic lin_solve waits
// for the one above before it gives up and reports (eqf_ctx_set_wait_limit).
constexpr uint32_t LEX_POLLS = 1u << 22;

// What launches read of a context; held by its scenes too, which a batch of another
// context may step after it is gone.
struct LaunchLimits {
  int cus = 256;  // compute units of the device
  std::atomic<uint32_t> wait_polls{LEX_POLLS};
};

struct eqf_ctx {
  int device;
  std::shared_ptr<HostStaging> staging;
  std::shared_ptr<LaunchLimits> limits;
};

struct eqf_scene {
  eqf_ctx* ctx = nullptr;
  std::shared_ptr<HostStaging> staging;  // the context's
  std::shared_ptr<LaunchLimits> limits;  // the context's
  uint64_t uid = 0;  // unique per scene object of the process (never reused)
  eqf_params p{};
  int S = 0, N = 0;
  int64_t fstride = 0;
  std::vector<uint8_t> mask;  // row-major, host copy
  bool bnd_dirty = true;
  hipStream_t stream = nullptr;
  float* d_fld = nullptr;
  float* d_src = nullptr;
  int src_mask = 0;           // frame sources set: bit 0 density, 1 vx, 2 vy
  uint8_t* d_code = nullptr;
  uint8_t* d_rowf = nullptr;
  float* d_hand = nullptr;    // exact mode: hand-off values of its lin_solves
  int slots = 1;              // lin_solves of a frame that may run at once (scene_slots)
  int ring_copies = 0;        // Passive ring cells that copy their neighbour
  void* d_main = nullptr;     // one allocation: pad, fields, rule bytes, rowf, hand-off
  float* d_stage = nullptr;   // staging for eqf_add_source (lazy)
  uint8_t* d_mask = nullptr;  // mask + scratch for the boundary build (lazy)
  eqf::SceneDesc desc{};
  // Fields (a bit each) whose contents a failed frame left undefined, until they
  // are uploaded whole; frames that failed so far (frame_collect).
  std::atomic<uint32_t> invalid{0}, failures{0};
  struct eqf_snapshot* rings = nullptr;  // its snapshot rings (eqf_render.hip)
  int in_batch = 0;
  // Batch membership: the batch advances the scene on its own stream.  Work
  // queued on the scene's stream meanwhile first waits for the batch's last
  // step (eqf_internal_scene_enter), and the batch's next step waits for it
  // (ev_ops, recorded when ops_pending).
  struct eqf_batch* batch = nullptr;
  hipEvent_t ev_ops = nullptr;
  bool ops_pending = false;
  bool owns_stream = true;
  void* work = nullptr;     // frame workspace (eqf_frame.hip)
  // Scenes of a server allocate from the server's memory pool, ordered on
  // pool_stream (hipMallocFromPoolAsync / hipFreeAsync): freeing a retired
  // scene then waits for nothing else on the device, where hipFree would wait
  // for every stream.  Other scenes use hipMalloc / hipFree.
  hipMemPool_t pool = nullptr;
  hipStream_t pool_stream = nullptr;
};

// Device memory of a scene (see eqf_scene::pool).
hipError_t eqf_scene_malloc(eqf_scene* s, void** p, size_t bytes);
void eqf_scene_mfree(eqf_scene* s, void* p);

// Runtime services shared with the server (eqf_runtime.hip).
int eqf_internal_prepare(eqf_scene* s);  // boundary rules + descriptor
int eqf_internal_error(int code, const std::string& msg);
// Device address of eqf_render_rgba_noalloc's fixed scratch on `device`
// (eqf_render.hip), looked up once per device at context creation.
int eqf_internal_scratch_init(int device);
// Orders work about to be queued on the scene's stream after the last step of
// the scene's batch (no-op outside a batch).
int eqf_internal_scene_enter(eqf_scene* s);
// EQF_EDEVICE if a frame that has ended failed and left one of `fields` (a bit
// each) undefined.
int eqf_internal_check(const eqf_scene* s, uint32_t fields);
// The scene goes; its snapshot rings keep their captures.
void eqf_internal_rings_drop(eqf_scene* s);
int eqf_internal_check_params(const eqf_params* p);
// eqf_scene_create on a caller-owned stream (the server's admission stream),
// allocating from `pool` in that stream's order when `pool` is set; `slots` as
// scene_slots or 1.
int eqf_internal_scene_create(eqf_ctx* ctx, const eqf_params* p, hipStream_t stream, hipMemPool_t pool, int slots,
                              eqf_scene** out);
// Device memory of a scene that was prepared (with frame sources or without) and
// of its share of a launch group's tables.
uint64_t eqf_internal_scene_bytes(const eqf_params* p, int slots, bool sources);

// Device-side setup (eqf_setup.hip).
int eqf_dev_init_fields(eqf_scene* s, int times);
int eqf_dev_upload(eqf_scene* s, float* dst, float* dst2, const float* host, int add);
int eqf_dev_download(eqf_scene* s, const float* src, float* host);
// src field -> another device array, queued on the scene's stream.
int eqf_dev_copy_async(eqf_scene* s, const float* src, float* dst);
int eqf_dev_rebuild_bnd(eqf_scene* s);
size_t eqf_dev_mask_bytes(int S);
void eqf_dev_trim(eqf_scene* s);

namespace eqf {

// One scene of a launch group: a single scene, or every scene of a batch.
// Each frame kernel covers all scenes of its group in one launch.
struct RbScene {
  SceneDesc d;  // the scene's descriptor (a copy): fields, sizes, coefficients, rule bytes
  float* tmp[3];  // its ping-pong fields (red-black mode)
};

// Lexicographic lin_solve (eqf_lex.hip).  A launch covers up to three
// lin_solves (slots) of every scene; a task is one strip of one of them.
struct LexTask {
  int scene, slot;
  int strip, nstrips;
  int flag;      // its progress count; the strip above has the one before
  int pad;
  float* hand;  // its hand-off values (of the strip above: lex_handoff_floats before)
};
struct LexSpec {
  int mode, x_role, x0_role, coef;
};
struct LexArgs {
  LexSpec sp[3];
  int round, press;  // round of sweeps; which iteration count (0 diffusion, 1 pressure)
  uint32_t polls;    // how often a strip looks for the one above before it gives up (and reports)
};
// ctl: ticket, ended workgroups, then nflags progress counts, all zero before
// the first launch; a launch leaves them zero.  maxN: the largest scene's; cus: the
// device's compute units.
void lex_launch(hipStream_t st, const RbScene* scs, const LexTask* tasks, int ntasks, const LexArgs& args,
                uint32_t* ctl, int nflags, uint32_t* err, int maxN, int cus);

// ... of many small scenes, whole solves (eqf_lex_small.hip).  Class of a size (-1:
// none), solves of one kind that a wave takes (ntasks is a multiple of them;
// tasks: {scene, slot}, scene -1: none, not the first of a wave).
int lex_small_class(int S);
int lex_small_group(int cls);
constexpr int LEX_SMALL_CLASSES = 5;
void lex_small_launch(hipStream_t st, const RbScene* scs, const int2* tasks, int cls, int ntasks, const LexArgs& args);

// Frames (eqf_frame.hip).  A launch group's scenes share one mode.
void* frame_create(eqf_scene* s, std::string& err);
void frame_destroy(eqf_scene* s);
int frame_step(eqf_scene* s, int64_t nframes, std::string& err);
int frame_set_tiling(eqf_scene* s, int tile, int tsweeps);
// A batch of scenes of one mode: every frame kernel covers all of them.
void* group_create(const std::vector<eqf_scene*>& scenes, hipStream_t st, std::string& err);
void group_destroy(void* g);
int group_set_tiling(void* g, int tile, int tsweeps);
int group_step_frames(void* g, int64_t nframes, std::string& err);
void group_set_scenes(void* g, const std::vector<eqf_scene*>& scenes);
// A wait inside a kernel of the group that gave up (never in a sound run): marks
// its scenes (eqf_scene::invalid, failures), and lets the next step set the
// group's counters up again.  For frames that have ended.
bool group_collect(void* g);
bool frame_collect(const eqf_scene* s);
// Device bytes of a scene's share of its group's tables.
int64_t frame_table_bytes(int S, bool exact);
}  // namespace eqf
