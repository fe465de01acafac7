// Dense RGB-D tracker: the reference's RGBDTracking
// (RGBDFusion/src/RGBDTracking.cu, RGBDFusion/include/TrackingUtils.h) and the
// image operations it uses (RGBDFusion/src/ImageProc.cu).
//
// MI355X design: the whole Gauss-Newton loop stays on the device, with no
// host round trip and no fence inside a kernel (on the multi-XCD gfx950 an
// agent-scope fence writes back the L2): the separate passes meet at kernel
// boundaries, and the workgroups of the one-launch solve wait for each other's
// words, which carry their iteration.  One iteration is:
//   pass 1   grid-stride over the level's pixels: ICP point-to-plane rows
//            (28 upper-triangle products + count) and photometric residuals
//            with per-thread Welford statistics; each workgroup reduces its
//            values (transpose butterfly across the 64 lanes, LDS across
//            waves) into one row of partials.
//   pass 2   (photometric) every workgroup folds pass 1's statistics rows in
//            the same fixed order, so all agree on mean, sigma and the Huber
//            threshold, then reduces the weighted photometric rows.
//   update   one workgroup folds the partial rows in a fixed order, solves
//            the 6x6 system in FP64 (the reference's Eigen LDLT, restated),
//            applies T <- exp(xi) T in FP64 and keeps the best pose.
// A full solve runs all of its iterations in one launch (k_solve,
// yas_solve_dev.hpp) where its workgroups can be resident at once
// (solve_in_one says when); otherwise it takes each update but the last at the
// start of the next pass 1: every workgroup of that pass folds the same rows
// and takes the same step, one launch fewer per iteration.  The values are the
// same either way.
// Results are deterministic run to run.
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "yas_internal.hpp"
#include "yas_frame_dev.hpp"
#include "yas_frame_host.hpp"
#include "yas_tracker_dev.hpp"
#include "yas_solve_dev.hpp"
#include "yas_server_dev.hpp"

using namespace yas;

constexpr int kMaxSolveDevices = 64;
constexpr long long kSolveMaxPixels = 1 << 26;  // 32-bit byte offsets in yas_solve_dev.hpp
// 20 ms: between two words that a workgroup waits for lies at most an
// iteration (16 us at 640x480, 0.8 ms at 4096x3072, 4 ms at kSolveMaxPixels),
// and its workgroups wait for a CU at most as long as other kernels hold one.
constexpr unsigned long long kSolveWaitTicks = 2000000ull;
// Solves that are separate passes after one that was lost, twice as many after
// the next loss, up to kMaxPasses; a solve in one launch begins anew.  A lost
// solve costs its wait and, queued, the rescue (3.4 ms at 320x240 with depth
// alone, 65 ms at 640x480 with both terms); the passes cost 0.03 to 0.11 ms a
// solve more than the one launch (150 / 180 us and 306 / 415 us waited for).
constexpr int kFirstPasses = 64, kMaxPasses = 8192;

namespace {

__global__ void __launch_bounds__(256) k_rgb_to_gray(const uint8_t* rgb, size_t sp, float* dst, size_t dp, int W,
                                                     int H, int mode) {
  rgb_to_gray_at(rgb, sp, dst, dp, W, H, mode, blockIdx.x, blockIdx.y);
}

__global__ void __launch_bounds__(256) k_pyrdown_gauss(const float* src, size_t sp, int sw, int sh, float* dst,
                                                       size_t dp, int dw, int dh) {
  pyrdown_gauss_at(src, sp, sw, sh, dst, dp, dw, dh, blockIdx.x, blockIdx.y);
}

__global__ void __launch_bounds__(256) k_gradient(const float* s, size_t sp, float* gx, float* gy, size_t dp, int W,
                                                  int H) {
  gradient_at(s, sp, gx, gy, dp, W, H, blockIdx.x, blockIdx.y);
}

__global__ void __launch_bounds__(256) k_invdepth(const float* z, size_t sp, float* o, size_t dp, int W, int H) {
  invdepth_at(z, sp, o, dp, W, H, blockIdx.x, blockIdx.y);
}

__global__ void __launch_bounds__(256) k_pyrdown_depth(const float* s, size_t sp, float* o, size_t dp, int W, int H) {
  pyrdown_depth_at(s, sp, o, dp, W, H, blockIdx.x, blockIdx.y);
}

__global__ void __launch_bounds__(256) k_vertex(const float* inv, size_t sp, float4* v, size_t dp, int W, int H,
                                                float invfx, float invfy, float cx, float cy, float cut) {
  vertex_at(inv, sp, v, dp, W, H, invfx, invfy, cx, cy, cut, blockIdx.x, blockIdx.y);
}

__global__ void __launch_bounds__(256) k_normal(const float4* v, size_t sp, float4* n, size_t dp, int W, int H) {
  normal_at(v, sp, n, dp, W, H, blockIdx.x, blockIdx.y);
}

__global__ void __launch_bounds__(256) k_vmap_to_depth(const float4* v, size_t sp, float* d, size_t dp, int W, int H) {
  vmap_to_depth_at(v, sp, d, dp, W, H, blockIdx.x, blockIdx.y);
}

template <bool ICP, bool RGB>
__global__ void __launch_bounds__(256) k_pass1(Level L, TrackBufs B, const TrackState* st, float* part_icp,
                                               float* part_res, float sin2_max, float dist2_max) {
  pass1_at<ICP, RGB, true>(L, B, st, part_icp, part_res, sin2_max, dist2_max, blockIdx.x, gridDim.x);
}
__global__ void __launch_bounds__(256) k_pass2(Level L, TrackBufs B, TrackState* st, const float* part_res, int g1,
                                               float* part_rgb) {
  pass2_at<true>(L, B, st, part_res, g1, part_rgb, blockIdx.x, gridDim.x);
}
__global__ void __launch_bounds__(256) k_update(TrackState* st, const float* part_icp, int gi, const float* part_rgb,
                                                int gr, int mode, int first_of_level, int do_step, int record,
                                                float wrh, float wrb, float wih, float wib) {
  update_at(st, part_icp, gi, part_rgb, gr, mode, first_of_level, do_step, record, wrh, wrb, wih, wib);
}
// The last step of a solve, from the state buffer the last pass used into the
// tracker's state; in host memory (if `host`), that solve `number` has ended.
__global__ void __launch_bounds__(256) k_update_into(const TrackState* st_in, TrackState* st_out, StepArgs a,
                                                     HostState* host, unsigned number) {
  if (host && threadIdx.x == 0)
    __hip_atomic_store(&host->ended, number, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  gn_update(st_in, st_out, true, a.part_icp, a.gi, a.part_rgb, a.gr, a.mode, a.first_of_level, 1, a.record, a.wrh,
            a.wrb, a.wih, a.wib, nullptr);
}
// Step of the previous linearisation, then pass 1 at the new pose.
template <bool ICP, bool RGB>
__global__ void __launch_bounds__(256) k_step_pass1(Level L, TrackBufs B, StepArgs a, float* part_icp,
                                                    float* part_res, float sin2_max, float dist2_max) {
  pass1_at<ICP, RGB, true, true>(L, B, nullptr, part_icp, part_res, sin2_max, dist2_max, blockIdx.x, gridDim.x, &a);
}
// The whole solve in one launch (yas_solve_dev.hpp).  1024 threads a
// workgroup, so 128 registers a lane; one workgroup per CU.  Bound by the
// chain of an iteration (15.8 us at 640x480 with both terms, 7.4 us at 320x240
// with depth alone): the pixels' gathers, the wavefronts' sums and the fold,
// two or three messages between workgroups of about 1.4 us each, the step
// 2.4 us.  The launch-per-pass iteration took 27 us (24 us at small sizes).
template <bool ICP, bool RGB>
__global__ void __launch_bounds__(kSolveThreads) k_solve(SolveArgs a) {
  solve_body<ICP, RGB>(solve_lds(), a);
}
// Takes a solve whose workgroups did not meet; nothing to do otherwise, but to
// say in host memory that solve `number` has ended (and how many it took).
template <bool ICP, bool RGB>
__global__ void __launch_bounds__(256) k_solve_rescue(SolveArgs a, HostState* host, unsigned number) {
  if (threadIdx.x == 0) {
    if (!a.x->ok) {
      a.x->rescued++;
      __hip_atomic_store(&host->rescued, a.x->rescued, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    __hip_atomic_store(&host->ended, number, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  solve_rescue<ICP, RGB>(a);
}
// The epochs that a lost solve may have used are skipped.
__global__ void k_solve_skip(SolveXchg* x, unsigned iterations) {
  if (threadIdx.x == 0) x->epoch += iterations;
}
// All levels of an image, a depth image or a model in one launch (yas_frame_dev.hpp).
__global__ void __launch_bounds__(256) k_image_levels(ImageArgs<SrcF32> a) {
  __shared__ ImageLds S;
  image_tile(a, blockIdx.x, S);
}
__global__ void __launch_bounds__(256) k_depth_levels(DepthArgs<SrcF32> a) { depth_tile(a, blockIdx.x); }
__global__ void __launch_bounds__(256) k_model_levels(ModelArgs a) { model_tile(a, blockIdx.x); }
__global__ void k_track_init(TrackState* st, Mat44 T) { track_init_at(st, T.m); }
__global__ void k_track_init_identity(TrackState* st) { track_init_identity_at(st); }

inline dim3 grid64x4(int W, int H) { return dim3((W + 63) / 64, (H + 3) / 4); }

}  // namespace

// ------------------------------------------------------------------ host
struct yas_tracker {
  yas_ctx* ctx;
  int W, H;
  yas_tracker_params P;
  Level lv[kMaxLevels];
  float *cur_int[kMaxLevels], *ref_int[kMaxLevels], *gx[kMaxLevels], *gy[kMaxLevels];
  float *cur_inv[kMaxLevels], *ref_inv[kMaxLevels];
  float4 *cur_v[kMaxLevels], *ref_v[kMaxLevels];
  float4 *cur_p[kMaxLevels], *ref_p[kMaxLevels];  // ICP point maps (what the ICP term reads)
  float4 *cur_n[kMaxLevels], *ref_n[kMaxLevels];    // normal maps, formed on request (yas_tracker_level)
  float3* resid[kMaxLevels];
  float* part_icp;  // [kRedGroups][32]
  float* part_icp2;  // the other of the pair a solve alternates between
  float* part_res;  // [kRedGroups][4]
  float* part_rgb;  // [kRedGroups][32]
  TrackState* st;
  TrackState* st2;  // a solve's steps alternate between st and st2
  HostState* host_st;
  SolveXchg* xchg;               // words the one-launch solve's workgroups exchange
  unsigned long long wait_ticks; // bound of its waits (100 MHz clock)
  unsigned solves;               // number of the last solve enqueued (but those recorded into graphs)
  bool listed, one;              // in its device's list (g_solves); the last solve is a one-launch solve
  yas_tracker* next;             // in that list
  unsigned tried, last_tried;    // one-launch solves launched, and the last one's number
  unsigned lost_waited;          // those lost that were waited for (the others: host_st->rescued)
  unsigned by_passes;            // solves that were separate passes from the start
  unsigned lost_seen, tried_seen;  // lost solves known, and solves tried when the last was found
  int passes_left, passes_next;  // solves to take by passes, and after the next loss
  float sin2_max, dist2_max;
  float* raw_depth;  // depth uploaded by the host-image setters (W*H, lazily allocated)
  float* raw_image;  // intensity uploaded by the host-image setters
};

static int image_pyramid(yas_tracker* t, const float* g, size_t pitch, float** pyr, bool grads) {
  hipStream_t s = t->ctx->stream;
  // three levels a launch; the next launch starts at the last of them
  for (int base = 0; base == 0 || base + 1 < t->P.levels; base += kImageLevels - 1) {
    ImageArgs<SrcF32> a;
    if (base == 0) a.src = SrcF32{g, pitch};
    else a.src = SrcF32{pyr[base], (size_t)t->lv[base].w * 4};
    fill_image(a, t->lv, t->P.levels, base, pyr, grads ? t->gx : nullptr, grads ? t->gy : nullptr);
    hipLaunchKernelGGL(k_image_levels, dim3(a.tiles), dim3(256), 0, s, a);
  }
  YAS_LAUNCH_CHECK();
  return YAS_OK;
}

static int depth_pyramid(yas_tracker* t, const float* d, size_t pitch, float** inv, float4** v, float4** pt) {
  DepthArgs<SrcF32> a;
  a.src = SrcF32{d, pitch};
  fill_depth(a, t->lv, t->P.levels, inv, v, pt);
  hipLaunchKernelGGL(k_depth_levels, dim3(a.t.first[a.t.n]), dim3(256), 0, t->ctx->stream, a);
  YAS_LAUNCH_CHECK();
  return YAS_OK;
}

static int model_pyramid(yas_tracker* t, const float* vmap, size_t pitch) {
  ModelArgs a;
  a.src = (const float4*)vmap;
  a.pitch = pitch;
  fill_tiles(a.t, t->lv, t->P.levels);
  for (int l = 0; l < t->P.levels; ++l) {
    a.v[l] = t->ref_v[l];
    a.p[l] = t->ref_p[l];
  }
  hipLaunchKernelGGL(k_model_levels, dim3(a.t.first[a.t.n]), dim3(256), 0, t->ctx->stream, a);
  YAS_LAUNCH_CHECK();
  return YAS_OK;
}

static int groups_for(const Level& a) {
  int n = (a.w * a.h + 1023) / 1024;  // about 4 pixels per thread
  return n < 1 ? 1 : (n > kRedGroups ? kRedGroups : n);
}

static TrackBufs bufs(yas_tracker* t, int l) {
  TrackBufs B;
  B.ref_v = t->ref_v[l]; B.ref_p = t->ref_p[l]; B.cur_v = t->cur_v[l]; B.cur_p = t->cur_p[l];
  B.ref_inv = t->ref_inv[l]; B.ref_int = t->ref_int[l]; B.cur_int = t->cur_int[l];
  B.gx = t->gx[l]; B.gy = t->gy[l]; B.resid = t->resid[l];
  return B;
}

// One linearisation at level l (icp / rgb terms as requested) followed by the
// fold and, when do_step, one Gauss-Newton step.
static int launch_iteration(yas_tracker* t, int l, bool icp, bool rgb, bool do_step, bool first_of_level) {
  const Level& a = t->lv[l];
  hipStream_t s = t->ctx->stream;
  const int G = groups_for(a);
  TrackBufs B = bufs(t, l);
  if (icp && rgb)
    hipLaunchKernelGGL((k_pass1<true, true>), dim3(G), dim3(256), 0, s, a, B, (const TrackState*)t->st, t->part_icp,
                       t->part_res, t->sin2_max, t->dist2_max);
  else if (icp)
    hipLaunchKernelGGL((k_pass1<true, false>), dim3(G), dim3(256), 0, s, a, B, (const TrackState*)t->st, t->part_icp,
                       t->part_res, t->sin2_max, t->dist2_max);
  else
    hipLaunchKernelGGL((k_pass1<false, true>), dim3(G), dim3(256), 0, s, a, B, (const TrackState*)t->st, t->part_icp,
                       t->part_res, t->sin2_max, t->dist2_max);
  if (rgb)
    hipLaunchKernelGGL(k_pass2, dim3(G), dim3(256), 0, s, a, B, t->st, (const float*)t->part_res, G, t->part_rgb);
  hipLaunchKernelGGL(k_update, dim3(1), dim3(256), 0, s, t->st, (const float*)t->part_icp, icp ? G : 0,
                     (const float*)t->part_rgb, rgb ? G : 0, t->P.mode, first_of_level ? 1 : 0, do_step ? 1 : 0,
                     l == 0 ? 1 : 0, t->P.w_rgb_h, t->P.w_rgb_b, t->P.w_icp_h, t->P.w_icp_b);
  YAS_LAUNCH_CHECK();
  return YAS_OK;
}

// Coarse-to-fine Gauss-Newton from the pose already in the device state:
// the same linearisations and steps as launch_iteration in sequence, with
// each step (but the last) taken at the start of the next pass 1, which
// saves one launch per iteration.  Step i reads the state buffer of step
// i - 1 and writes the other one, and the ICP partial rows alternate the
// same way, since that pass 1 reads the previous rows while writing its own.
static int solve_by_passes(yas_tracker* t, bool numbered) {
  const bool icp = t->P.mode != YAS_TRACK_RGB, rgb = t->P.mode != YAS_TRACK_DEPTH;
  hipStream_t s = t->ctx->stream;
  TrackState* S[2] = {t->st, t->st2};
  float* PI[2] = {t->part_icp, t->part_icp2};
  StepArgs a = {};
  int i = 0;
  for (int l = t->P.levels - 1; l >= 0; --l)
    for (int it = 0; it < t->P.iters[l]; ++it, ++i) {
      const Level& lv = t->lv[l];
      const int G = groups_for(lv);
      const TrackBufs B = bufs(t, l);
      TrackState* cur = S[i & 1];
      float* pic = PI[i & 1];
      if (i == 0) {
        if (icp && rgb)
          hipLaunchKernelGGL((k_pass1<true, true>), dim3(G), dim3(256), 0, s, lv, B, (const TrackState*)cur, pic,
                             t->part_res, t->sin2_max, t->dist2_max);
        else if (icp)
          hipLaunchKernelGGL((k_pass1<true, false>), dim3(G), dim3(256), 0, s, lv, B, (const TrackState*)cur, pic,
                             t->part_res, t->sin2_max, t->dist2_max);
        else
          hipLaunchKernelGGL((k_pass1<false, true>), dim3(G), dim3(256), 0, s, lv, B, (const TrackState*)cur, pic,
                             t->part_res, t->sin2_max, t->dist2_max);
      } else {
        a.st_in = S[(i - 1) & 1];
        a.st_out = cur;
        if (icp && rgb)
          hipLaunchKernelGGL((k_step_pass1<true, true>), dim3(G), dim3(256), 0, s, lv, B, a, pic, t->part_res,
                             t->sin2_max, t->dist2_max);
        else if (icp)
          hipLaunchKernelGGL((k_step_pass1<true, false>), dim3(G), dim3(256), 0, s, lv, B, a, pic, t->part_res,
                             t->sin2_max, t->dist2_max);
        else
          hipLaunchKernelGGL((k_step_pass1<false, true>), dim3(G), dim3(256), 0, s, lv, B, a, pic, t->part_res,
                             t->sin2_max, t->dist2_max);
      }
      if (rgb)
        hipLaunchKernelGGL(k_pass2, dim3(G), dim3(256), 0, s, lv, B, cur, (const float*)t->part_res, G, t->part_rgb);
      // the step of this linearisation, taken by the next launch
      a.part_icp = pic;
      a.gi = icp ? G : 0;
      a.part_rgb = t->part_rgb;
      a.gr = rgb ? G : 0;
      a.mode = t->P.mode;
      a.first_of_level = it == 0 ? 1 : 0;
      a.record = l == 0 ? 1 : 0;
      a.wrh = t->P.w_rgb_h; a.wrb = t->P.w_rgb_b; a.wih = t->P.w_icp_h; a.wib = t->P.w_icp_b;
    }
  if (i > 0)
    hipLaunchKernelGGL(k_update_into, dim3(1), dim3(256), 0, s, (const TrackState*)S[(i - 1) & 1], t->st, a,
                       numbered ? t->host_st : (HostState*)nullptr, t->solves);
  YAS_LAUNCH_CHECK();
  return YAS_OK;
}

// The solves of a device that have not ended, by tracker, as each tracker's
// host memory says.  (Asking the runtime whether another stream is idle breaks
// a capture in the global mode that any thread may have begun.)
static std::mutex g_solve_mu;
static struct {
  yas_tracker* head;
  int crowded;  // solves since two streams' overlapped, counted down from kCrowd
} g_solves[kMaxSolveDevices];
constexpr int kCrowd = 32;

static void list_solve(yas_tracker* t, yas_tracker*& head) {
  if (!t->listed) {
    t->next = head;
    head = t;
    t->listed = true;
  }
}
static void forget_solves(const yas_tracker* t) {
  std::lock_guard<std::mutex> lk(g_solve_mu);
  for (auto& d : g_solves)
    for (yas_tracker** p = &d.head; *p; p = &(*p)->next)
      if (*p == t) {
        *p = t->next;
        break;
      }
}
// Whether solves of other streams than s are there, and one-launch solves among
// them; those that have ended leave the list.
static void other_solves(yas_tracker*& head, hipStream_t s, bool& any, bool& one) {
  any = one = false;
  for (yas_tracker** p = &head; *p;) {
    yas_tracker* q = *p;
    if (__atomic_load_n(&q->host_st->ended, __ATOMIC_ACQUIRE) == q->solves) {
      *p = q->next;
      q->listed = false;
      continue;
    }
    if (q->ctx->stream != s || s == hipStreamPerThread) {  // (whose handle is not one stream)
      any = true;
      one |= q->one;
    }
    p = &q->next;
  }
}

static bool solve_fits(const yas_ctx* ctx, const void* kernel, int grid) {
  static std::mutex mu;
  static int room[kMaxSolveDevices][3];  // workgroups that fit on a CU at once, + 1; 0 = not asked yet
  int per_cu = 0;
  const int k = kernel == (const void*)k_solve<true, true> ? 0 : kernel == (const void*)k_solve<true, false> ? 1 : 2;
  std::lock_guard<std::mutex> lk(mu);
  int& r = room[ctx->device][k];
  if (r == 0) {
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kSolveThreads, 0) != hipSuccess) {
      (void)hipGetLastError();
      per_cu = 0;
    }
    r = per_cu + 1;
  }
  return grid <= (r - 1) * ctx->cus;
}

static bool is_capturing(hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &st) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return st != hipStreamCaptureStatusNone;
}

static SolveArgs solve_args(yas_tracker* t) {
  SolveArgs a;
  std::memset(&a, 0, sizeof(a));
  a.levels = t->P.levels;
  for (int l = 0; l < t->P.levels; ++l) {
    a.lv[l] = t->lv[l];
    a.tb[l] = bufs(t, l);
    a.iters[l] = t->P.iters[l];
    a.groups[l] = groups_for(t->lv[l]);
  }
  a.mode = t->P.mode;
  a.sin2_max = t->sin2_max;
  a.dist2_max = t->dist2_max;
  a.wrh = t->P.w_rgb_h; a.wrb = t->P.w_rgb_b; a.wih = t->P.w_icp_h; a.wib = t->P.w_icp_b;
  a.st = t->st;
  a.x = t->xchg;
  a.part_icp = t->part_icp; a.part_res = t->part_res; a.part_rgb = t->part_rgb;
  a.wait_ticks = t->wait_ticks;
  return a;
}
static void launch_rescue(yas_tracker* t) {
  const SolveArgs a = solve_args(t);
  HostState* h = t->host_st;
  hipStream_t s = t->ctx->stream;
  const dim3 one(1), threads(256);
  if (a.mode == YAS_TRACK_RGBD) hipLaunchKernelGGL((k_solve_rescue<true, true>), one, threads, 0, s, a, h, t->solves);
  else if (a.mode == YAS_TRACK_DEPTH)
    hipLaunchKernelGGL((k_solve_rescue<true, false>), one, threads, 0, s, a, h, t->solves);
  else hipLaunchKernelGGL((k_solve_rescue<false, true>), one, threads, 0, s, a, h, t->solves);
}

static unsigned lost_solves(const yas_tracker* t) {
  return t->lost_waited + __atomic_load_n(&t->host_st->rescued, __ATOMIC_ACQUIRE);
}
// Whether the tracker's last solves let the next one be tried as one launch.
// Its workgroups do not meet while something keeps them off a CU that nothing
// here can ask for (another process, an application's kernels), and then the
// next solve's mostly don't either.  Queued solves are found lost when their
// rescue has run.
static bool may_try(yas_tracker* t) {
  const bool ended = (int)(__atomic_load_n(&t->host_st->ended, __ATOMIC_ACQUIRE) - t->last_tried) >= 0;
  const unsigned lost = lost_solves(t);
  if (lost != t->lost_seen) {
    t->lost_seen = lost;
    if (t->tried != t->tried_seen) {  // else of the solves queued behind one found before
      t->tried_seen = t->tried;
      t->passes_left = t->passes_next;
      t->passes_next = std::min(2 * t->passes_next, kMaxPasses);
    }
  } else if (ended && t->tried != t->tried_seen) {
    t->passes_next = kFirstPasses;
  }
  if (t->passes_left == 0) return true;
  t->passes_left--;
  return false;
}

// The solve in one launch from `init` (null: the state's pose), its result to
// `host` too when not null, where it may run so (`one`, else nothing is
// launched).  Solves recorded into a graph, whose replays nothing here orders,
// may not; the others are numbered.
//
// All workgroups must find a CU at once, so no two one-launch solves run
// together.  One that takes more than half of the CUs also keeps other streams'
// kernels waiting (k_view, which needs half of a CU's LDS, above all), so while
// solves of several streams overlap they all take the passes: two cameras of
// 640x480 with both terms 3076 frames/s, four 4820; with one of the streams in
// one launch 2590 and 3830, and one camera alone 2080 against 1695 by passes.
// At 320x240 (75 workgroups) two cameras take 3850 against 3970 frames/s, but
// four that one thread enqueues 6900 against 5550.
static int solve_in_one(yas_tracker* t, const Mat44* init, HostState* host, bool& one, bool& numbered) {
  hipStream_t s = t->ctx->stream;
  const int device = t->ctx->device, mode = t->P.mode;
  int grid = 0;
  for (int l = t->P.levels - 1; l >= 0; --l)
    if (t->P.iters[l] > 0) grid = groups_for(t->lv[l]);
  one = numbered = false;
  if (grid == 0 || device >= kMaxSolveDevices || is_capturing(s)) return YAS_OK;
  const void* kernel = mode == YAS_TRACK_RGBD ? (const void*)k_solve<true, true>
                                              : mode == YAS_TRACK_DEPTH ? (const void*)k_solve<true, false>
                                                                        : (const void*)k_solve<false, true>;
  bool may = (long long)t->W * t->H <= kSolveMaxPixels && t->H <= kFastRows && solve_fits(t->ctx, kernel, grid) &&
             may_try(t);
  std::lock_guard<std::mutex> lk(g_solve_mu);
  auto& d = g_solves[device];
  bool others, other_one;
  other_solves(d.head, s, others, other_one);
  if (2 * grid <= t->ctx->cus) may &= !other_one;
  else may &= !others && d.crowded == 0;
  if (others) d.crowded = kCrowd;
  else if (d.crowded > 0) d.crowded--;
  t->solves++;
  t->one = may;
  list_solve(t, d.head);
  numbered = true;
  if (!may) return YAS_OK;
  SolveArgs a = solve_args(t);
  if (init) a.init = *init;
  a.has_init = init != nullptr;
  a.host = host;
  const dim3 threads(kSolveThreads);
  if (mode == YAS_TRACK_RGBD) hipLaunchKernelGGL((k_solve<true, true>), dim3(grid), threads, 0, s, a);
  else if (mode == YAS_TRACK_DEPTH) hipLaunchKernelGGL((k_solve<true, false>), dim3(grid), threads, 0, s, a);
  else hipLaunchKernelGGL((k_solve<false, true>), dim3(grid), threads, 0, s, a);
  YAS_LAUNCH_CHECK();
  t->tried++;
  t->last_tried = t->solves;
  one = true;
  return YAS_OK;
}

int yas_tracker_solve_async(yas_tracker* t) {
  bool one, numbered;
  int rc = solve_in_one(t, nullptr, nullptr, one, numbered);
  if (rc) return rc;
  if (!one) {
    t->by_passes++;
    return solve_by_passes(t, numbered);
  }
  launch_rescue(t);
  YAS_LAUNCH_CHECK();
  return YAS_OK;
}

// A solve from `init`, waited for; its state is left in host_st->s.  The one
// launch takes the pose as an argument and leaves its result in host memory,
// so the state's initialisation and the result's copy, 4 to 5 us each, are
// launched only where it did not run or did not complete, and then with the
// separate passes.
static int solve_and_wait(yas_tracker* t, const Mat44& init) {
  hipStream_t s = t->ctx->stream;
  t->host_st->ok = 0;
  bool one, numbered;
  int rc = solve_in_one(t, &init, t->host_st, one, numbered);
  if (rc) return rc;
  if (one) {
    YAS_HIP(hipStreamSynchronize(s));
    if (t->host_st->ok) {
      __atomic_store_n(&t->host_st->ended, t->solves, __ATOMIC_RELEASE);
      return YAS_OK;
    }
    unsigned iterations = 0;
    for (int l = 0; l < t->P.levels; ++l) iterations += t->P.iters[l] > 0 ? t->P.iters[l] : 0;
    hipLaunchKernelGGL(k_solve_skip, dim3(1), dim3(64), 0, s, t->xchg, iterations);
    t->lost_waited++;
  } else {
    t->by_passes++;
  }
  hipLaunchKernelGGL(k_track_init, dim3(1), dim3(64), 0, s, t->st, init);
  YAS_LAUNCH_CHECK();
  if ((rc = solve_by_passes(t, numbered))) return rc;
  YAS_HIP(hipMemcpyAsync(&t->host_st->s, t->st, sizeof(TrackState), hipMemcpyDeviceToHost, s));
  YAS_HIP(hipStreamSynchronize(s));
  return YAS_OK;
}

extern "C" {

int yas_tracker_set_wait_ticks(yas_tracker* t, unsigned long long ticks) {
  YAS_REQUIRE(t, "null tracker");
  t->wait_ticks = ticks;
  // the next solve is tried as if none had been lost or had overlapped another
  if (t->ctx->device < kMaxSolveDevices) {
    std::lock_guard<std::mutex> lk(g_solve_mu);
    g_solves[t->ctx->device].crowded = 0;
  }
  t->lost_seen = lost_solves(t);
  t->tried_seen = t->tried;
  t->passes_left = 0;
  t->passes_next = kFirstPasses;
  return YAS_OK;
}

int yas_tracker_solve_routes(yas_tracker* t, int routes[3]) {
  YAS_REQUIRE(t && routes, "yas_tracker_solve_routes: null argument");
  YAS_HIP(hipSetDevice(t->ctx->device));
  YAS_HIP(hipStreamSynchronize(t->ctx->stream));
  const unsigned lost = lost_solves(t);
  routes[0] = (int)(t->tried - lost);
  routes[1] = (int)lost;
  routes[2] = (int)t->by_passes;
  return YAS_OK;
}

}  // extern "C"

int yas_tracker_init_identity_async(yas_tracker* t) {
  hipLaunchKernelGGL(k_track_init_identity, dim3(1), dim3(64), 0, t->ctx->stream, t->st);
  YAS_LAUNCH_CHECK();
  return YAS_OK;
}

// Buffers and constants of this tracker, for the serving engine's batched
// kernels (which keep the buffer roles fixed and copy the current frame's
// pyramids into the reference ones instead of swapping them).
int yas_tracker_fill(yas_tracker* t, StreamDev& d) {
  YAS_REQUIRE(t->P.levels <= kTrackMaxLevels, "tracker levels");
  d.levels = t->P.levels;
  for (int l = 0; l < t->P.levels; ++l) {
    d.lv[l] = t->lv[l];
    d.tb[l] = bufs(t, l);
    d.cur_inv[l] = t->cur_inv[l];
    d.groups[l] = groups_for(t->lv[l]);
  }
  d.part_icp = t->part_icp;
  d.part_res = t->part_res;
  d.part_rgb = t->part_rgb;
  d.st = t->st;
  d.sin2_max = t->sin2_max;
  d.dist2_max = t->dist2_max;
  return YAS_OK;
}
const yas_tracker_params& yas_tracker_params_of(yas_tracker* t) { return t->P; }

// Device pointers of the solver's result (camera pose change and status).
const double* yas_tracker_result_dev(yas_tracker* t) { return t->st->last_ok; }
const int* yas_tracker_good_dev(yas_tracker* t) { return &t->st->good; }
// The state a solve starts from (the pipeline resets it in its first launch).
TrackState* yas_tracker_state_dev(yas_tracker* t) { return t->st; }

// The current frame's image and depth levels from the camera's own images,
// for the pipeline's first launch.  Levels past the third follow from
// yas_tracker_coarse_levels.
int yas_tracker_frame_args(yas_tracker* t, ImageArgs<SrcRgb>& im, DepthArgs<SrcU16>& d) {
  fill_image(im, t->lv, t->P.levels, 0, t->cur_int, t->gx, t->gy);
  fill_depth(d, t->lv, t->P.levels, t->cur_inv, t->cur_v, t->cur_p);
  return YAS_OK;
}
int yas_tracker_coarse_levels(yas_tracker* t) {
  for (int base = kImageLevels - 1; base + 1 < t->P.levels; base += kImageLevels - 1) {
    ImageArgs<SrcF32> a;
    a.src = SrcF32{t->cur_int[base], (size_t)t->lv[base].w * 4};
    fill_image(a, t->lv, t->P.levels, base, t->cur_int, t->gx, t->gy);
    hipLaunchKernelGGL(k_image_levels, dim3(a.tiles), dim3(256), 0, t->ctx->stream, a);
  }
  YAS_LAUNCH_CHECK();
  return YAS_OK;
}
// The model's levels from a ray-cast vertex map, as set_reference_model.
int yas_tracker_set_model_dev(yas_tracker* t, const float* vmap, size_t pitch) { return model_pyramid(t, vmap, pitch); }

int yas_rgb_to_gray_async(yas_ctx* ctx, const uint8_t* rgb, size_t sp, float* dst, size_t dp, int W, int H, int mode) {
  hipLaunchKernelGGL(k_rgb_to_gray, grid64x4(W, H), dim3(256), 0, ctx->stream, rgb, sp, dst, dp, W, H, mode);
  YAS_LAUNCH_CHECK();
  return YAS_OK;
}

// The largest float whose square root, rounded, is below `limit` (or equal to
// it, `inclusive`): the passes compare squares with it instead of taking two
// roots a pixel, with the same outcome.
static float largest_square(float limit, bool inclusive) {
  auto within = [&](float v) { return inclusive ? std::sqrt(v) <= limit : std::sqrt(v) < limit; };
  float v = limit * limit;
  while (within(std::nextafter(v, FLT_MAX))) v = std::nextafter(v, FLT_MAX);
  while (!within(v)) v = std::nextafter(v, 0.0f);
  return v;
}

extern "C" {

int yas_tracker_create(yas_ctx* ctx, int W, int H, const double K[4], const yas_tracker_params* P, yas_tracker** out) {
  YAS_REQUIRE(ctx && K && P && out, "yas_tracker_create: null argument");
  YAS_REQUIRE(P->levels >= 1 && P->levels <= kMaxLevels, "yas_tracker_create: levels must be 1..5");
  YAS_REQUIRE(P->mode >= 0 && P->mode <= 2, "yas_tracker_create: unknown mode");
  YAS_REQUIRE(W > 0 && H > 0 && W % (1 << (P->levels - 1)) == 0 && H % (1 << (P->levels - 1)) == 0,
              "yas_tracker_create: width and height must be divisible by 2^(levels-1)");
  YAS_REQUIRE((W >> (P->levels - 1)) >= 4 && (H >> (P->levels - 1)) >= 4,
              "yas_tracker_create: the coarsest level must be at least 4x4");
  YAS_HIP(hipSetDevice(ctx->device));
  yas_tracker* t = new yas_tracker();
  std::memset(t, 0, sizeof(*t));
  t->ctx = yas_ctx_retain(ctx);
  t->W = W;
  t->H = H;
  t->P = *P;
  // RGBDTracking.cu:432-433: sin(20 deg) computed in float, 1 cm.
  t->sin2_max = largest_square((float)std::sin(20.f * 3.14159254f / 180.f), false);
  t->dist2_max = largest_square(0.01f, true);
  t->wait_ticks = kSolveWaitTicks;
  t->passes_next = kFirstPasses;
  hipError_t e = hipSuccess;
  auto alloc = [&](void** p, size_t bytes) {
    if (e == hipSuccess) e = hipMalloc(p, bytes);
  };
  for (int l = 0; l < P->levels; ++l) {
    Level& a = t->lv[l];
    double s = (double)(1 << l);
    a.Kd[0] = K[0] / s; a.Kd[1] = K[1] / s; a.Kd[2] = K[2] / s; a.Kd[3] = K[3] / s;
    a.w = W >> l;
    a.h = H >> l;
    a.fx = (float)a.Kd[0]; a.fy = (float)a.Kd[1]; a.cx = (float)a.Kd[2]; a.cy = (float)a.Kd[3];
    a.invfx = (float)(1.0 / a.Kd[0]);
    a.invfy = (float)(1.0 / a.Kd[1]);
    a.Kinv[0] = 1.0 / a.Kd[0];
    a.Kinv[1] = 1.0 / a.Kd[1];
    a.Kinv[2] = -a.Kd[2] / a.Kd[0];
    a.Kinv[3] = -a.Kd[3] / a.Kd[1];
    size_t n = (size_t)a.w * a.h;
    for (float** p : {&t->cur_int[l], &t->ref_int[l], &t->gx[l], &t->gy[l], &t->cur_inv[l], &t->ref_inv[l]})
      alloc((void**)p, n * sizeof(float));
    for (float4** p : {&t->cur_v[l], &t->cur_n[l], &t->ref_v[l], &t->ref_n[l]}) alloc((void**)p, n * sizeof(float4));
    alloc((void**)&t->resid[l], n * sizeof(float3));
    for (float4** p : {&t->cur_p[l], &t->ref_p[l]}) alloc((void**)p, n * sizeof(IcpPoint));
  }
  alloc((void**)&t->part_icp, sizeof(float) * 32 * kRedGroups);
  alloc((void**)&t->part_icp2, sizeof(float) * 32 * kRedGroups);
  alloc((void**)&t->part_res, sizeof(float) * 4 * kRedGroups);
  alloc((void**)&t->part_rgb, sizeof(float) * 32 * kRedGroups);
  alloc((void**)&t->st, sizeof(TrackState));
  alloc((void**)&t->st2, sizeof(TrackState));
  alloc((void**)&t->xchg, sizeof(SolveXchg));
  if (e == hipSuccess) e = hipHostMalloc((void**)&t->host_st, sizeof(HostState), hipHostMallocDefault);
  if (e != hipSuccess) {
    yas_set_error("yas_tracker_create: %s", hipGetErrorString(e));
    yas_tracker_destroy(t);
    return YAS_E_HIP;
  }
  // zeroed images, zeroed state (tickets armed)
  for (int l = 0; l < P->levels; ++l) {
    size_t n = (size_t)t->lv[l].w * t->lv[l].h;
    for (float* p : {t->cur_int[l], t->ref_int[l], t->gx[l], t->gy[l], t->cur_inv[l], t->ref_inv[l]})
      YAS_HIP(hipMemsetAsync(p, 0, n * sizeof(float), ctx->stream));
    for (float4* p : {t->cur_v[l], t->cur_n[l], t->ref_v[l], t->ref_n[l]})
      YAS_HIP(hipMemsetAsync(p, 0, n * sizeof(float4), ctx->stream));
    YAS_HIP(hipMemsetAsync(t->resid[l], 0, n * sizeof(float3), ctx->stream));
    for (float4* p : {t->cur_p[l], t->ref_p[l]}) YAS_HIP(hipMemsetAsync(p, 0, n * sizeof(IcpPoint), ctx->stream));
  }
  YAS_HIP(hipMemsetAsync(t->st, 0, sizeof(TrackState), ctx->stream));
  YAS_HIP(hipMemsetAsync(t->st2, 0, sizeof(TrackState), ctx->stream));
  YAS_HIP(hipMemsetAsync(t->xchg, 0, sizeof(SolveXchg), ctx->stream));
  std::memset(t->host_st, 0, sizeof(HostState));
  int rc = yas_tracker_init_identity_async(t);
  if (rc) {
    yas_tracker_destroy(t);
    return rc;
  }
  *out = t;
  return YAS_OK;
}

int yas_tracker_destroy(yas_tracker* t) {
  if (!t) return YAS_OK;
  hipSetDevice(t->ctx->device);
  hipStreamSynchronize(t->ctx->stream);
  forget_solves(t);
  for (int l = 0; l < kMaxLevels; ++l) {
    for (float* p : {t->cur_int[l], t->ref_int[l], t->gx[l], t->gy[l], t->cur_inv[l], t->ref_inv[l]}) hipFree(p);
    for (float4* p : {t->cur_v[l], t->cur_n[l], t->ref_v[l], t->ref_n[l]}) hipFree(p);
    hipFree(t->resid[l]);
    for (float4* p : {t->cur_p[l], t->ref_p[l]}) hipFree(p);
  }
  hipFree(t->part_icp);
  hipFree(t->part_icp2);
  hipFree(t->part_res);
  hipFree(t->part_rgb);
  hipFree(t->st);
  hipFree(t->st2);
  hipFree(t->xchg);
  hipFree(t->raw_depth);
  hipFree(t->raw_image);
  if (t->host_st) hipHostFree(t->host_st);
  yas_ctx_release(t->ctx);
  delete t;
  return YAS_OK;
}

int yas_tracker_set_reference_image(yas_tracker* t, const float* g, size_t pitch) {
  YAS_REQUIRE(t && g && pitch >= (size_t)t->W * 4, "yas_tracker_set_reference_image: bad argument");
  return image_pyramid(t, g, pitch, t->ref_int, false);
}
int yas_tracker_set_tracking_image(yas_tracker* t, const float* g, size_t pitch) {
  YAS_REQUIRE(t && g && pitch >= (size_t)t->W * 4, "yas_tracker_set_tracking_image: bad argument");
  return image_pyramid(t, g, pitch, t->cur_int, true);
}
int yas_tracker_set_reference_depth(yas_tracker* t, const float* d, size_t pitch) {
  YAS_REQUIRE(t && d && pitch >= (size_t)t->W * 4, "yas_tracker_set_reference_depth: bad argument");
  return depth_pyramid(t, d, pitch, t->ref_inv, t->ref_v, t->ref_p);
}
int yas_tracker_set_tracking_depth(yas_tracker* t, const float* d, size_t pitch) {
  YAS_REQUIRE(t && d && pitch >= (size_t)t->W * 4, "yas_tracker_set_tracking_depth: bad argument");
  return depth_pyramid(t, d, pitch, t->cur_inv, t->cur_v, t->cur_p);
}
// Host images (RGBDTracking.h:17-21 take cv::Mat): the reference converts an
// 8-bit gray image to float on the host and uploads it (RGBDTracking.cu:68-
// 71,104-107), and uploads float depth into one raw-depth buffer
// (mGpuBufferRawDepth, RGBDTracking.cu:86-87,122-123) that
// GetReferenceDepth returns.  The copy waits for the stream, so the host
// buffer may be reused when the call returns.
static int upload_host(yas_tracker* t, float** dst, const void* src, size_t pitch, bool gray_u8) {
  YAS_HIP(hipSetDevice(t->ctx->device));
  const size_t row = (size_t)t->W * sizeof(float);
  if (!*dst) YAS_HIP(hipMalloc((void**)dst, row * t->H));
  std::vector<float> conv;
  const void* from = src;
  size_t from_pitch = pitch;
  if (gray_u8) {
    conv.resize((size_t)t->W * t->H);
    for (int y = 0; y < t->H; ++y) {
      const uint8_t* r = (const uint8_t*)src + (size_t)y * pitch;
      for (int x = 0; x < t->W; ++x) conv[(size_t)y * t->W + x] = (float)r[x];
    }
    from = conv.data();
    from_pitch = row;
  }
  YAS_HIP(hipMemcpy2DAsync(*dst, row, from, from_pitch, row, t->H, hipMemcpyHostToDevice, t->ctx->stream));
  YAS_HIP(hipStreamSynchronize(t->ctx->stream));
  return YAS_OK;
}

int yas_tracker_set_reference_image_host(yas_tracker* t, const uint8_t* g, size_t pitch) {
  YAS_REQUIRE(t && g && pitch >= (size_t)t->W, "yas_tracker_set_reference_image_host: bad argument");
  int rc = upload_host(t, &t->raw_image, g, pitch, true);
  return rc ? rc : image_pyramid(t, t->raw_image, (size_t)t->W * 4, t->ref_int, false);
}
int yas_tracker_set_tracking_image_host(yas_tracker* t, const uint8_t* g, size_t pitch) {
  YAS_REQUIRE(t && g && pitch >= (size_t)t->W, "yas_tracker_set_tracking_image_host: bad argument");
  int rc = upload_host(t, &t->raw_image, g, pitch, true);
  return rc ? rc : image_pyramid(t, t->raw_image, (size_t)t->W * 4, t->cur_int, true);
}
int yas_tracker_set_reference_depth_host(yas_tracker* t, const float* d, size_t pitch) {
  YAS_REQUIRE(t && d && pitch >= (size_t)t->W * 4, "yas_tracker_set_reference_depth_host: bad argument");
  int rc = upload_host(t, &t->raw_depth, d, pitch, false);
  return rc ? rc : depth_pyramid(t, t->raw_depth, (size_t)t->W * 4, t->ref_inv, t->ref_v, t->ref_p);
}
int yas_tracker_set_tracking_depth_host(yas_tracker* t, const float* d, size_t pitch) {
  YAS_REQUIRE(t && d && pitch >= (size_t)t->W * 4, "yas_tracker_set_tracking_depth_host: bad argument");
  int rc = upload_host(t, &t->raw_depth, d, pitch, false);
  return rc ? rc : depth_pyramid(t, t->raw_depth, (size_t)t->W * 4, t->cur_inv, t->cur_v, t->cur_p);
}

// GetReferenceDepth (RGBDTracking.cu:547-550) returns the raw-depth buffer,
// i.e. the depth most recently uploaded from the host (NULL before any).
int yas_tracker_raw_depth(yas_tracker* t, float** depth, size_t* pitch) {
  YAS_REQUIRE(t && depth && pitch, "yas_tracker_raw_depth: null argument");
  *depth = t->raw_depth;
  *pitch = (size_t)t->W * sizeof(float);
  return YAS_OK;
}

// WriteDebugImages (RGBDTracking.cu:557-568): the level-0 current and
// reference intensity and the two gradient images, as 8-bit binary PGM
// files curr_image.pgm, last_image.pgm, gx.pgm, gy.pgm in `dir` (values
// rounded to nearest and clamped to [0, 255]).
int yas_tracker_write_debug_images(yas_tracker* t, const char* dir) {
  YAS_REQUIRE(t && dir, "yas_tracker_write_debug_images: null argument");
  YAS_HIP(hipSetDevice(t->ctx->device));
  YAS_HIP(hipStreamSynchronize(t->ctx->stream));
  const size_t n = (size_t)t->W * t->H;
  const struct {
    const char* name;
    const float* img;
  } out[4] = {{"curr_image.pgm", t->cur_int[0]}, {"last_image.pgm", t->ref_int[0]}, {"gx.pgm", t->gx[0]},
              {"gy.pgm", t->gy[0]}};
  std::vector<float> f(n);
  std::vector<unsigned char> b(n);
  for (const auto& o : out) {
    YAS_HIP(hipMemcpy(f.data(), o.img, n * sizeof(float), hipMemcpyDeviceToHost));
    for (size_t i = 0; i < n; ++i) {
      float v = std::nearbyint(f[i]);
      b[i] = (unsigned char)(v != v ? 0.f : std::min(255.f, std::max(0.f, v)));
    }
    std::string path = std::string(dir) + "/" + o.name;
    FILE* fp = std::fopen(path.c_str(), "wb");
    if (!fp) {
      yas_set_error("yas_tracker_write_debug_images: cannot open %s", path.c_str());
      return YAS_E_INVALID;
    }
    std::fprintf(fp, "P5\n%d %d\n255\n", t->W, t->H);
    bool ok = std::fwrite(b.data(), 1, n, fp) == n;
    ok = (std::fclose(fp) == 0) && ok;
    if (!ok) {
      yas_set_error("yas_tracker_write_debug_images: write to %s failed", path.c_str());
      return YAS_E_INVALID;
    }
  }
  return YAS_OK;
}

int yas_tracker_set_reference_model(yas_tracker* t, const float* vmap, size_t pitch) {
  YAS_REQUIRE(t && vmap && pitch >= (size_t)t->W * 16, "yas_tracker_set_reference_model: bad argument");
  return model_pyramid(t, vmap, pitch);
}

}  // extern "C"

// After yas_tracker_swap_frame_buffer: the copies that restore the previous
// reference intensity and inverse depth (the buffers now named current).
int yas_tracker_unswap_copies(yas_tracker* t, RefRestore& r) {
  r.count = 0;
  for (int l = 0; l < t->P.levels; ++l) {
    const int n = t->lv[l].w * t->lv[l].h;
    r.dst[r.count] = t->ref_int[l]; r.src[r.count] = t->cur_int[l]; r.n[r.count++] = n;
    r.dst[r.count] = t->ref_inv[l]; r.src[r.count] = t->cur_inv[l]; r.n[r.count++] = n;
  }
  return YAS_OK;
}

extern "C" {

int yas_tracker_swap_frame_buffer(yas_tracker* t) {
  YAS_REQUIRE(t, "null tracker");
  for (int l = 0; l < kMaxLevels; ++l) {
    std::swap(t->ref_v[l], t->cur_v[l]);
    std::swap(t->ref_p[l], t->cur_p[l]);
    std::swap(t->ref_inv[l], t->cur_inv[l]);
    std::swap(t->ref_int[l], t->cur_int[l]);
  }
  return YAS_OK;
}

int yas_tracker_get_transform(yas_tracker* t, const double init[16], int swap, double out[16], yas_track_stats* stats) {
  YAS_REQUIRE(t && out, "yas_tracker_get_transform: null argument");
  YAS_HIP(hipSetDevice(t->ctx->device));
  Mat44 M;
  if (init) std::memcpy(M.m, init, sizeof(M.m));
  else
    for (int i = 0; i < 16; ++i) M.m[i] = (i % 5 == 0) ? 1.0 : 0.0;
  int rc = solve_and_wait(t, M);
  if (rc) return rc;
  const TrackState& h = t->host_st->s;
  // RGBDTracking.cu:187-191: a NaN update returns before the buffer swap
  if (swap && h.good) yas_tracker_swap_frame_buffer(t);
  if (h.good) std::memcpy(out, h.last_ok, sizeof(h.last_ok));
  else
    for (int i = 0; i < 16; ++i) out[i] = (i % 5 == 0) ? 1.0 : 0.0;
  if (stats) {
    stats->good = h.good;
    stats->icp_inliers = h.icp_inliers;
    stats->rgb_inliers = h.rgb_inliers;
    stats->last_error = h.last_err;
  }
  return h.good ? YAS_OK : YAS_E_DIVERGED;
}

int yas_tracker_is_tracking_good(yas_tracker* t, int* good) {
  YAS_REQUIRE(t && good, "null argument");
  YAS_HIP(hipMemcpyAsync(&t->host_st->s, t->st, sizeof(TrackState), hipMemcpyDeviceToHost, t->ctx->stream));
  YAS_HIP(hipStreamSynchronize(t->ctx->stream));
  *good = t->host_st->s.good;
  return YAS_OK;
}

int yas_tracker_step_sums(yas_tracker* t, int level, const double T[16], int kind, float out[29], float stats[4]) {
  YAS_REQUIRE(t && T && out, "yas_tracker_step_sums: null argument");
  YAS_REQUIRE(level >= 0 && level < t->P.levels, "yas_tracker_step_sums: bad level");
  YAS_HIP(hipSetDevice(t->ctx->device));
  Mat44 M;
  std::memcpy(M.m, T, sizeof(M.m));
  hipLaunchKernelGGL(k_track_init, dim3(1), dim3(64), 0, t->ctx->stream, t->st, M);
  int rc = launch_iteration(t, level, kind == 0, kind != 0, false, false);
  if (rc) return rc;
  YAS_HIP(hipMemcpyAsync(&t->host_st->s, t->st, sizeof(TrackState), hipMemcpyDeviceToHost, t->ctx->stream));
  YAS_HIP(hipStreamSynchronize(t->ctx->stream));
  const float* s = kind == 0 ? t->host_st->s.sums_icp : t->host_st->s.sums_rgb;
  std::memcpy(out, s, sizeof(float) * 29);
  if (stats) std::memcpy(stats, t->host_st->s.rgb_stats, sizeof(float) * 4);
  return YAS_OK;
}

namespace {
// One wavefront per system: the Gauss-Newton step's 6x6 solve as the
// tracker's kernels run it (ldlt_solve6_wave), for yas_tracker_solve6.
__global__ void __launch_bounds__(64) k_solve6(const float* H, const float* b, double* x) {
  __shared__ float sH[36], sb[6];
  __shared__ double sx[6];
  const size_t s = blockIdx.x;
  const int lane = threadIdx.x;
  if (lane < 36) sH[lane] = H[s * 36 + lane];
  if (lane < 6) sb[lane] = b[s * 6 + lane];
  wave_lds_sync();
  double xi[6];
  ldlt_solve6_wave(sH, sb, sx, xi);
  if (lane == 0) {
#pragma unroll
    for (int i = 0; i < 6; ++i) x[s * 6 + i] = xi[i];
  }
}
}  // namespace

int yas_tracker_solve6(yas_ctx* ctx, const float* H, const float* b, double* x, int n) {
  YAS_REQUIRE(ctx && H && b && x, "yas_tracker_solve6: null argument");
  YAS_REQUIRE(n >= 1 && n <= (1 << 20), "yas_tracker_solve6: n must be 1..2^20");
  YAS_HIP(hipSetDevice(ctx->device));
  const size_t nh = (size_t)n * 36 * sizeof(float), nb = (size_t)n * 6 * sizeof(float), nx = (size_t)n * 6 * sizeof(double);
  char* buf = nullptr;
  YAS_HIP(hipMalloc((void**)&buf, nh + nb + nx));
  float* dH = (float*)buf;
  float* db = (float*)(buf + nh);
  double* dx = (double*)(buf + nh + nb);
  hipStream_t s = ctx->stream;
  hipError_t e = hipMemcpyAsync(dH, H, nh, hipMemcpyHostToDevice, s);
  if (e == hipSuccess) e = hipMemcpyAsync(db, b, nb, hipMemcpyHostToDevice, s);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_solve6, dim3(n), dim3(64), 0, s, dH, db, dx);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpyAsync(x, dx, nx, hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  else hipStreamSynchronize(s);
  hipFree(buf);
  YAS_HIP(e);
  return YAS_OK;
}

int yas_tracker_level(yas_tracker* t, int which, int level, void** ptr, size_t* pitch, int* w, int* h) {
  YAS_REQUIRE(t && ptr, "null argument");
  YAS_REQUIRE(level >= 0 && level < t->P.levels, "bad level");
  const Level& a = t->lv[level];
  void* one[6] = {t->cur_int[level], t->ref_int[level], t->gx[level], t->gy[level], t->cur_inv[level], t->ref_inv[level]};
  void* vec[5] = {t->cur_v[level], t->cur_n[level], t->ref_v[level], t->ref_n[level], t->resid[level]};
  YAS_REQUIRE(which >= 0 && which < 11, "bad buffer id");
  if (which == 7 || which == 9) {
    // The passes read vertex and normal as ICP points; the float4 normal
    // map is formed here from the vertex map, as the pyramid kernels would.
    YAS_HIP(hipSetDevice(t->ctx->device));
    hipLaunchKernelGGL(k_normal, grid64x4(a.w, a.h), dim3(256), 0, t->ctx->stream,
                       which == 7 ? t->cur_v[level] : t->ref_v[level], (size_t)a.w * 16,
                       which == 7 ? t->cur_n[level] : t->ref_n[level], (size_t)a.w * 16, a.w, a.h);
    YAS_LAUNCH_CHECK();
    YAS_HIP(hipStreamSynchronize(t->ctx->stream));
  }
  *ptr = which < 6 ? one[which] : vec[which - 6];
  if (pitch) *pitch = (size_t)a.w * (which < 6 ? 4 : which < 10 ? 16 : 12);
  if (w) *w = a.w;
  if (h) *h = a.h;
  return YAS_OK;
}

int yas_rgb_to_intensity(yas_ctx* ctx, const uint8_t* rgb, size_t sp, float* dst, size_t dp, int W, int H, int mode) {
  YAS_REQUIRE(ctx && rgb && dst && W > 0 && H > 0, "yas_rgb_to_intensity: bad argument");
  return yas_rgb_to_gray_async(ctx, rgb, sp, dst, dp, W, H, mode);
}
int yas_depth_to_invdepth(yas_ctx* ctx, const float* d, size_t sp, float* inv, size_t dp, int W, int H) {
  YAS_REQUIRE(ctx && d && inv && W > 0 && H > 0, "bad argument");
  hipLaunchKernelGGL(k_invdepth, grid64x4(W, H), dim3(256), 0, ctx->stream, d, sp, inv, dp, W, H);
  YAS_LAUNCH_CHECK();
  return YAS_OK;
}
int yas_pyrdown_depth(yas_ctx* ctx, const float* s, size_t sp, float* d, size_t dp, int W, int H) {
  YAS_REQUIRE(ctx && s && d && W > 0 && H > 0, "bad argument");
  hipLaunchKernelGGL(k_pyrdown_depth, grid64x4(W, H), dim3(256), 0, ctx->stream, s, sp, d, dp, W, H);
  YAS_LAUNCH_CHECK();
  return YAS_OK;
}
int yas_pyrdown_gauss(yas_ctx* ctx, const float* s, size_t sp, int sw, int sh, float* d, size_t dp) {
  YAS_REQUIRE(ctx && s && d && sw >= 4 && sh >= 4, "yas_pyrdown_gauss: source must be at least 4x4");
  int dw = sw / 2, dh = sh / 2;
  hipLaunchKernelGGL(k_pyrdown_gauss, dim3((dw + 15) / 16, (dh + 15) / 16), dim3(256), 0, ctx->stream, s, sp, sw, sh, d,
                     dp, dw, dh);
  YAS_LAUNCH_CHECK();
  return YAS_OK;
}
int yas_compute_vertex_map(yas_ctx* ctx, const float* inv, size_t sp, float* v, size_t dp, int W, int H, const float K[4],
                           float cutoff) {
  YAS_REQUIRE(ctx && inv && v && K && W > 0 && H > 0, "bad argument");
  Intr k = make_intr(K);
  hipLaunchKernelGGL(k_vertex, grid64x4(W, H), dim3(256), 0, ctx->stream, inv, sp, (float4*)v, dp, W, H, k.invfx,
                     k.invfy, k.cx, k.cy, cutoff);
  YAS_LAUNCH_CHECK();
  return YAS_OK;
}
int yas_compute_normal_map(yas_ctx* ctx, const float* v, size_t sp, float* n, size_t dp, int W, int H) {
  YAS_REQUIRE(ctx && v && n && W > 0 && H > 0, "bad argument");
  hipLaunchKernelGGL(k_normal, grid64x4(W, H), dim3(256), 0, ctx->stream, (const float4*)v, sp, (float4*)n, dp, W, H);
  YAS_LAUNCH_CHECK();
  return YAS_OK;
}
int yas_image_gradient(yas_ctx* ctx, const float* s, size_t sp, float* gx, float* gy, size_t dp, int W, int H) {
  YAS_REQUIRE(ctx && s && gx && gy && W > 0 && H > 0, "bad argument");
  hipLaunchKernelGGL(k_gradient, grid64x4(W, H), dim3(256), 0, ctx->stream, s, sp, gx, gy, dp, W, H);
  YAS_LAUNCH_CHECK();
  return YAS_OK;
}
int yas_vmap_to_depth(yas_ctx* ctx, const float* v, size_t sp, float* d, size_t dp, int W, int H) {
  YAS_REQUIRE(ctx && v && d && W > 0 && H > 0, "bad argument");
  hipLaunchKernelGGL(k_vmap_to_depth, grid64x4(W, H), dim3(256), 0, ctx->stream, (const float4*)v, sp, d, dp, W, H);
  YAS_LAUNCH_CHECK();
  return YAS_OK;
}

}  // extern "C"
