// Ray casting of a TSDF volume into a camera-frame vertex map: the
// reference's RayTraceEngine (RGBDFusion/src/RayTraceEngine.cu:11-454).
//
// The kernels' bodies are in yas_raycast_dev.hpp.
#include <cstring>
#include <mutex>

#include "yas_internal.hpp"
#include "yas_raycast_dev.hpp"
#include "yas_server_dev.hpp"

using namespace yas;

MapView yas_map_view(yas_map* map);
const PosePair* yas_map_pose_dev(yas_map* map);
Intr yas_map_intr(yas_map* map);
yas_ctx* yas_map_ctx(yas_map* map);
int yas_map_visible_async(yas_map* map, const double T[16], int W, int H);
int yas_map_visible_prepared(yas_map* map, int W, int H);

struct yas_raycaster {
  yas_ctx* ctx;
  int W, H, cols, rows;
  Intr K;
  float4* vmap;
  unsigned* zmin;
  unsigned* zmax;
  unsigned* occ;  // coarse occupancy of the map cast last
  int* host_ctr;
  yas_map* last_map;
  float* depth;  // VMapToDepth of the last vertex map (lazily allocated)
};

// The cells and the occupancy before a ray cast, and the map's visible counter.
__global__ void __launch_bounds__(256) k_cells_init(unsigned* zmin, unsigned* zmax, int n, unsigned* occ, int* ctr) {
  zrange_init_at(zmin, zmax, n, blockIdx.x, gridDim.x);
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < kOccWords; i += gridDim.x * blockDim.x) occ[i] = 0u;
  if (blockIdx.x == 0 && threadIdx.x == 0) ctr[kCtrVisible] = 0;
}

// Visibility and z-range cells (view_scan).  Workgroup b: slice b / chunks of
// the block list, chunk b % chunks of the cell rows (rows_per each).  A slice
// has a few hundred blocks at most; the threads are for the cells, cleared and
// merged (1280x960: 14.7 us with 256, 11.9 us with 1024).
template <class P>
__global__ void __launch_bounds__(1024) k_view(MapView m, P pose, Intr Kmap, Intr K, int W, int H, int cols, int rows,
                                              unsigned* zmin, unsigned* zmax, unsigned* occ, int slices, int chunks,
                                              int rows_per) {
  extern __shared__ unsigned lz[];
  const int chunk = blockIdx.x % chunks, r0 = chunk * rows_per;
  view_scan(m, pose.Tinv(), Kmap, K, W, H, cols, rows, zmin, zmax, occ, lz, blockIdx.x / chunks, slices, r0,
            min(rows, r0 + rows_per), chunk == 0);
}

// The cells of an image too wide for k_view's chunks, straight into memory
// (after the map's visibility pass), and the occupancy.
__global__ void __launch_bounds__(256) k_zrange(MapView m, const PosePair* pose, Intr K, int cols, int rows,
                                                unsigned* zmin, unsigned* zmax, unsigned* occ) {
  zrange_at(m, pose, K, cols, rows, zmin, zmax, blockIdx.x, gridDim.x);
  occ_scan_at(m, occ, blockIdx.x, gridDim.x);
}

template <class VT, class P>
__global__ void __launch_bounds__(256) k_march(MapView m, P pose, Intr K, int W, int H, int cols, const float* zmin,
                                               const float* zmax, const unsigned* occ, float4* vmap, float vsinv,
                                               float step_scale, int rows) {
  march_at<VT>(m, pose.T(), pose.Tinv(), K, W, H, cols, zmin, zmax, occ, vmap, vsinv, step_scale, rows, blockIdx.x);
}

// Visibility and z-range cells, then the march (RayTraceEngine.cu:412-450):
// cells zmin/zmax of (W/8)*(H/8), vertex map `vmap` dense W*H float4.  The
// pose is T's, or with T null the map's pose pair on the device; the map's
// visible counter and the cells have been reset on this stream.
template <class P>
static int launch_view_march(hipStream_t s, yas_map* map, const P& pose, const double* T, const Intr& K, int W, int H,
                             unsigned* zmin, unsigned* zmax, unsigned* occ, float4* vmap, hipEvent_t before_march,
                             const hipEvent_t* march_ev) {
  MapView v = yas_map_view(map);
  const int cols = W / 8, rows = H / 8, cus = yas_map_ctx(map)->cus;
  if (cols <= kViewCells) {
    // equal chunks of whole cell rows; the block list in slices, one
    // workgroup a CU in all
    const int most = kViewCells / cols, chunks = (rows + most - 1) / most, rows_per = (rows + chunks - 1) / chunks;
    const int slices = chunks < cus ? cus / chunks : 1;
    hipLaunchKernelGGL(k_view<P>, dim3(slices * chunks), dim3(1024),
                       sizeof(unsigned) * (kOccWords + 2 * (size_t)rows_per * cols), s, v, pose, yas_map_intr(map), K, W, H,
                       cols, rows, zmin, zmax, occ, slices, chunks, rows_per);
  } else {
    int r = T ? yas_map_visible_async(map, T, W, H) : yas_map_visible_prepared(map, W, H);
    if (r) return r;
    int g = (v.num_blocks + 255) / 256;
    if (g > 2048) g = 2048;
    hipLaunchKernelGGL(k_zrange, dim3(g), dim3(256), 0, s, v, yas_map_pose_dev(map), K, cols, rows, zmin, zmax, occ);
  }
  YAS_LAUNCH_CHECK();
  if (before_march) YAS_HIP(hipEventRecord(before_march, s));
  const float vsinv = (float)(1.0 / (double)v.voxel_size);
  const float step_scale = v.trunc / v.voxel_size;
  const int mr = march_rows(W, H, cus);
  dim3 grid(march_tiles(W, H, mr));
  const float* zn = (const float*)zmin;
  const float* zf = (const float*)zmax;
  switch (v.format) {
    case YAS_VOXEL_I16_U8:
      launch_timed(k_march<VoxI16, P>, grid, dim3(256), s, march_ev, v, pose, K, W, H, cols, zn, zf, occ, vmap, vsinv,
                   step_scale, mr);
      break;
    case YAS_VOXEL_F16_U16:
      launch_timed(k_march<VoxF16, P>, grid, dim3(256), s, march_ev, v, pose, K, W, H, cols, zn, zf, occ, vmap, vsinv,
                   step_scale, mr);
      break;
    default:
      launch_timed(k_march<VoxF32, P>, grid, dim3(256), s, march_ev, v, pose, K, W, H, cols, zn, zf, occ, vmap, vsinv,
                   step_scale, mr);
  }
  YAS_LAUNCH_CHECK();
  return YAS_OK;
}

// A whole ray cast at pose T: the cells and the visible counter reset, then
// launch_view_march.
static int launch_raycast_to(yas_map* map, const double T[16], const Intr& K, int W, int H, unsigned* zmin,
                             unsigned* zmax, unsigned* occ, float4* vmap) {
  hipStream_t s = yas_map_ctx(map)->stream;
  const int ncell = (W / 8) * (H / 8);
  hipLaunchKernelGGL(k_cells_init, dim3((ncell + 255) / 256), dim3(256), 0, s, zmin, zmax, ncell, occ,
                     yas_map_view(map).ctr);
  YAS_LAUNCH_CHECK();
  PoseVal pose;
  pose_pair_from(T, pose.p);
  return launch_view_march(s, map, pose, T, K, W, H, zmin, zmax, occ, vmap, nullptr, nullptr);
}

// ------------------------------------------------------------------ ray cast without allocation
// yas_raycast_into keeps its only scratch, the two z-range maps and the coarse
// occupancy, in this file-scope device array: zmin in the first kScratchCells
// words, zmax in the next, then the occupancy (260 KiB, held on every device
// the library runs on until the process ends).  The kernels get its device
// address, looked up once per device with that device current; the array's
// name itself is a host-side stand-in and is never passed to a kernel.
constexpr int kScratchCells = 32768;
static __device__ __align__(256) unsigned scratch[2 * kScratchCells + kOccWords];

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static unsigned* g_scratch_dev[kMaxDevices];

static int scratch_on_device(int device, unsigned** out) {
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  YAS_REQUIRE(device >= 0 && device < kMaxDevices, "yas_raycast_into: device index out of range");
  if (!g_scratch_dev[device]) {
    void* p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      yas_set_error("yas_raycast_into: hipGetSymbolAddress(scratch) failed: %s", hipGetErrorString(e));
      return YAS_E_HIP;
    }
    g_scratch_dev[device] = (unsigned*)p;
  }
  *out = g_scratch_dev[device];
  return YAS_OK;
}

// Ray cast whose set-up the caller has already enqueued on this stream: the
// map's pose pair written, its visible counter cleared and this ray caster's
// cells reset (the pipeline does all three in its first launch).
// `before_march` (optional) is recorded between the view and march kernels.
int yas_raycast_prepared(yas_raycaster* rc, yas_map* map, hipEvent_t before_march, const hipEvent_t* march_ev) {
  int r = launch_view_march(rc->ctx->stream, map, PoseDev{yas_map_pose_dev(map)}, (const double*)nullptr, rc->K, rc->W,
                            rc->H, rc->zmin, rc->zmax, rc->occ, rc->vmap, before_march, march_ev);
  if (r) return r;
  rc->last_map = map;
  return YAS_OK;
}

float4* yas_raycaster_vmap_dev(yas_raycaster* rc) { return rc->vmap; }
void yas_raycaster_zrange_dev(yas_raycaster* rc, unsigned** zmin, unsigned** zmax, unsigned** occ, int* ncell) {
  *occ = rc->occ;
  *zmin = rc->zmin;
  *zmax = rc->zmax;
  *ncell = rc->cols * rc->rows;
}

// Buffers and launch constants of this ray caster for the serving engine.
int yas_raycaster_fill(yas_raycaster* rc, const MapView& v, StreamDev& d) {
  d.cols = rc->cols;
  d.rows = rc->rows;
  d.zmin = rc->zmin;
  d.zmax = rc->zmax;
  d.vmap = rc->vmap;
  d.vsinv = (float)(1.0 / (double)v.voxel_size);
  d.step_scale = v.trunc / v.voxel_size;
  int g = (v.num_blocks + 255) / 256;
  d.zr_groups = g > 2048 ? 2048 : g;
  return YAS_OK;
}

extern "C" {

int yas_raycaster_create(yas_ctx* ctx, int W, int H, const float K[4], yas_raycaster** out) {
  YAS_REQUIRE(ctx && K && out, "yas_raycaster_create: null argument");
  YAS_REQUIRE(W >= 8 && H >= 8, "yas_raycaster_create: image too small");
  YAS_REQUIRE(W % 8 == 0 && H % 8 == 0, "yas_raycaster_create: width and height must be multiples of 8");
  YAS_HIP(hipSetDevice(ctx->device));
  yas_raycaster* rc = new yas_raycaster();
  rc->ctx = yas_ctx_retain(ctx);
  rc->W = W;
  rc->H = H;
  rc->cols = W / 8;
  rc->rows = H / 8;
  rc->K = make_intr(K);
  hipError_t e = hipMalloc((void**)&rc->vmap, sizeof(float4) * (size_t)W * H);
  if (e == hipSuccess) e = hipMalloc((void**)&rc->zmin, sizeof(unsigned) * rc->cols * rc->rows);
  if (e == hipSuccess) e = hipMalloc((void**)&rc->zmax, sizeof(unsigned) * rc->cols * rc->rows);
  if (e == hipSuccess) e = hipMalloc((void**)&rc->occ, sizeof(unsigned) * kOccWords);
  if (e == hipSuccess) e = hipHostMalloc((void**)&rc->host_ctr, sizeof(int) * kCtrCount, hipHostMallocDefault);
  if (e != hipSuccess) {
    yas_set_error("yas_raycaster_create: %s", hipGetErrorString(e));
    yas_raycaster_destroy(rc);
    return YAS_E_HIP;
  }
  // nothing traced yet: every pixel invalid
  YAS_HIP(hipMemsetAsync(rc->vmap, 0, sizeof(float4) * (size_t)W * H, ctx->stream));
  *out = rc;
  return YAS_OK;
}

int yas_raycaster_destroy(yas_raycaster* rc) {
  if (!rc) return YAS_OK;
  hipSetDevice(rc->ctx->device);
  hipStreamSynchronize(rc->ctx->stream);
  hipFree(rc->vmap);
  hipFree(rc->zmin);
  hipFree(rc->zmax);
  hipFree(rc->occ);
  hipFree(rc->depth);
  if (rc->host_ctr) hipHostFree(rc->host_ctr);
  yas_ctx_release(rc->ctx);
  delete rc;
  return YAS_OK;
}

int yas_raycast(yas_raycaster* rc, yas_map* map, const double T[16]) {
  YAS_REQUIRE(rc && map && T, "yas_raycast: null argument");
  YAS_REQUIRE_ACTIVE(map);
  YAS_HIP(hipSetDevice(rc->ctx->device));
  YAS_REQUIRE(yas_map_ctx(map)->stream == rc->ctx->stream, "yas_raycast: map and ray caster must share a stream");
  int r = launch_raycast_to(map, T, rc->K, rc->W, rc->H, rc->zmin, rc->zmax, rc->occ, rc->vmap);
  if (r) return r;
  rc->last_map = map;
  return YAS_OK;
}

int yas_raycast_into(yas_map* map, const double T[16], const float K[4], int W, int H, float* vmap, size_t pitch) {
  YAS_REQUIRE(map && T && K && vmap, "yas_raycast_into: null argument");
  YAS_REQUIRE(W >= 8 && H >= 8 && W % 8 == 0 && H % 8 == 0,
              "yas_raycast_into: width and height must be multiples of 8");
  YAS_REQUIRE((long long)(W / 8) * (H / 8) <= kScratchCells,
              "yas_raycast_into: image exceeds the 32768 z-range cells of the scratch array "
              "((width/8)*(height/8); e.g. 1280x960 fits, 2048x1152 does not)");
  YAS_REQUIRE(pitch == sizeof(float4) * (size_t)W, "yas_raycast_into: the vertex map must be dense (pitch = 16 * width)");
  YAS_REQUIRE_ACTIVE(map);
  yas_ctx* ctx = yas_map_ctx(map);
  YAS_HIP(hipSetDevice(ctx->device));
  unsigned* zr = nullptr;
  int r = scratch_on_device(ctx->device, &zr);
  if (r) return r;
  return launch_raycast_to(map, T, make_intr(K), W, H, zr, zr + kScratchCells, zr + 2 * kScratchCells,
                            (float4*)vmap);
}

int yas_raycaster_vmap(yas_raycaster* rc, float** vmap, size_t* pitch) {
  YAS_REQUIRE(rc && vmap, "null argument");
  *vmap = (float*)rc->vmap;
  if (pitch) *pitch = sizeof(float4) * (size_t)rc->W;
  return YAS_OK;
}

// GetRayTracingResultDepth (VoxelMap.cu:981-987): VMapToDepth
// (ImageProc.cu:262-285) of the last vertex map into the ray caster's depth
// image (overwritten by the next call; the reference returns a new GpuMat).
// With a host buffer the image is also copied there and the call waits.
int yas_raycaster_depth(yas_raycaster* rc, float** depth, size_t* pitch, float* host, size_t host_pitch) {
  YAS_REQUIRE(rc, "yas_raycaster_depth: null ray caster");
  YAS_REQUIRE(!host || host_pitch >= sizeof(float) * (size_t)rc->W, "yas_raycaster_depth: host pitch too small");
  YAS_HIP(hipSetDevice(rc->ctx->device));
  const size_t row = sizeof(float) * (size_t)rc->W;
  if (!rc->depth) YAS_HIP(hipMalloc((void**)&rc->depth, row * rc->H));
  int r = yas_vmap_to_depth(rc->ctx, (const float*)rc->vmap, sizeof(float4) * (size_t)rc->W, rc->depth, row, rc->W,
                            rc->H);
  if (r) return r;
  if (host) {
    YAS_HIP(hipMemcpy2DAsync(host, host_pitch, rc->depth, row, row, rc->H, hipMemcpyDeviceToHost, rc->ctx->stream));
    YAS_HIP(hipStreamSynchronize(rc->ctx->stream));
  }
  if (depth) *depth = rc->depth;
  if (pitch) *pitch = row;
  return YAS_OK;
}

int yas_raycaster_zrange(yas_raycaster* rc, float** zmin, float** zmax, int* cols, int* rows) {
  YAS_REQUIRE(rc, "null argument");
  if (zmin) *zmin = (float*)rc->zmin;
  if (zmax) *zmax = (float*)rc->zmax;
  if (cols) *cols = rc->cols;
  if (rows) *rows = rc->rows;
  return YAS_OK;
}

int yas_raycaster_num_visible(yas_raycaster* rc, int* count) {
  YAS_REQUIRE(rc && count, "null argument");
  *count = 0;
  if (!rc->last_map) return YAS_OK;
  MapView v = yas_map_view(rc->last_map);
  YAS_HIP(hipMemcpyAsync(rc->host_ctr, v.ctr, sizeof(int) * kCtrCount, hipMemcpyDeviceToHost, rc->ctx->stream));
  YAS_HIP(hipStreamSynchronize(rc->ctx->stream));
  *count = rc->host_ctr[kCtrVisible];
  return YAS_OK;
}

}  // extern "C"
