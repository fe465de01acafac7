// The whole Gauss-Newton solve of one tracker in one launch.
//
// The launch-per-pass solve (k_pass1, k_step_pass1, k_pass2, k_update_into)
// is bound by launches: 37 dependent ones of 5-20 us, where about 5 us of
// each is the launch itself, every launch starts with cold caches, and a
// workgroup of four wavefronts (one per SIMD) walks its four or five pixels
// a thread one after the other.  Here the same workgroups stay resident for
// the solve and exchange their partial sums through memory.
//
// A workgroup of 1024 threads does the work of one 256-thread workgroup of
// the launch-per-pass solve: thread (t, q), t < 256, q < 4, takes the pixel
// slots q, q + 4, ... of that workgroup's thread t, so up to four pixels of
// a thread's run are worked on at once.  Each pixel's row goes to LDS, and
// the rows of a run are then summed in slot order (a quarter of the products
// by each q), so every sum has the launch-per-pass solve's order and bits.
//
// Exchange: a partial sum, a statistic or a pose word travels as one 8-byte
// word {value, epoch}, stored and polled with relaxed agent-scope atomics.
// The epoch (one per iteration, never reused) says that the word is this
// iteration's, so no fence (an L2 write-back on each XCD) and no counter is
// needed.  Workgroup 0 folds the rows, takes the step and publishes the next
// pose; the residual statistics are folded by every workgroup.  A word is
// overwritten only after all its readers have gone on: the next iteration's
// rows follow the pose that workgroup 0 publishes after reading this one's,
// and workgroups that a level has no work for wait only for the last pose
// before their first level.
//
// All workgroups must be resident at once.  The host takes this path only
// when the device holds the grid, and for one solve at a time.  Every wait
// is bounded by the clock all the same: a workgroup whose wait runs out
// leaves, the tracker's state stays as it was before the solve, and
// k_solve_rescue takes the whole solve in one workgroup with the
// launch-per-pass code (the same sums, so the same bits).  It follows each
// queued solve on the stream.  A caller that waits for the solve sees in host
// memory whether it completed, and else takes the separate passes.  After a
// lost solve the tracker takes the passes for a while.
#pragma once

#include <type_traits>

#include "yas_tracker_dev.hpp"

namespace yas {

constexpr int kSolveThreads = 1024;
constexpr int kSolveSlots = kSolveThreads / 256;  // pixel slots worked on at once
constexpr int kSolveBatch = 2;                    // slots of a thread whose rows are in LDS at once

// Words exchanged between the workgroups of a solve (zeroed at creation).
struct SolveXchg {
  unsigned epoch;  // of the last iteration of the last solve
  int ok;          // set when a solve completes, cleared by k_solve_rescue
  unsigned rescued;  // solves that k_solve_rescue took
  int pad[29];
  unsigned long long pose[32];  // float pose (12) and warp (12) of the next iteration
  unsigned long long stat[kRedGroups][4];
  unsigned long long icp[kRedGroups][32];
  unsigned long long rgb[kRedGroups][32];
};

// A solve's result in host memory, for the caller that waits for it.
struct HostState {
  TrackState s;
  int ok;          // the solve completed
  unsigned ended;  // number of the tracker's last solve that has ended
  unsigned rescued;  // its queued solves that the rescue took
};

struct SolveArgs {
  Level lv[kMaxLevels];
  TrackBufs tb[kMaxLevels];
  int iters[kMaxLevels];
  int groups[kMaxLevels];  // workgroups of the level's passes
  int levels, mode;
  float sin2_max, dist2_max;
  float wrh, wrb, wih, wib;
  TrackState* st;
  SolveXchg* x;
  float* part_icp;  // the rescue's partial rows
  float* part_res;
  float* part_rgb;
  unsigned long long wait_ticks;  // bound of a wait, 100 MHz clock ticks
  Mat44 init;      // the pose to start from when `has_init`, else the state's
  int has_init;
  HostState* host;  // when set, a completed solve's state goes there too (and `ok` is its)
};

// The thread index, as a value the compiler takes as new at each call: what
// is derived from it (LDS and word addresses above all) is then formed again
// in each phase of each iteration instead of being kept in registers, or
// spilled, across the whole solve.
__device__ inline int fresh_tid() {
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

// ------------------------------------------------------------------ lanes
// Wavefront sums of 8 values in wave_sum32's order (partners at 32, 16, 8,
// 4, 2, 1): lane l returns the total of value wave_sum8_index(l).
__device__ inline float wave_sum8(const float (&v)[8]) {
  const float y0 = pair32(v[0], v[4]), y1 = pair32(v[1], v[5]), y2 = pair32(v[2], v[6]), y3 = pair32(v[3], v[7]);
  const float z0 = pair16(y0, y2), z1 = pair16(y1, y3);
  const bool hi = (threadIdx.x & 8) != 0;
  const float keep = hi ? z1 : z0, send = hi ? z0 : z1;
  float u = keep + lane_xor<8>(send);
  u = u + lane_xor<4>(u);
  u = u + lane_xor<2>(u);
  return u + lane_xor<1>(u);
}
__device__ inline int wave_sum8_index(int lane) {
  return ((lane >> 5) & 1) * 4 + ((lane >> 4) & 1) * 2 + ((lane >> 3) & 1);
}

// wave_stats with the lanes' values exchanged by data-parallel moves instead
// of LDS permutes, the lower lane's values first: lane 0 gets the wavefront's
// (the others' are of no use, which spares telling which lane is the lower).
// (Not for the passes: there it made the pixel loop spill.)
template <int M>
__device__ inline float lane_above(float v) {  // lane l + M's of the same 16; 0 past them
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x100 + M, 0xF, 0xF, true));
}
template <int M>
__device__ inline void merge_above(float& n, float& mean, float& m2) {
  chan_merge(n, mean, m2, lane_above<M>(n), lane_above<M>(mean), lane_above<M>(m2));
}
// {v of the lower, v of the upper lane} of partners at 16 and 32.
__device__ inline float2 both16(float v) {
  const unsigned u = __builtin_bit_cast(unsigned, v);
  const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  return make_float2(__builtin_bit_cast(float, (unsigned)r[0]), __builtin_bit_cast(float, (unsigned)r[1]));
}
__device__ inline float2 both32(float v) {
  const unsigned u = __builtin_bit_cast(unsigned, v);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return make_float2(__builtin_bit_cast(float, (unsigned)r[0]), __builtin_bit_cast(float, (unsigned)r[1]));
}
__device__ inline void wave_stats_moves(float& n, float& mean, float& m2) {
  merge_above<1>(n, mean, m2);
  merge_above<2>(n, mean, m2);
  merge_above<4>(n, mean, m2);
  merge_above<8>(n, mean, m2);
  float2 a = both16(n), b = both16(mean), c = both16(m2);
  n = a.x; mean = b.x; m2 = c.x;
  chan_merge(n, mean, m2, a.y, b.y, c.y);
  a = both32(n); b = both32(mean); c = both32(m2);
  n = a.x; mean = b.x; m2 = c.x;
  chan_merge(n, mean, m2, a.y, b.y, c.y);
}

// ------------------------------------------------------------------ words
__device__ inline void put_word(unsigned long long* p, unsigned v, unsigned epoch) {
  __hip_atomic_store(p, ((unsigned long long)epoch << 32) | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void put_word(unsigned long long* p, float v, unsigned epoch) {
  put_word(p, __builtin_bit_cast(unsigned, v), epoch);
}
__device__ inline unsigned long long get_word(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline float word_value(unsigned long long w) { return __builtin_bit_cast(float, (unsigned)w); }

// The values of the N words at byte offsets at(i) from `base` (those with
// want(i), 0 for the others, which must be readable too) once all carry
// `epoch`; false when the wait's bound passes first.  All words are loaded
// together.  STEPS (one word): the bound begins again whenever the word's epoch
// has changed, for a workgroup that waits for a level's iterations together.
template <int N, bool STEPS = false, class P, class W>
__device__ inline bool wait_words(const void* base, P at, W want, unsigned epoch, unsigned long long ticks,
                                  float (&out)[N]) {
  static_assert(!STEPS || N == 1, "the epoch of one word");
  unsigned long long t0 = 0;
  unsigned seen = 0;
  for (unsigned looks = 0;; ++looks) {
    unsigned long long w[N];
#pragma unroll
    for (int i = 0; i < N; ++i) w[i] = get_word((const unsigned long long*)((const char*)base + (unsigned)at(i)));
    unsigned miss = 0;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      miss |= want(i) ? (unsigned)(w[i] >> 32) ^ epoch : 0u;
      out[i] = want(i) ? word_value(w[i]) : 0.0f;
    }
    const bool all = miss == 0;
    if (all) return true;
    const unsigned every = ticks ? 31u : 0u;
    if ((looks & every) == every) {  // the clock is read at every 32nd look
      const unsigned long long now = wall_clock64();
      if (looks == every || (STEPS && (unsigned)(w[0] >> 32) != seen)) t0 = now;
      if (STEPS) seen = (unsigned)(w[0] >> 32);
      if (now - t0 >= ticks) return false;
    }
  }
}

// ------------------------------------------------------------------ LDS
// Rows of a batch of slots, [slot][element][thread]; element 7 is the weight
// (pass 2), `r` the residual of each slot (pass 1).  The small arrays lie
// first: an LDS instruction's offset reaches 64 KB, and an array beyond that
// takes a register for each of its addresses, which the compiler then keeps,
// and spills, over the whole solve.
struct SolveLds {
  float part[29][4];                         // a row's wavefront sums
  int count[16];                             // matches by wavefront
  float stats[4][3];
  float fold[2][16][32];
  float sums[2][32];
  float pose[12], warp[12];
  double est[16];
  float H[36], b[6];
  double xs[6], W[9], E[16];
  double Kinv[2][9];  // inverse intrinsics of this level and of the next one with iterations
  TrackState s;  // workgroup 0's running state
  int lost;      // a wait ran out
  float r[kSolveBatch * kSolveSlots][256];
  float kept[kSolveBatch][6][kSolveThreads];  // residual, gradients and warped point, for pass 2
  float row[kSolveBatch * kSolveSlots][8][256];
};

// The products of the upper triangle of a 7-element row that quarter q sums
// over slots first .. first + 3, in that order; 7 products each:
//   q 0: row 0; q 1: row 1 and (6,6); q 2: rows 2 and 5; q 3: rows 3 and 4
template <bool WEIGHTED, int N>
__device__ inline void add_slots(const SolveLds& S, int first, int q, int t, float (&acc)[8]) {
#pragma unroll
  for (int s = first; s < first + N; ++s) {
    const float w = WEIGHTED ? S.row[s][7][t] : 1.0f;
    // wt * row[i] * row[j] is summed as (wt * row[i]) * row[j]
    auto lead = [&](float x) { return WEIGHTED ? w * x : x; };
    if (q == 0) {
      const float a = lead(S.row[s][0][t]);
      acc[0] += a * S.row[s][0][t];
#pragma unroll
      for (int j = 1; j < 7; ++j) acc[j] += a * S.row[s][j][t];
    } else if (q == 1) {
      const float a = lead(S.row[s][1][t]), z = S.row[s][6][t];
#pragma unroll
      for (int j = 1; j < 6; ++j) acc[j - 1] += a * S.row[s][j][t];
      acc[5] += a * z;
      acc[6] += lead(z) * z;
    } else if (q == 2) {
      const float x2 = S.row[s][2][t], x5 = S.row[s][5][t], x6 = S.row[s][6][t];
      const float a = lead(x2), c = lead(x5);
      acc[0] += a * x2;
      acc[1] += a * S.row[s][3][t];
      acc[2] += a * S.row[s][4][t];
      acc[3] += a * x5;
      acc[4] += a * x6;
      acc[5] += c * x5;
      acc[6] += c * x6;
    } else {
      const float x3 = S.row[s][3][t], x4 = S.row[s][4][t], x5 = S.row[s][5][t], x6 = S.row[s][6][t];
      const float a = lead(x3), c = lead(x4);
      acc[0] += a * x3;
      acc[1] += a * x4;
      acc[2] += a * x5;
      acc[3] += a * x6;
      acc[4] += c * x4;
      acc[5] += c * x5;
      acc[6] += c * x6;
    }
  }
}
// Slots 0 .. n - 1 of a batch.
template <bool WEIGHTED>
__device__ inline void add_products(const SolveLds& S, int n, int q, int t, float (&acc)[8]) {
  int s = 0;
#pragma unroll 1
  for (; s + kSolveSlots <= n; s += kSolveSlots) add_slots<WEIGHTED, kSolveSlots>(S, s, q, t, acc);
#pragma unroll 1
  for (; s < n; ++s) add_slots<WEIGHTED, 1>(S, s, q, t, acc);
}
// Where quarter q's v-th product lies in the packed 28.
__device__ inline int product_index(int q, int v) {
  if (q == 0) return v;
  if (q == 1) return v < 6 ? 7 + v : 27;
  if (q == 2) return v < 5 ? 13 + v : 25 + v - 5;
  return 18 + v;
}
// The wavefront sums of a pass's products and match counts into LDS
// (S.part, S.count); the caller synchronises and reads row_total.
__device__ inline void put_sums(SolveLds& S, int q, const float (&acc)[8], int count) {
  const int tid = fresh_tid();
  const int lane = tid & 63, wave = tid >> 6;
  const float u = wave_sum8(acc);
  const int v = wave_sum8_index(lane);
  if ((lane & 7) == 0 && v < 7) S.part[product_index(q, v)][wave & 3] = u;
  if (lane == 0) S.count[wave] = count;
}
// Element c < 29 of the workgroup's partial row.
__device__ inline float row_total(const SolveLds& S, int c) {
  if (c < 28) return ((S.part[c][0] + S.part[c][1]) + S.part[c][2]) + S.part[c][3];
  int n = 0;
#pragma unroll
  for (int w = 0; w < 16; ++w) n += S.count[w];
  return (float)n;
}

// ------------------------------------------------------------------ passes
// Pixel k's row and column: the quotient by a float product, set right where
// it is off by one; the integer division was 25 instructions of each pixel.
// The product's relative error is below 2^-22, so it is off by no more than
// one in images of up to 2^22 rows (kFastRows).
constexpr int kFastRows = 1 << 22;
__device__ inline void pixel_xy(int k, int w, float winv, int& x, int& y) {
  y = (int)((float)k * winv);
  x = k - y * w;
  if (x < 0) {
    x += w;
    --y;
  }
  if (x >= w) {
    x -= w;
    ++y;
  }
}

// Element `at` of an array by a 32-bit byte offset from its (uniform) base:
// one register an address instead of two.  Images here have at most 2^26
// pixels (the host checks).
template <class T>
__device__ inline T& elem(T* base, int at) {
  typedef typename std::conditional<std::is_const<T>::value, const char, char>::type C;
  return *(T*)((C*)base + (unsigned)at * (unsigned)sizeof(T));
}
__device__ inline IcpPoint solve_icp_point(const float4* m, int n, int k) {
  const float4 a = elem(m, k);
  const float2 b = elem(reinterpret_cast<const float2*>(m + n), k);
  IcpPoint p;
  p.vx = a.x; p.vy = a.y; p.vz = a.z; p.nx = a.w; p.ny = b.x; p.nz = b.y;
  return p;
}
template <bool ICP, bool RGB>
__device__ inline RefPixel solve_ref_pixel(const TrackBufs& B, int n, int k) {
  RefPixel r = {};
  if (ICP) r.p = solve_icp_point(B.ref_p, n, k);
  if (RGB) {
    r.iz = elem(B.ref_inv, k);
    r.inten = elem(B.ref_int, k);
  }
  return r;
}

// A pixel's ICP row (icp_pixel's arithmetic) and photometric residual
// (rgb_pixel's) with the gathers of both issued before either is used; a
// pixel with no match has a zero row (which adds +0, an identity here: a sum
// that starts at +0 is never -0), one with no residual a NaN r.
struct PixelTerms {
  float row[7];
  bool icp;
  float r, gx, gy;  // photometric row as stored (NaN, 0, 0 where none)
  float px, py, pz;
};
template <bool ICP, bool RGB>
__device__ inline PixelTerms pixel_terms(const Level& L, const TrackBufs& B, const PoseF& T, const float* wp,
                                         float sin2_max, float dist2_max, float winv, int k, bool in,
                                         const RefPixel& ref) {
  PixelTerms o;
  float vx = 0.f, vy = 0.f, vz = 1.f;
  bool hit = false, rgb = false;
  IcpPoint c = {};
  if (ICP) {
    xform(T, ref.p.vx, ref.p.vy, ref.p.vz, vx, vy, vz);
    const float invz = 1.0f / vz;
    const int u = floor_sat(L.fx * vx * invz + L.cx + 0.5f);
    const int v = floor_sat(L.fy * vy * invz + L.cy + 0.5f);
    hit = in && ref.p.vx == ref.p.vx && !(u < 0 || v < 0 || u >= L.w || v >= L.h);
    c = solve_icp_point(B.cur_p, L.w * L.h, hit ? v * L.w + u : 0);
  }
  float fu = 0.f, fv = 0.f, tap[3][4];
  if (RGB) {
    int x, y;
    pixel_xy(k, L.w, winv, x, y);
    const float4 p = warp_ref_xy(wp, x, y, in ? ref.iz : 0.0f);
    o.px = p.x; o.py = p.y; o.pz = p.z;
    const float u = L.fx * p.x / p.z + L.cx;
    const float v = L.fy * p.y / p.z + L.cy;
    rgb = p.w > 0.0f && u > 0.0f && v > 0.0f && u < (float)(L.w - 1) && v < (float)(L.h - 1);
    const float su = rgb ? u : 0.0f, sv = rgb ? v : 0.0f;
    const int iu = (int)floorf(su), iv = (int)floorf(sv);
    fu = su - (float)iu;
    fv = sv - (float)iv;
    const int at = iv * L.w + iu;
    const float* m[3] = {B.cur_int, B.gx, B.gy};
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const float* row0 = &elem(m[i], at);
      const float* row1 = &elem(m[i], at + L.w);
      tap[i][0] = row0[0];
      tap[i][1] = row0[1];
      tap[i][2] = row1[0];
      tap[i][3] = row1[1];
    }
  }
  if (ICP) {
    float nx, ny, nz;
    rot3(T, ref.p.nx, ref.p.ny, ref.p.nz, nx, ny, nz);
    const float dx = vx - c.vx, dy = vy - c.vy, dz = vz - c.vz;
    const float dist2 = dx * dx + dy * dy + dz * dz;
    const float c0 = c.ny * nz - c.nz * ny, c1 = c.nz * nx - c.nx * nz, c2 = c.nx * ny - c.ny * nx;
    const float sin2 = c0 * c0 + c1 * c1 + c2 * c2;
    o.icp = hit && sin2 <= sin2_max && dist2 <= dist2_max;
    const float row[7] = {nx, ny, nz, vy * nz - vz * ny, vz * nx - vx * nz, vx * ny - vy * nx,
                          nx * (c.vx - vx) + ny * (c.vy - vy) + nz * (c.vz - vz)};
#pragma unroll
    for (int i = 0; i < 7; ++i) o.row[i] = o.icp ? row[i] : 0.0f;
  }
  if (RGB) {
    auto lerp = [&](const float* q) {
      return (q[0] * (1.0f - fu) + q[1] * fu) * (1.0f - fv) + (q[2] * (1.0f - fu) + q[3] * fu) * fv;
    };
    const float r = lerp(tap[0]) - ref.inten, gx = lerp(tap[1]), gy = lerp(tap[2]);
    const bool ok = rgb && (gx * gx + gy * gy) > 0.0f && isfinite(r);
    o.r = ok ? r : __builtin_nanf("");
    o.gx = ok ? gx : 0.0f;
    o.gy = ok ? gy : 0.0f;
  }
  return o;
}

// Pixel slots of a workgroup's thread t < 256 (a last one may be past the
// image), worked on in rounds of kSolveSlots, and of those the batch's from
// round r0.  Slots past the count are left out: their zero rows add +0.
__device__ inline int solve_slots(int N, int nb) { return (N + nb * 256 - 1) / (nb * 256); }
__device__ inline int solve_rounds(int slots) { return (slots + kSolveSlots - 1) / kSolveSlots; }
__device__ inline int batch_slots(int slots, int r0) {
  const int n = slots - r0 * kSolveSlots;
  return n < kSolveBatch * kSolveSlots ? n : kSolveBatch * kSolveSlots;
}

// Pass 1 of workgroup bx of nb: the rows of the last batch of slots in LDS
// (the ICP products of the batches before it are in `acc`), the residuals'
// statistics by wavefront in S.stats.  The products of the last batch are
// left to the caller, who publishes the statistics first: pass 2 of every
// workgroup waits for those.
template <bool ICP, bool RGB>
__device__ inline void solve_pass1(SolveLds& S, const Level& L, const TrackBufs& B, const PoseF& T, const float* wp,
                                   float sin2_max, float dist2_max, int bx, int nb, RefPixel nxt, float (&acc)[8],
                                   int& count) {
  const int tid = fresh_tid();
  const int t = tid & 255;
  const int q = __builtin_amdgcn_readfirstlane(tid >> 8);
  const int N = L.w * L.h, stride = nb * 256;
  const int slots = solve_slots(N, nb), rounds = solve_rounds(slots);
  const float winv = 1.0f / (float)L.w;
  float n = 0.0f, mean = 0.0f, m2 = 0.0f;
  int k = bx * 256 + t + q * stride;
#pragma unroll 1
  for (int r0 = 0; r0 < rounds; r0 += kSolveBatch) {
    if (r0 > 0) __syncthreads();  // the last batch's rows have been read
    const int ns = batch_slots(slots, r0);
#pragma unroll 1
    for (int r = 0; r * kSolveSlots + q < ns; ++r, k += kSolveSlots * stride) {
      const RefPixel cur = nxt;
      const int kn = k + kSolveSlots * stride;
      if ((r0 + r + 1) * kSolveSlots + q < slots) nxt = solve_ref_pixel<ICP, RGB>(B, N, kn < N ? kn : N - 1);
      const bool in = k < N;
      PixelTerms o = {};
      o.r = __builtin_nanf("");
      // a wavefront past the image (most of a last round) has no pixel to do
      if (__any(in)) o = pixel_terms<ICP, RGB>(L, B, T, wp, sin2_max, dist2_max, winv, k, in, cur);
      const int slot = r * kSolveSlots + q;
      if (ICP) {
#pragma unroll
        for (int i = 0; i < 7; ++i) S.row[slot][i][t] = o.row[i];
        count += __popcll(__ballot(o.icp));
      }
      if (RGB) {
        S.r[slot][t] = o.r;
        if (in) elem(B.resid, k) = make_float3(o.r, o.gx, o.gy);
        if (r0 == 0) {
          float(&kp)[6][kSolveThreads] = S.kept[r];
          kp[0][tid] = o.r; kp[1][tid] = o.gx; kp[2][tid] = o.gy;
          kp[3][tid] = o.px; kp[4][tid] = o.py; kp[5][tid] = o.pz;
        }
      }
    }
    __syncthreads();
    if (RGB && q == 3) {
#pragma unroll 4
      for (int s = 0; s < ns; ++s) {
        const float e = S.r[s][t];
        if (e == e) {
          n += 1.0f;
          const float d = e - mean;
          mean = mean + d / n;
          m2 = m2 + d * (e - mean);
        }
      }
    }
    if (ICP && r0 + kSolveBatch < rounds) add_products<false>(S, ns, q, t, acc);
  }
  if (RGB && q == 3) {
    wave_stats_moves(n, mean, m2);
    if ((tid & 63) == 0) {
      float* st = S.stats[(tid >> 6) & 3];
      st[0] = n; st[1] = mean; st[2] = m2;
    }
  }
}
// The ICP products of pass 1's last batch, then S.part / S.count.
__device__ inline void solve_pass1_end(SolveLds& S, int slots, float (&acc)[8], int count) {
  const int tid = fresh_tid();
  const int q = __builtin_amdgcn_readfirstlane(tid >> 8);
  const int last = (solve_rounds(slots) - 1) / kSolveBatch * kSolveBatch;  // the last batch's first round
  add_products<false>(S, batch_slots(slots, last), q, tid & 255, acc);
  put_sums(S, q, acc, count);
}

// Pass 2 of workgroup bx of nb with Huber threshold th: S.part / S.count.
__device__ inline void solve_pass2(SolveLds& S, const Level& L, const TrackBufs& B, const float* wp, float th, int bx,
                                   int nb) {
  const int tid = fresh_tid();
  const int t = tid & 255;
  const int q = __builtin_amdgcn_readfirstlane(tid >> 8);
  const int N = L.w * L.h, stride = nb * 256;
  const int slots = solve_slots(N, nb), rounds = solve_rounds(slots);
  float acc[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) acc[i] = 0.0f;
  int count = 0;
  int k = bx * 256 + t + q * stride;
#pragma unroll 1
  for (int r0 = 0; r0 < rounds; r0 += kSolveBatch) {
    if (r0 > 0) __syncthreads();  // the last batch's rows have been read
    const int ns = batch_slots(slots, r0);
#pragma unroll 1
    for (int r = 0; r * kSolveSlots + q < ns; ++r, k += kSolveSlots * stride) {
      float e, gx, gy, px, py, pz;
      if (r0 == 0) {
        const float(&kp)[6][kSolveThreads] = S.kept[r];
        e = kp[0][tid]; gx = kp[1][tid]; gy = kp[2][tid];
        px = kp[3][tid]; py = kp[4][tid]; pz = kp[5][tid];
      } else {
        // this thread stored the row in pass 1
        const float3 f = k < N ? B.resid[k] : make_float3(__builtin_nanf(""), 0.f, 0.f);
        const float4 p = warp_ref(L, wp, k, k < N ? B.ref_inv[k] : 0.0f);
        e = f.x; gx = f.y; gy = f.z;
        px = p.x; py = p.y; pz = p.z;
      }
      const bool has = e == e;
      float row[7] = {}, wt = 0.0f;
      if (has) {
        const float zinv = 1.0f / pz;
        wt = 1.0f;
        if (fabsf(e) > th) wt = th / fabsf(e);
        row[0] = gx * L.fx * zinv;
        row[1] = gy * L.fy * zinv;
        row[2] = -(row[0] * px + row[1] * py) * zinv;
        row[3] = row[2] * py - gy * L.fy;
        row[4] = -row[2] * px + gx * L.fx;
        row[5] = -row[0] * py + row[1] * px;
        row[6] = -e;
      }
      const int slot = r * kSolveSlots + q;
#pragma unroll
      for (int i = 0; i < 7; ++i) S.row[slot][i][t] = row[i];
      S.row[slot][7][t] = wt;
      count += __popcll(__ballot(has));
    }
    __syncthreads();
    add_products<true>(S, ns, q, t, acc);
  }
  put_sums(S, q, acc, count);
}

// Workgroup 0: the partial rows of one kind folded in gn_update's order
// (rows as threads of four wavefronts: partners at 32, 16, 8, 4, 2, 1, then
// the wavefronts in turn), by W = 8 or 16 wavefronts.  Thread (value i,
// part) takes the rows that differ in the high bits of the lower six (5, 4,
// 3, and 2 when W is 8); lane bit 5 is the next bit, and the wavefront holds
// row bits 7, 6 and the rest.  The wavefronts' sums go to `fold`.
template <int W>
__device__ inline void solve_fold(SolveLds& S, const unsigned long long (*rows)[32], float (*fold)[32], int wave,
                                  int nb, unsigned epoch, unsigned long long ticks) {
  constexpr int J = 128 / W;                    // rows a thread takes
  constexpr int kLow = W == 16 ? 2 : 1;         // row bits below the lane's
  const int tid = fresh_tid();
  const int i = tid & 31, half = (tid >> 5) & 1;
  const int row0 = (wave >> kLow) * 64 + (half << kLow) + (wave & ((1 << kLow) - 1));
  float v[J];
  auto row = [&](int j) { return row0 + (j << (kLow + 1)); };
  const bool ok = wait_words<J>(rows, [&](int j) { return (row(j) * 32 + i) * 8; },
                                [&](int j) { return i < 29 && row(j) < nb; }, epoch, ticks, v);
  if (!ok) S.lost = 1;
#pragma unroll
  for (int h = J / 2; h > 0; h >>= 1)
#pragma unroll
    for (int j = 0; j < h; ++j) v[j] = v[j] + v[j + h];
  const float w = pair32(v[0], v[0]);
  if (half == 0) fold[wave][i] = w;
}
// Value i's total of the wavefronts' sums.
template <int W>
__device__ inline float solve_fold_total(const float (*fold)[32], int i) {
  float s = 0.0f;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    float e;
    if (W == 16) {
      const float a = fold[4 * w][i] + fold[4 * w + 2][i];      // row bit 1, bit 0 clear
      const float b = fold[4 * w + 1][i] + fold[4 * w + 3][i];  // row bit 1, bit 0 set
      e = a + b;
    } else {
      e = fold[2 * w][i] + fold[2 * w + 1][i];  // row bit 0
    }
    s = w == 0 ? e : s + e;
  }
  return s;
}

// The Huber threshold of the level's nb statistics rows, folded as
// huber_threshold does; every thread gets it.  Workgroup 0 records the
// statistics (`record`).  S.lost is set when the wait runs out (synchronised here).
template <bool ICP>
__device__ inline float solve_threshold(SolveLds& S, const SolveXchg* x, int nb, unsigned epoch,
                                        unsigned long long ticks, bool record) {
  const int tid = fresh_tid();
  // workgroup 0 folds the ICP rows meanwhile, with the upper wavefronts
  if (ICP && record && tid >= 512)
    solve_fold<8>(S, x->icp, S.fold[0], (tid >> 6) - 8, nb, epoch, ticks);
  if (tid < 256) {
    float n = 0.0f, mean = 0.0f, m2 = 0.0f;
    const int g = tid;
    if (g < nb) {
      float v[3];
      if (!wait_words<3>(x->stat, [&](int i) { return (g * 4 + i) * 8; }, [](int) { return true; }, epoch, ticks, v)) S.lost = 1;
      chan_merge(n, mean, m2, v[0], v[1], v[2]);
    }
    wave_stats_moves(n, mean, m2);
    if ((tid & 63) == 0) {
      float* st = S.stats[tid >> 6];
      st[0] = n; st[1] = mean; st[2] = m2;
    }
  }
  __syncthreads();
  float n = S.stats[0][0], mean = S.stats[0][1], m2 = S.stats[0][2];
#pragma unroll
  for (int w = 1; w < 4; ++w) chan_merge(n, mean, m2, S.stats[w][0], S.stats[w][1], S.stats[w][2]);
  const float sigma = sqrtf(m2 / (n - 1.0f));
  const float th = (float)(4.685 * (double)sigma);
  if (record && tid == 0) {
    S.s.rgb_stats[0] = n * mean;
    S.s.rgb_stats[1] = n;
    S.s.rgb_stats[2] = mean;
    S.s.rgb_stats[3] = th;
  }
  return th;
}

__device__ inline SolveLds& solve_lds() {
  __shared__ SolveLds S;
  return S;
}

// Workgroup 0's step (wavefront 0) into S.est, a function of its own: the
// pixel loops' registers and the double-precision solve's do not fit together,
// and inlined the solve spilled (RGB-D, 640x480, with its inputs: 347 us against 320 us).
__device__ __attribute__((noinline)) GnStep solve_step(int mode, float wrh, float wrb, float wih, float wib) {
  SolveLds& S = solve_lds();
  GnStep g = {false, false, 0.0f};
  double t = 0.0;
  if (S.s.good) g = gn_step_pose(S.sums, S.est, mode, wrh, wrb, wih, wib, S.H, S.b, S.xs, S.W, S.E, t);
  if (g.moved && (threadIdx.x & 63) < 16) S.est[threadIdx.x & 63] = t;
  return g;
}

// load_warp with the inverse intrinsics' matrix in LDS.
__device__ inline void solve_load_warp(const double* T, const double* Ki, float* out) {
  if (threadIdx.x >= 16 && threadIdx.x < 28) {
    const int q = threadIdx.x - 16, i = q / 4, j = q % 4;
    if (j < 3) out[3 * i + j] = (float)(T[4 * i] * Ki[j] + T[4 * i + 1] * Ki[3 + j] + T[4 * i + 2] * Ki[6 + j]);
    else out[9 + i] = (float)T[4 * i + 3];
  }
}

template <bool ICP, bool RGB>
__device__ inline void solve_body(SolveLds& S, const SolveArgs& a) {
  const int bx = blockIdx.x;
  unsigned epoch = a.x->epoch;
  if (threadIdx.x < 16) S.est[threadIdx.x] = a.has_init ? a.init.m[threadIdx.x] : a.st->est[threadIdx.x];
  if (threadIdx.x == 0) S.lost = 0;
  if (bx == 0) {
    for (int w = threadIdx.x; w < (int)(sizeof(TrackState) / 4); w += kSolveThreads)
      ((int*)&S.s)[w] = ((const int*)a.st)[w];
    if (a.has_init) {
      __syncthreads();
      track_init_at(&S.s, a.init.m);
    }
  }
  __syncthreads();
  bool fresh = true;  // the pose in LDS is for this level's first iteration
#pragma unroll 1
  for (int l = a.levels - 1; l >= 0; --l) {
    const int iters = a.iters[l];
    if (iters <= 0) continue;
    const int nb = a.groups[l];
    int below = l - 1;  // the next level with iterations
    while (below >= 0 && a.iters[below] <= 0) --below;
    if (RGB && bx == 0 && threadIdx.x < 18) {  // read after the barriers of an iteration
      const int m = threadIdx.x < 9 ? 0 : 1, e = threadIdx.x - 9 * m;
      const double* K = a.lv[m == 0 || below < 0 ? l : below].Kinv;
      S.Kinv[m][e] = e == 0 ? K[0] : e == 2 ? K[2] : e == 4 ? K[1] : e == 5 ? K[3] : e == 8 ? 1.0 : 0.0;
    }
    if (bx >= nb) {  // no work at this level: its poses are not read here
      epoch += iters;
      fresh = false;
      continue;
    }
#pragma unroll 1
    for (int it = 0; it < iters; ++it) {
      // the level's constants are read again in each iteration: kept over
      // all of them they would not fit the scalar registers
      int lc = l;
      asm volatile("" : "+s"(lc));
      const Level& L = a.lv[lc];
      const TrackBufs& B = a.tb[lc];
      // the first pixel's reference values, in flight while the pose is awaited
      RefPixel ref;
      {
        const int tid = fresh_tid(), N = L.w * L.h;
        const int k = bx * 256 + (tid & 255) + (tid >> 8) * nb * 256;
        ref = solve_ref_pixel<ICP, RGB>(B, N, k < N ? k : N - 1);
      }
      // the pose: the state's for the solve's first iteration, else the
      // word that workgroup 0 published after the one before
      if (fresh) {
        load_pose_f(S.est, S.pose);
        if (RGB) load_warp(S.est, L.Kinv, S.warp);
        fresh = false;
      } else if (bx != 0) {
        const int w = fresh_tid();
        if (w < 64) {
          float v[1];
          const bool ok = wait_words<1, true>(a.x->pose, [&](int) { return (w & 31) * 8; }, [&](int) { return w < (RGB ? 24 : 12); },
                                        epoch, a.wait_ticks, v);
          if (!ok) S.lost = 1;
          if (w < 12) S.pose[w] = v[0];
          else if (w < 24) S.warp[w - 12] = v[0];
        }
      }
      __syncthreads();
      const int lost = S.lost;  // looked at once the pose is on its way too
      PoseF T;
#pragma unroll
      for (int i = 0; i < 9; ++i) T.r[i] = wave_uniform(S.pose[i]);
#pragma unroll
      for (int i = 0; i < 3; ++i) T.t[i] = wave_uniform(S.pose[9 + i]);
      float wu[12];
#pragma unroll
      for (int i = 0; i < 12; ++i) wu[i] = RGB ? wave_uniform(S.warp[i]) : 0.0f;
      if (lost) return;
      ++epoch;
      float acc[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[i] = 0.0f;
      int count = 0;
      solve_pass1<ICP, RGB>(S, L, B, T, wu, a.sin2_max, a.dist2_max, bx, nb, ref, acc, count);
      if (RGB) {
        __syncthreads();
        if (fresh_tid() == 64) {
          float n = S.stats[0][0], mean = S.stats[0][1], m2 = S.stats[0][2];
#pragma unroll
          for (int w = 1; w < 4; ++w) chan_merge(n, mean, m2, S.stats[w][0], S.stats[w][1], S.stats[w][2]);
          put_word(&a.x->stat[bx][0], n, epoch);
          put_word(&a.x->stat[bx][1], mean, epoch);
          put_word(&a.x->stat[bx][2], m2, epoch);
        }
      }
      if (ICP) {
        solve_pass1_end(S, solve_slots(L.w * L.h, nb), acc, count);
        __syncthreads();
        const int tid = fresh_tid();
        if (tid < 29) put_word(&a.x->icp[bx][tid], row_total(S, tid), epoch);
      }
      if (RGB) {
        __syncthreads();  // S.stats and S.part are written again below
        const float th = solve_threshold<ICP>(S, a.x, nb, epoch, a.wait_ticks, bx == 0);
        if (S.lost) return;  // set before the barrier in solve_threshold
        solve_pass2(S, L, B, wu, th, bx, nb);
        __syncthreads();
        const int tid = fresh_tid();
        if (tid < 29) put_word(&a.x->rgb[bx][tid], row_total(S, tid), epoch);
      }
      if (bx != 0) continue;
      // workgroup 0: the step, and the next iteration's pose
      const int wave = fresh_tid() >> 6;
      if (RGB) solve_fold<16>(S, a.x->rgb, S.fold[1], wave, nb, epoch, a.wait_ticks);
      else solve_fold<16>(S, a.x->icp, S.fold[0], wave, nb, epoch, a.wait_ticks);
      __syncthreads();
      if (S.lost) return;
      const int lane = fresh_tid();
      if (lane < 64) {
        const int i = lane & 31;
        if (lane < 32) {
          if (ICP) S.sums[0][i] = RGB ? solve_fold_total<8>(S.fold[0], i) : solve_fold_total<16>(S.fold[0], i);
        } else if (RGB) {
          S.sums[1][i] = solve_fold_total<16>(S.fold[1], i);
        }
        wave_lds_sync();
      }
      if (lane < 64) {
        const GnStep g = solve_step(a.mode, a.wrh, a.wrb, a.wih, a.wib);
        wave_lds_sync();
        const int nl = it + 1 < iters ? l : below;
        if (nl >= 0) {
          load_pose_f(S.est, S.pose);
          if (RGB) solve_load_warp(S.est, S.Kinv[it + 1 < iters ? 0 : 1], S.warp);
          wave_lds_sync();
          const int w = fresh_tid();
          if (w < 12) put_word(&a.x->pose[w], S.pose[w], epoch);
          else if (RGB && w < 24) put_word(&a.x->pose[w], S.warp[w - 12], epoch);
        }
        // the state, while the pose is on its way
        const int e = fresh_tid();
        if (e < 29) {
          if (ICP) S.s.sums_icp[e] = S.sums[0][e];
          if (RGB) S.s.sums_rgb[e] = S.sums[1][e];
        }
        gn_step_record(&S.s, S.sums, S.s.last_err, ICP ? nb : 0, RGB ? nb : 0, it == 0, l == 0, g,
                       S.est[e & 15]);
      }
      __syncthreads();
    }
  }
  if (bx != 0) return;
  for (int w = threadIdx.x; w < (int)(sizeof(TrackState) / 4); w += kSolveThreads)
    ((int*)a.st)[w] = ((const int*)&S.s)[w];
  if (a.host)
    for (int w = threadIdx.x; w < (int)(sizeof(TrackState) / 4); w += kSolveThreads)
      ((int*)&a.host->s)[w] = ((const int*)&S.s)[w];
  if (threadIdx.x == 0) {
    a.x->epoch = epoch;
    *(a.host ? &a.host->ok : &a.x->ok) = 1;
  }
}

// The launch-per-pass solve by one workgroup of 256 threads, for a solve
// whose workgroups did not meet.  The epochs that it may have used are
// skipped.
template <bool ICP, bool RGB>
__device__ inline void solve_rescue(const SolveArgs& a) {
  const int ok = a.x->ok;
  __syncthreads();
  if (threadIdx.x == 0) a.x->ok = 0;
  if (ok) return;
  int used = 0;
  for (int l = a.levels - 1; l >= 0; --l)
    for (int it = 0; it < a.iters[l]; ++it, ++used) {
      const int G = a.groups[l];
      for (int b = 0; b < G; ++b) {
        pass1_at<ICP, RGB>(a.lv[l], a.tb[l], a.st, a.part_icp, a.part_res, a.sin2_max, a.dist2_max, b, G);
        __syncthreads();
      }
      if (RGB)
        for (int b = 0; b < G; ++b) {
          pass2_at(a.lv[l], a.tb[l], a.st, a.part_res, G, a.part_rgb, b, G);
          __syncthreads();
        }
      gn_update(a.st, a.st, true, a.part_icp, ICP ? G : 0, a.part_rgb, RGB ? G : 0, a.mode, it == 0 ? 1 : 0, 1,
                l == 0 ? 1 : 0, a.wrh, a.wrb, a.wih, a.wib, nullptr);
      __syncthreads();
    }
  if (threadIdx.x == 0) a.x->epoch += used;
}

}  // namespace yas
