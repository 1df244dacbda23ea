// Temporal gradient of stateful accumulators (phasor, accum) and the
// swept-phasor bank that exercises it.
//
// Reference: temporalIncrementGradient (Sources/DGen/Gradients.swift:209-261)
// emits three phases (Sources/DGen/Emit+TemporalGradient.swift:15-105): store
// the output gradient and the reset flag per frame, a static reverse scan per
// element (one thread each, over all frames), then a frame-parallel read
// divided by the sample rate for a phasor.  The scan is the reset-aware
// exclusive suffix sum
//   active = reset[n] > 0 ? 0 : carry;  out[n] = active;  carry = g[n] + active
// run from the last frame down.
//
// Here the scan is parallel in time too: it is an affine recurrence in the
// carry, so frames are cut into chunks of kChunk:
//   k_tg_chunk  per (element, chunk): the chunk run from a zero carry; its map
//               carry_out = alpha * carry_in + gamma (alpha = 0 when the
//               chunk holds a reset, else 1)
//   k_tg_carry  per element: the maps composed from the last chunk down ->
//               the carry entering every chunk
//   k_tg_apply  per (element, chunk): the chunk re-run from its carry in the
//               reference's order, writing out[n] (/ sample rate)
// Only the carries between chunks are reassociated.  g, out: [T][E] (a
// wave reads 64 consecutive elements of one frame); reset: [T].
#pragma clang fp contract(off)

#include "internal.h"

namespace dgen {
namespace {

constexpr int kChunk = 256;   // frames per scan chunk
constexpr float kTwoPi = 2.0f * 3.14159265358979323846f;
constexpr int kThreads = 256;

__device__ __forceinline__ bool is_reset(const float* __restrict__ reset, int n) {
  return reset && reset[n] > 0.0f;
}

// The chunk passes read kBatch frames ahead of the additions that use them:
// the carry is one dependent add a frame, so a loop that waited for each
// frame's load ran at one memory latency a frame (the three kernels took
// 219 us at E = 256, T = 65536, 201 MB; batched 59 us).
constexpr int kBatch = 16;

// f(n, g[n][e], reset[n]) for n = n1-1 down to n0, loads a batch at a time.
template <class F>
__device__ __forceinline__ void walk_back(const float* __restrict__ g, const float* __restrict__ reset, int E, int e,
                                          int n0, int n1, F&& f) {
  int n = n1;
  for (; n - kBatch >= n0; n -= kBatch) {
    float gv[kBatch];
    bool rv[kBatch];
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      gv[j] = g[(size_t)(n - 1 - j) * E + e];
      rv[j] = is_reset(reset, n - 1 - j);
    }
#pragma unroll
    for (int j = 0; j < kBatch; ++j) f(n - 1 - j, gv[j], rv[j]);
  }
  for (--n; n >= n0; --n) f(n, g[(size_t)n * E + e], is_reset(reset, n));
}

__global__ __launch_bounds__(kThreads) void k_tg_chunk(const float* __restrict__ g, const float* __restrict__ reset,
                                                       float* __restrict__ gamma, float* __restrict__ alpha, int E,
                                                       int T) {
  const int e = blockIdx.x * kThreads + threadIdx.x, c = blockIdx.y;
  if (e >= E) return;
  const int n0 = c * kChunk, n1 = min(T, n0 + kChunk);
  float carry = 0.0f;
  bool cut = false;
  walk_back(g, reset, E, e, n0, n1, [&](int, float v, bool rs) {
    cut |= rs;
    carry = v + (rs ? 0.0f : carry);
  });
  gamma[(size_t)c * E + e] = carry;
  if (e == 0) alpha[c] = cut ? 0.0f : 1.0f;
}

// Workgroup: 64 elements x kCarryGroups groups of consecutive chunks.  Each
// thread composes its group's maps, the groups are joined in LDS, and each
// thread replays its group from the carry entering it.  (One thread per
// element over all chunks waited out a load batch every 16 chunks: 41 us for
// 256 elements x 256 chunks, 5 us now.)
constexpr int kCarryGroups = 16;
__global__ __launch_bounds__(64 * kCarryGroups) void k_tg_carry(const float* __restrict__ gamma,
                                                                const float* __restrict__ alpha,
                                                                float* __restrict__ carry_in, int E, int C) {
  __shared__ float s_a[kCarryGroups][64], s_g[kCarryGroups][64];
  const int l = threadIdx.x & 63, grp = threadIdx.x >> 6;
  const int e = min((int)blockIdx.x * 64 + l, E - 1);
  const bool live = (int)blockIdx.x * 64 + l < E;
  const int per = (C + kCarryGroups - 1) / kCarryGroups;
  // group grp: chunks hi-1 down to lo, group 0 the last ones
  const int hi = max(0, C - grp * per), lo = max(0, hi - per);
  auto walk = [&](auto&& f) {
    int c = hi;
    for (; c - kBatch >= lo; c -= kBatch) {
      float gv[kBatch], av[kBatch];
#pragma unroll
      for (int j = 0; j < kBatch; ++j) {
        gv[j] = gamma[(size_t)(c - 1 - j) * E + e];
        av[j] = alpha[c - 1 - j];
      }
#pragma unroll
      for (int j = 0; j < kBatch; ++j) f(c - 1 - j, av[j], gv[j]);
    }
    for (--c; c >= lo; --c) f(c, alpha[c], gamma[(size_t)c * E + e]);
  };
  float A = 1.0f, G = 0.0f;
  walk([&](int, float a, float g) {
    A = a * A;
    G = a * G + g;
  });
  s_a[grp][l] = A;
  s_g[grp][l] = G;
  __syncthreads();
  float k = 0.0f;  // nothing follows the last frame
  for (int h = 0; h < grp; ++h) k = s_a[h][l] * k + s_g[h][l];
  walk([&](int c, float a, float g) {
    if (live) carry_in[(size_t)c * E + e] = k;
    k = a * k + g;
  });
}

__global__ __launch_bounds__(kThreads) void k_tg_apply(const float* __restrict__ g, const float* __restrict__ reset,
                                                       const float* __restrict__ carry_in, float* __restrict__ out,
                                                       int E, int T, float sr, int scale) {
  const int e = blockIdx.x * kThreads + threadIdx.x, c = blockIdx.y;
  if (e >= E) return;
  const int n0 = c * kChunk, n1 = min(T, n0 + kChunk);
  float carry = carry_in[(size_t)c * E + e];
  walk_back(g, reset, E, e, n0, n1, [&](int n, float v, bool rs) {
    const float active = rs ? 0.0f : carry;
    out[(size_t)n * E + e] = scale ? active / sr : active;
    carry = v + active;
  });
}

// The swept-phasor bank (Tests/DGenLazyTests/TemporalGradientTests.swift:
// 24-60), one lane per thread: f = base + slope[e] * time[n], the stateful
// phasor of f with reset (u_phasor / u_accum order, Definitions.swift:
// 96-102, 215-246; output = the state before the frame's update), and the
// mse loss against `target` of the phase, or with `smooth` of sin(2 pi
// phase) (continuous across the phase's wraps): per-lane loss sums and the
// upstream gradient of every frame.
__global__ __launch_bounds__(kThreads) void k_swept_phasor(const float* __restrict__ slope,
                                                           const float* __restrict__ time,
                                                           const float* __restrict__ reset, float* __restrict__ phase,
                                                           float* __restrict__ gout, float* __restrict__ lossp, int E,
                                                           int T, float sr, float base, float target, int smooth) {
  const int e = blockIdx.x * kThreads + threadIdx.x;
  if (e >= E) return;
  const float s = slope[e];
  float ph = 0.0f;
  // fp64 loss sum: in fp32, small terms added to a running sum near 2e4
  // (ulp 2e-3) round the same way every frame and bias the loss
  double ls = 0.0;
  for (int n = 0; n < T; ++n) {
    const bool rs = is_reset(reset, n);
    const float f = base + s * time[n];
    const float acc = ph;
    const float next = rs ? 0.0f : acc + f / sr;
    float w = next - floorf(next);
    if (w >= 1.0f) w = w - 1.0f;
    ph = rs ? 0.0f : w;
    // sin / cos of 2 pi acc: the transcendental unit takes revolutions
    const float v = smooth ? sin_2pif_hw(acc) : acc;
    const float d = v - target;
    ls = ls + (double)(d * d);
    if (phase) phase[(size_t)n * E + e] = acc;
    gout[(size_t)n * E + e] = smooth ? 2.0f * d * (cos_2pif_hw(acc) * kTwoPi) : 2.0f * d;
  }
  lossp[e] = (float)ls;
}

// The same bank with a scratch cell [T][E], in passes.  Only the phase
// recurrence is sequential, and it has to round as the reference does, frame
// by frame; the increments before it and the loss after it are not.  One
// thread per lane doing all of it left one wave per 64 lanes issuing ~80
// instructions a frame and waiting out a load each frame: 16.4 ms at
// E = 256, T = 65536.
//   k_sp_inc    every increment (base + slope time) / sr in quads of frames,
//               [group of 64 lanes][T/4][lane][4] in the scratch cell, a reset
//               frame's replaced by kSpReset; and a word per 64-frame interval
//               and group (SpKind) at the start of the upstream cell, which
//               k_sp_apply overwrites
//   k_sp_chain  the phase, one lane per thread.  A plain interval (every
//               increment in [0, 1e30), no reset) is an add and a fract a
//               frame: next >= 0, so next - floor(next) is exact, below 1 and
//               what v_fract_f32 returns; others keep the full wrap and
//               resets.  The phase entering every segment goes into its first
//               quad's word 0, whose increment has been used
//   k_sp_apply  every (lane, segment) replayed from that phase with the sines,
//               the upstream gradient and an fp64 loss sum (words 2-3 of the
//               same quad); k_sp_loss adds a lane's segments
// Segments are the 64-frame intervals, the last one taking a remainder of up
// to 3 frames so that every segment starts on a whole quad.
//
// The chain wave is alone on its SIMD; the two dependent instructions take
// ~9.2 cycles a frame, and 256 bytes have to arrive in that time on each of
// the few CUs that run a chain.  Loading them into registers 192 frames ahead
// (48 KB in flight) left it waiting on memory: 521 us for 65536 frames, 19
// cycles a frame.  So two other waves copy the tape to a 128 KB LDS ring seven
// intervals ahead (load-to-LDS, 112 KB in flight, no registers), and the chain
// reads the next interval from LDS half by half between its steps: 355 us, 13
// cycles a frame (k_sp_inc 18 us, k_sp_apply 26 us, k_sp_loss 8 us).
constexpr int kSpSeg = 64;               // frames per interval and segment
constexpr int kSpQ = kSpSeg / 4;         // quads per interval
constexpr int kSpRing = 8;               // intervals in the LDS ring
constexpr int kSpAhead = kSpRing - 1;    // intervals the copies run ahead
constexpr uint32_t kSpReset = 0x7fc0dead;  // a quiet NaN no increment is stored as
enum SpKind : uint32_t { kSpPlain = 0, kSpOdd = 1, kSpAllReset = 2 };

__host__ __device__ constexpr int sp_segments(int T) { return T < kSpSeg + 4 ? 1 : (T - 4) / kSpSeg + 1; }

__device__ __forceinline__ float sp_wrap(float next) {
  float w = next - floorf(next);
  if (w >= 1.0f) w = w - 1.0f;
  return w;
}

// Quad q of lane e in the tape.
__device__ __forceinline__ size_t sp_quad(int q, int e, int E, int T) {
  const int g = e & ~63;
  return (size_t)g * (T / 4) + (size_t)q * min(64, E - g) + (e - g);
}

// Workgroup: 4 waves = 4 intervals of the same 64 lanes.
__global__ __launch_bounds__(kThreads) void k_sp_inc(const float* __restrict__ slope, const float* __restrict__ time,
                                                     const float* __restrict__ reset, float4* __restrict__ tape,
                                                     uint32_t* __restrict__ kinds, int E, int T, float sr, float base) {
  const int lane = threadIdx.x & 63, e = blockIdx.x * 64 + lane;
  const int iv = __builtin_amdgcn_readfirstlane(blockIdx.y * (kThreads / 64) + (threadIdx.x >> 6));
  const int nint = T / kSpSeg, n0 = iv * kSpSeg;
  if (iv >= nint) return;  // the chain forms a last partial interval itself
  const float s = e < E ? slope[e] : 0.0f;
  const uint64_t rs = __ballot(is_reset(reset, n0 + lane));
  bool plain = rs == 0;
#pragma unroll 4
  for (int q = 0; q < kSpQ; ++q) {
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[j] = (base + s * time[n0 + 4 * q + j]) / sr;
      plain = plain && v[j] >= 0.0f && v[j] < 1e30f;
      if (v[j] != v[j]) v[j] = __builtin_nanf("");
      if ((rs >> (4 * q + j)) & 1) v[j] = __builtin_bit_cast(float, kSpReset);
    }
    if (e < E) tape[sp_quad(n0 / 4 + q, e, E, T)] = make_float4(v[0], v[1], v[2], v[3]);
  }
  const uint64_t odd = __ballot(e < E && !plain);
  if (lane == 0)
    kinds[(size_t)blockIdx.x * nint + iv] = rs == ~uint64_t(0) ? kSpAllReset : (odd ? kSpOdd : kSpPlain);
}

__global__ __launch_bounds__(192) void k_sp_chain(const float* __restrict__ slope, const float* __restrict__ time,
                                                  const float* __restrict__ reset, float4* tape,
                                                  const uint32_t* __restrict__ kinds, int E, int T, float sr,
                                                  float base) {
  __shared__ __align__(16) float4 ring[kSpRing][kSpQ][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ee = blockIdx.x * 64 + lane, e = min(ee, E - 1);
  const int nint = T / kSpSeg, nseg = sp_segments(T);
  if (wave > 0) {
    if (nint == 0) return;
    // wave 1 copies the even quads, wave 2 the odd ones
    auto issue = [&](int iv) {
      const int c = min(iv, nint - 1);
#pragma unroll
      for (int i = 0; i < kSpQ / 2; ++i) {
        const int q = 2 * i + wave - 1;
        __builtin_amdgcn_global_load_lds(tape + sp_quad(c * kSpQ + q, e, E, T),
                                         (__attribute__((address_space(3))) void*)&ring[iv % kSpRing][q][0], 16, 0, 0);
      }
    };
    for (int i = 0; i < kSpAhead; ++i) issue(i);
    // intervals 0 and 1 have landed: the other five still in flight
    asm volatile("s_waitcnt vmcnt(40)" ::: "memory");
    lds_barrier();
    for (int i = 0; i < nint; ++i) {
      issue(i + kSpAhead);  // into the slot of interval i - 1
      // intervals up to i + 2 have landed, i + 3 .. i + 7 in flight
      asm volatile("s_waitcnt vmcnt(40)" ::: "memory");
      lds_barrier();
    }
    // no copy outlives the workgroup's LDS
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    return;
  }
  static_assert(kSpAhead == 7 && kSpQ / 2 == 8, "the waits count 8 copies per wave and interval, 5 intervals in flight");
  float ph = 0.0f;
  auto checkpoint = [&](int n) {
    if (ee < E) reinterpret_cast<float*>(tape + sp_quad(n / 4, e, E, T))[0] = ph;
  };
  if (nint > 0) {
    const uint32_t* kp = kinds + (size_t)blockIdx.x * nint;
    uint32_t kv = kp[min(lane, nint - 1)], kn = 0;  // kinds of 64 intervals, and of the next 64
    float4 v[kSpQ], nv[kSpQ];
    lds_barrier();
#pragma unroll
    for (int q = 0; q < kSpQ; ++q) v[q] = ring[0][q][lane];
    auto interval = [&](int i, float4 (&c)[kSpQ], float4 (&x)[kSpQ]) {
      if (i % 64 == 0) {
        if (i) kv = kn;
        kn = kp[min(i + 64 + lane, nint - 1)];
      }
      const uint32_t kind = __builtin_amdgcn_readlane(kv, i % 64);
      checkpoint(i * kSpSeg);
      const int ns = (i + 1) % kSpRing;  // (past the end: a slot that is not used)
      if (kind == kSpPlain) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
          for (int q = 0; q < kSpQ / 2; ++q) x[h * kSpQ / 2 + q] = ring[ns][h * kSpQ / 2 + q][lane];
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int q = 0; q < kSpQ / 2; ++q) {
            const float4 f = c[h * kSpQ / 2 + q];
            ph = __builtin_amdgcn_fractf(ph + f.x);
            ph = __builtin_amdgcn_fractf(ph + f.y);
            ph = __builtin_amdgcn_fractf(ph + f.z);
            ph = __builtin_amdgcn_fractf(ph + f.w);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
#pragma unroll
        for (int q = 0; q < kSpQ; ++q) x[q] = ring[ns][q][lane];
        if (kind == kSpAllReset) {
          ph = 0.0f;
        } else {
#pragma unroll
          for (int q = 0; q < kSpQ; ++q) {
            const float f[4] = {c[q].x, c[q].y, c[q].z, c[q].w};
#pragma unroll
            for (int j = 0; j < 4; ++j)
              ph = __builtin_bit_cast(uint32_t, f[j]) == kSpReset ? 0.0f : sp_wrap(ph + f[j]);
          }
        }
      }
      lds_barrier();
    };
    int i = 0;
    for (; i + 1 < nint; i += 2) {
      interval(i, v, nv);
      interval(i + 1, nv, v);
    }
    if (i < nint) interval(i, v, nv);
  }
  const float s = slope[e];
  for (int n = nint * kSpSeg; n < T; ++n) {
    if (n % kSpSeg == 0 && n / kSpSeg < nseg) checkpoint(n);
    const float inc = (base + s * time[n]) / sr;
    ph = is_reset(reset, n) ? 0.0f : sp_wrap(ph + inc);
  }
}

__global__ __launch_bounds__(kThreads) void k_sp_apply(const float* __restrict__ slope, const float* __restrict__ time,
                                                       const float* __restrict__ reset, float4* __restrict__ tape,
                                                       float* __restrict__ phase, float* __restrict__ gout, int E,
                                                       int T, float sr, float base, float target, int smooth) {
  const int e = blockIdx.x * 64 + (threadIdx.x & 63);
  const int seg = __builtin_amdgcn_readfirstlane(blockIdx.y * (kThreads / 64) + (threadIdx.x >> 6));
  const int nseg = sp_segments(T);
  if (e >= E || seg >= nseg) return;
  const int n0 = seg * kSpSeg, n1 = seg + 1 < nseg ? n0 + kSpSeg : T;
  float* slot = reinterpret_cast<float*>(tape + sp_quad(n0 / 4, e, E, T));
  float ph = slot[0];
  const float s = slope[e];
  double ls = 0.0;
#pragma unroll 4
  for (int n = n0; n < n1; ++n) {
    const float acc = ph;
    const float inc = (base + s * time[n]) / sr;
    ph = is_reset(reset, n) ? 0.0f : sp_wrap(acc + inc);
    const float v = smooth ? sin_2pif_hw(acc) : acc;
    const float d = v - target;
    ls = ls + (double)(d * d);
    if (phase) phase[(size_t)n * E + e] = acc;
    gout[(size_t)n * E + e] = smooth ? 2.0f * d * (cos_2pif_hw(acc) * kTwoPi) : 2.0f * d;
  }
  *reinterpret_cast<double*>(slot + 2) = ls;
}

// A lane's loss: its segments' fp64 sums, one wave per lane.
__global__ __launch_bounds__(64) void k_sp_loss(const float4* __restrict__ tape, float* __restrict__ lossp, int E,
                                                int T) {
  const int e = blockIdx.x, nseg = sp_segments(T);
  double ls = 0.0;
  for (int g = threadIdx.x; g < nseg; g += 64) {
    const float* slot = reinterpret_cast<const float*>(tape + sp_quad(g * kSpQ, e, E, T));
    ls += *reinterpret_cast<const double*>(slot + 2);
  }
  for (int off = 32; off > 0; off >>= 1) ls += __shfl_xor(ls, off, 64);
  if (threadIdx.x == 0) lossp[e] = (float)ls;
}

}  // namespace

int launch_temporal_grad_scan(const Launch& L, const dgen_hip_op& op) {
  // arg: [0]=g ([T][E]) [1]=reset ([T]) or -1 [2]=out ([T][E]) [3]=E [4]=T [5]=workspace
  //      (2*C*E + C floats, C = ceil(T/256)) [6]=divide by the sample rate (phasor: 1)
  // farg: [0]=sample rate
  const int64_t g = op.arg[0], rs = op.arg[1], out = op.arg[2], E = op.arg[3], T = op.arg[4], ws = op.arg[5],
                scale = op.arg[6];
  DGEN_REQUIRE(E > 0 && E <= (1 << 24) && T > 0 && T < (1ll << 30) && E * T < (1ll << 40) &&
                   (scale == 0 || scale == 1),
               "temporal_grad_scan: E %lld T %lld scale %lld", (long long)E, (long long)T, (long long)scale);
  DGEN_REQUIRE(!scale || (op.farg[0] > 0.f && op.farg[0] < 1e30f), "temporal_grad_scan: sample rate %g",
               (double)op.farg[0]);
  const int64_t C = (T + kChunk - 1) / kChunk;
  DGEN_REQUIRE(C <= 65535, "temporal_grad_scan: %lld chunks", (long long)C);
  DGEN_CHECK_CELL(L, g, E * T, "temporal_grad_scan.g");
  if (rs >= 0) DGEN_CHECK_CELL(L, rs, T, "temporal_grad_scan.reset");
  DGEN_CHECK_CELL(L, out, E * T, "temporal_grad_scan.out");
  DGEN_CHECK_CELL(L, ws, 2 * C * E + C, "temporal_grad_scan.workspace");
  if (L.dry) return 0;
  float* gamma = cell(L, ws);
  float* kin = gamma + C * E;
  float* alpha = kin + C * E;
  const float* r = rs >= 0 ? cell(L, rs) : nullptr;
  const unsigned eb = (unsigned)((E + kThreads - 1) / kThreads);
  hipLaunchKernelGGL(k_tg_chunk, dim3(eb, (unsigned)C), dim3(kThreads), 0, L.stream, cell(L, g), r, gamma, alpha,
                     (int)E, (int)T);
  DGEN_LAUNCH_CHECK("k_tg_chunk");
  hipLaunchKernelGGL(k_tg_carry, dim3((unsigned)((E + 63) / 64)), dim3(64 * kCarryGroups), 0, L.stream, gamma, alpha,
                     kin, (int)E, (int)C);
  DGEN_LAUNCH_CHECK("k_tg_carry");
  hipLaunchKernelGGL(k_tg_apply, dim3(eb, (unsigned)C), dim3(kThreads), 0, L.stream, cell(L, g), r, kin,
                     cell(L, out), (int)E, (int)T, host_rate(L, op.farg[0]), (int)scale);
  DGEN_LAUNCH_CHECK("k_tg_apply");
  return 0;
}

int launch_swept_phasor(const Launch& L, const dgen_hip_op& op) {
  // arg: [0]=slope ([E]) [1]=time ([T]) [2]=reset ([T]) or -1 [3]=phase ([T][E]) or -1 [4]=upstream ([T][E])
  //      [5]=loss partials ([E]) [6]=E [7]=T [8]=smooth (loss on sin(2 pi phase))
  //      [9]=scratch ([T][E], 16-byte aligned) when [10]=1
  // farg: [0]=sample rate [1]=base frequency [2]=target
  const int64_t sl = op.arg[0], tm = op.arg[1], rs = op.arg[2], ph = op.arg[3], gu = op.arg[4], lp = op.arg[5],
                E = op.arg[6], T = op.arg[7], smooth = op.arg[8];
  DGEN_REQUIRE(E > 0 && E <= (1 << 24) && T > 0 && T < (1ll << 30) && E * T < (1ll << 40),
               "swept_phasor: E %lld T %lld", (long long)E, (long long)T);
  DGEN_REQUIRE(op.farg[0] > 0.f && op.farg[0] < 1e30f, "swept_phasor: sample rate %g", (double)op.farg[0]);
  DGEN_CHECK_CELL(L, sl, E, "swept_phasor.slope");
  DGEN_CHECK_CELL(L, tm, T, "swept_phasor.time");
  if (rs >= 0) DGEN_CHECK_CELL(L, rs, T, "swept_phasor.reset");
  if (ph >= 0) DGEN_CHECK_CELL(L, ph, E * T, "swept_phasor.phase");
  DGEN_CHECK_CELL(L, gu, E * T, "swept_phasor.upstream");
  DGEN_CHECK_CELL(L, lp, E, "swept_phasor.loss_partials");
  const bool scratch = op.arg[10] == 1;
  DGEN_REQUIRE(op.arg[10] == 0 || scratch, "swept_phasor: arg[10] %lld (0, or 1 with a scratch cell)",
               (long long)op.arg[10]);
  if (scratch) {
    DGEN_CHECK_CELL(L, op.arg[9], E * T, "swept_phasor.scratch");
    DGEN_REQUIRE(op.arg[9] % 4 == 0, "swept_phasor: scratch cell must be 16-byte aligned");
  }
  if (L.dry) return 0;
  // the passes need one whole quad and their blocks in the grid's second
  // dimension, and read slopes, times, resets and scratch after their first
  // writes; other lengths, ops that write over their inputs and ops without
  // scratch take the one-pass loop
  const int64_t groups = (E + 63) / 64, yblk = (T / kSpSeg + 3) / 4, yseg = (sp_segments((int)T) + 3) / 4;
  const bool apart = scratch && written_apart({{ph, E * T}, {gu, E * T}, {lp, E}, {op.arg[9], E * T}},
                                              {{sl, E}, {tm, T}, {rs, T}});
  if (apart && T >= 4 && yblk <= 65535 && yseg <= 65535) {
    const float sr = host_rate(L, op.farg[0]), base = op.farg[1];
    const float* rp = rs >= 0 ? cell(L, rs) : nullptr;
    float4* tape = reinterpret_cast<float4*>(cell(L, op.arg[9]));
    uint32_t* kinds = reinterpret_cast<uint32_t*>(cell(L, gu));
    if (yblk > 0) {
      hipLaunchKernelGGL(k_sp_inc, dim3((unsigned)groups, (unsigned)yblk), dim3(kThreads), 0, L.stream, cell(L, sl),
                         cell(L, tm), rp, tape, kinds, (int)E, (int)T, sr, base);
      DGEN_LAUNCH_CHECK("k_sp_inc");
    }
    hipLaunchKernelGGL(k_sp_chain, dim3((unsigned)groups), dim3(192), 0, L.stream, cell(L, sl), cell(L, tm), rp, tape,
                       kinds, (int)E, (int)T, sr, base);
    DGEN_LAUNCH_CHECK("k_sp_chain");
    hipLaunchKernelGGL(k_sp_apply, dim3((unsigned)groups, (unsigned)yseg), dim3(kThreads), 0, L.stream, cell(L, sl),
                       cell(L, tm), rp, tape, ph >= 0 ? cell(L, ph) : nullptr, cell(L, gu), (int)E, (int)T, sr, base,
                       op.farg[2], smooth ? 1 : 0);
    DGEN_LAUNCH_CHECK("k_sp_apply");
    hipLaunchKernelGGL(k_sp_loss, dim3((unsigned)E), dim3(64), 0, L.stream, tape, cell(L, lp), (int)E, (int)T);
    DGEN_LAUNCH_CHECK("k_sp_loss");
    return 0;
  }
  hipLaunchKernelGGL(k_swept_phasor, dim3((unsigned)((E + kThreads - 1) / kThreads)), dim3(kThreads), 0, L.stream,
                     cell(L, sl), cell(L, tm), rs >= 0 ? cell(L, rs) : nullptr, ph >= 0 ? cell(L, ph) : nullptr,
                     cell(L, gu), cell(L, lp), (int)E, (int)T, host_rate(L, op.farg[0]), op.farg[1], op.farg[2],
                     smooth ? 1 : 0);
  DGEN_LAUNCH_CHECK("k_swept_phasor");
  return 0;
}

}  // namespace dgen
