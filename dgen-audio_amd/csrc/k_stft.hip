// Hop-gated STFT round trip with learnable per-bin gains, and the gain
// gradient.
//
// Reference graph (the DGenLazy idiom of Tests/DGenLazyTests/
// STFTIdentityTests.swift:152-187): frame = x.buffer(size: N, hop: H)
// .reshape([N]) * hann(N) (bufferView, Sources/DGen/HigherOps.swift:738-792);
// (re, im) = signalTensorFFT(frame) (tensorFFT, HigherOps+FFT.swift:16-34);
// the spectrum times the gains; signalTensorIFFT (:36-59: real part, 1/N);
// overlapAdd(hop: H) (Emit+FFT.swift:6-62), so that
//   y[t] = sum over hop frames h (multiples of H) of z_h[t - h], 0 <= t-h < N,
// where window h holds x[h-N+1 .. h] (zero before frame 0).  The gains
// g[0..N/2] scale the one-sided spectrum as its Hermitian reconstruction:
// bins k and N-k both by g_k.
//
// k_stft_fwd: a workgroup owns an output tile [a0, a0 + kTile) of one signal
// and every window whose outputs reach it (hop frames in (a0-N, a0+kTile)),
// recomputing the few that straddle the tile's left edge instead of
// exchanging partial sums.  A real N-point transform is an N/2-point complex
// FFT (fft_lds.h) plus the even/odd split; after the gains, the Hermitian
// pre-processing and an N/2-point inverse FFT give two real output samples
// per complex value.  W windows (one per M/8-thread slot) are transformed at
// once, and each slot adds its outputs from registers to the tile accumulator
// (read, add, write; windows added at the same time do not overlap, so the
// sum is atomic-free, in an order that neither tile nor batch changes).  The
// tile then yields y, dL/dy = 2 (y - x)/T and its share of the loss sum
// (y - x)^2 / T.
//
// k_stft_bwd: dL/dg_k = sum over windows (c_k/N) Re(X_k conj(E_k)), with X
// the window's spectrum, E the spectrum of dL/dy over the window's outputs
// (zero past T) and c_k = 1 at k = 0, N/2, else 2.  Each workgroup sums a run
// of windows of one signal into a partial row; the column sum reduces them.
#include "fft_lds.h"

namespace dgen {
namespace {

constexpr int kThreads = 256;
constexpr int kTile = 8192;   // output samples owned by a forward workgroup unless the op says fewer
constexpr int kMinTile = 256;
constexpr int kRounds = 8;    // window rounds per backward workgroup unless the op says fewer

struct StftArgs {
  const float* x;      // [S][T]
  const float* win;    // [N]
  const float* gains;  // [N/2 + 1]
  const float* dyin;   // [S][T] (backward)
  float* y;            // [S][T] or null
  float* dy;           // [S][T] or null
  float* lossp;        // [S][ntiles] or null
  float* gpart;        // [S][nblk][N/2 + 1] (backward)
  int S, T, H, ntiles, nblk, tile, rounds;
  int logv;            // windows 2^logv hops apart do not overlap (forward)
  unsigned hmul;       // n / H = n hmul >> hshift for 0 <= n < 2^30 (forward)
  int hshift;
  float invT;
};

// Real N-point spectrum bins k and M-k (k = 0: bins 0 and M) from the
// N/2-point complex transform of the even/odd-packed signal: zk = Z[k],
// zm = Z[(M-k) mod M], wk = exp(-2 pi i k / N).
__device__ __forceinline__ void split_pair(c2 zk, c2 zm, int k, c2 wk, c2& Xk, c2& Xm) {
  const c2 e = {0.5f * (zk.x + zm.x), 0.5f * (zk.y - zm.y)};
  const c2 o = {0.5f * (zk.y + zm.y), 0.5f * (zm.x - zk.x)};
  const c2 wo = cmul(wk, o);
  Xk = cadd(e, wo);
  Xm = k == 0 ? c2{e.x - o.x, 0.0f} : cconj(csub(e, wo));
}

__device__ __forceinline__ float block_sum(float v, float* red) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
  const int wave = threadIdx.x / 64;
  if ((threadIdx.x & 63) == 0) red[wave] = v;
  __syncthreads();
  float t = 0.0f;
  if (threadIdx.x == 0)
    for (int w = 0; w < kThreads / 64; ++w) t += red[w];
  return t;
}

// Two consecutive samples at a 4-byte aligned address, one 8-byte load.
struct __attribute__((packed, aligned(4))) pair {
  float x, y;
};

// What a round costs is its VALU instructions, so everything a thread uses
// again every round (window values, pass and bin-pair twiddles) is in
// registers (within three waves per SIMD), windows inside the signal load
// without bounds tests, and a slot adds its outputs to the tile itself.
//
// The windows covering a sample are added by their residue w mod V, V the power
// of two from N/H on, which differs for any two that overlap: an order that
// depends on the windows' numbers alone, so a signal's y is the same bits
// whatever the tile and the batch.  A tile's windows are taken residue by
// residue, W at a time; those of one residue lie V hops apart, so one barrier
// orders the adds of a round within a residue, and a round that runs into the
// next residue adds one residue after the other.
// (Gathering a round's outputs position by position, 16 x 4 masked LDS reads a
// thread whatever the hop, took half of a round's 1200 instructions: 114 us at
// 8 x 2^20 samples, N = 1024, H = 256; 85 us so.  Slots on consecutive runs of
// windows instead, whose order depends on the tile, took 82.)
template <int LOGN>
__global__ __launch_bounds__(kThreads) void k_stft_fwd(StftArgs a) {
  constexpr int N = 1 << LOGN, M = N / 2, LOGM = LOGN - 1, P = M / 8, W = kThreads / P;
  constexpr int U = M / 2 / P + 1;  // bin pairs per thread
  // a window's P threads lie in one wave when P <= 64: its transforms and
  // bins need only wave-level ordering; the adds to the tile cross slots
  constexpr bool WL = P <= 64;
  static_assert(W * M == 2048, "window slots must fill the FFT buffer");
  extern __shared__ __align__(16) float acc[];  // [tile, whole 64s], sample i at at(i)
  // short windows: up to 16 slots of a wave add at once, N samples apart where H
  // divides N; swapping a block's eights spreads them over the banks (8 x 2^20,
  // N = 64, H = 16: 91 -> 77 us; at N = 256 and more it costs what it gives)
  auto at = [](int i) { return LOGN <= 7 ? i ^ (((i >> 6) & 7) << 3) : i; };
  __shared__ c2 lbuf[2048];
  __shared__ float red[kThreads / 64];
  __shared__ float gain[M + 1];
  const int tid = threadIdx.x, j = tid % P;
  const int slot = P >= 64 ? __builtin_amdgcn_readfirstlane(tid / P) : tid / P;
  const int s = blockIdx.y, tile = blockIdx.x, H = a.H;
  const int a0 = tile * a.tile, a1 = min(a.T, a0 + a.tile);
  const float* xs = a.x + (size_t)s * a.T;
  for (int i = tid; i <= M; i += kThreads) gain[i] = a.gains[i];
  for (int i = tid; i < ((a.tile + 63) & ~63); i += kThreads) acc[i] = 0.0f;
  // windows h = w*H with outputs [h, h+N) meeting [a0, a1)
  auto hops = [&](int n) { return (int)(((uint64_t)(unsigned)n * a.hmul) >> a.hshift); };  // n / H
  const int w_lo = a0 - N < 0 ? 0 : hops(a0 - N) + 1;
  const int w_hi = hops(a1 - 1);
  const SwzBuf buf(lbuf, slot * M);
  const int sj = buf.part(j);
  const HwRegTwiddle<LOGM> tw(j);
  // this thread's bin pairs k = j + u*P, M - k
  c2 wp[U];
#pragma unroll
  for (int u = 0; u < U; ++u) wp[u] = cis(-(float)(j + u * P) / (float)N);
  // The tile's windows in that order, k = 0, 1, ...: before(q) have a residue
  // below q; the first of residue q lies in block (of V) b0 or b0 + 1
  const int logv = a.logv, V = 1 << logv, b0 = w_lo >> logv, rl = w_lo & (V - 1), rh = w_hi & (V - 1);
  const int nw = w_hi - w_lo + 1, blocks = (w_hi >> logv) - b0 + 1;
  auto before = [&](int q) { return q * blocks - min(q, rl) - max(q - rh - 1, 0); };
  auto residue = [&](int k) {
    int q = 0;
    for (int b = V >> 1; b > 0; b >>= 1) q += before(q + b) <= k ? b : 0;
    return q;
  };
  // (a slot past the last window has none)
  auto window = [&](int k, int q) { return k < nw ? ((b0 + (q < rl) + k - before(q)) << logv) + q : w_hi + 1; };
  constexpr float invN = 1.0f / (float)N;
  // the window values this thread multiplies (samples 2n, 2n+1 of its first
  // pass inputs n), in registers for every round
  float2 hw[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int n = in_pos<M, pass_radix(LOGM, 0)>(j, e);
    hw[e] = float2{a.win[2 * n], a.win[2 * n + 1]};
  }
  // this thread's samples of window w (element e of the first pass
  // needs samples 2n and 2n+1 of the window, n = in_pos(j, e)); the next
  // round's are loaded while this one is transformed
  float px[16];
  auto fetch = [&](int w) {
    const int h = w * H, t00 = h - N + 1 + 2 * j;
    if (__ballot(w > w_hi || h < N - 1) == 0) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const pair v = *reinterpret_cast<const pair*>(xs + t00 + 2 * in_off<M, pass_radix(LOGM, 0)>(e));
        px[2 * e] = v.x;
        px[2 * e + 1] = v.y;
      }
      return;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int t0 = t00 + 2 * in_off<M, pass_radix(LOGM, 0)>(e);
      px[2 * e] = w <= w_hi && t0 >= 0 ? xs[t0] : 0.0f;
      px[2 * e + 1] = w <= w_hi && t0 + 1 >= 0 ? xs[t0 + 1] : 0.0f;
    }
  };
  // adds this thread's outputs of window w (complex output q holds samples
  // 2q, 2q+1) to the tile
  auto add = [&](int w, const c2 (&v)[8], const int (&op)[8]) {
    const int h = w * H, o = h - a0;
    const bool whole = w <= w_hi && o >= 0 && h + N <= a1;
    // pairs of the tile are 8-byte aligned where o is even: even hops from an
    // even tile start
    if (__ballot(!whole) == 0 && (H | a0) % 2 == 0) {
#pragma unroll
      for (int e0 = 0; e0 < 8; e0 += 4) {
        float2 t[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) t[e] = *reinterpret_cast<const float2*>(acc + at(o + 2 * op[e0 + e]));
#pragma unroll
        for (int e = 0; e < 4; ++e)
          *reinterpret_cast<float2*>(acc + at(o + 2 * op[e0 + e])) =
              float2{t[e].x + v[e0 + e].x * invN, t[e].y + v[e0 + e].y * invN};
        __builtin_amdgcn_sched_barrier(0);
      }
      return;
    }
    if (w > w_hi) return;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int i = o + 2 * op[e];
      if (i >= 0 && i < a1 - a0) acc[at(i)] += v[e].x * invN;
      if (i + 1 >= 0 && i + 1 < a1 - a0) acc[at(i + 1)] += v[e].y * invN;
    }
  };
  __syncthreads();
  int q = residue(slot), w = window(slot, q);
  int u = blocks == 1 ? rl : 0, end = before(u + 1);  // slot 0's residue, and its windows' end
  fetch(w);
  for (int k0 = 0; k0 < nw; k0 += W) {
    c2 v[8];
    int op[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = c2{px[2 * e] * hw[e].x, px[2 * e + 1] * hw[e].y};
    fft<LOGM, false, WL>(buf, j, v, op, tw);
    const int wc = w, qc = q;  // this round's, for its adds
    if (k0 + W < nw) {
      if (k0 + 2 * W <= end) {
        w += W << logv;
      } else {
        q = residue(k0 + W + slot);
        w = window(k0 + W + slot, q);
      }
      fetch(w);
    }
    fft_store<LOGM>(buf, j, v);
    lds_sync<WL>();
    // gains on the one-sided spectrum, then the Hermitian inverse
    // pre-processing: z'_k = (G_k + conj G_{M-k}) + i (G_k - conj G_{M-k}) W_N^{-k}
    // (each thread owns the pairs k, M-k with k = j + u*P, so the update is
    // in place; all of a thread's spectrum reads are issued first)
    c2 zk[U], zm[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      // k = j + u*P < M for every u (pairs past M/2 are read and skipped)
      zk[u] = buf.at(sj, u * P);
      zm[u] = buf[(M - j - u * P) & (M - 1)];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = j + u * P;
      if (k > M / 2) continue;
      c2 Xk, Xm;
      const c2 wk = wp[u];
      split_pair(zk[u], zm[u], k, wk, Xk, Xm);
      const float gk = gain[k], gm = gain[M - k];
      Xk = c2{Xk.x * gk, Xk.y * gk};
      Xm = c2{Xm.x * gm, Xm.y * gm};
      if (k == 0) {
        buf[0] = c2{Xk.x + Xm.x, Xk.x - Xm.x};
      } else {
        const c2 o1 = cmul(c2{Xk.x - Xm.x, Xk.y + Xm.y}, cconj(wk));
        buf[k] = c2{(Xk.x + Xm.x) - o1.y, (Xk.y - Xm.y) + o1.x};
        if (k != M - k) {
          const c2 o2 = cmul(c2{Xm.x - Xk.x, Xm.y + Xk.y}, c2{-wk.x, -wk.y});
          buf[M - k] = c2{(Xm.x + Xk.x) - o2.y, (Xm.y - Xk.y) + o2.x};
        }
      }
    }
    lds_sync<WL>();
    fft_load<LOGM>(buf, j, v);
    lds_sync<WL>();
    fft<LOGM, true, WL>(buf, j, v, op, tw);
    // a residue's adds at a time
    const int kn = min(k0 + W, nw);
    for (bool more = true; more;) {
      if (qc == u) add(wc, v, op);
      lds_barrier();
      more = end < kn;
      if (end <= kn && end < nw) {
        ++u;
        if (before(u + 1) == end) u = rl;  // only residues between rh and rl have no windows
        end = before(u + 1);
      }
    }
  }
  float ls = 0.0f;
  // the tile's input samples are loaded 8 at a time, all in flight before use
  for (int t8 = a0 + tid; t8 < a1; t8 += 8 * kThreads) {
    float xv[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) xv[q] = xs[min(t8 + q * kThreads, a1 - 1)];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int t = t8 + q * kThreads;
      if (t >= a1) break;
      const float yv = acc[at(t - a0)];
      const float d = yv - xv[q];
      const size_t i = (size_t)s * a.T + t;
      if (a.y) a.y[i] = yv;
      if (a.dy) a.dy[i] = 2.0f * d * a.invT;
      ls += d * d;
    }
  }
  if (a.lossp) {
    const float tot = block_sum(ls, red);
    if (tid == 0) a.lossp[(size_t)s * a.ntiles + tile] = tot * a.invT;
  }
}

struct BwdLds {
  c2 buf[2048];
  c2 aux[2048];
};

// (held to four waves per SIMD up to N = 1024, for 3 spilled registers at N =
// 512 and one at 1024: 53 -> 46 us at 8 x 2^20, N = 1024; at 2048 far more spill)
template <int LOGN>
__global__ __launch_bounds__(kThreads, LOGN <= 10 ? 4 : 2) void k_stft_bwd(StftArgs a) {
  constexpr int N = 1 << LOGN, M = N / 2, LOGM = LOGN - 1, P = M / 8, W = kThreads / P;
  constexpr int U = M / 2 / P + 1;  // bin pairs per thread
  constexpr bool WL = P <= 64;       // a window's threads lie in one wave
  static_assert(W * M == 2048, "window slots must fill the FFT buffer");
  __shared__ BwdLds L;
  const int tid = threadIdx.x, slot = tid / P, j = tid % P;
  const int s = blockIdx.y, blk = blockIdx.x, H = a.H;
  const int nwin = (a.T + H - 1) / H;
  const int wb = blk * a.rounds * W, we = min(nwin, wb + a.rounds * W);
  const float* xs = a.x + (size_t)s * a.T;
  const float* gs = a.dyin + (size_t)s * a.T;
  const SwzBuf buf(L.buf, slot * M);
  const SwzBuf spec(L.aux, slot * M);
  // the window values this thread multiplies, in registers for every round
  float2 hw[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int n = in_pos<M, pass_radix(LOGM, 0)>(j, e);
    hw[e] = float2{a.win[2 * n], a.win[2 * n + 1]};
  }
  constexpr float invN = 1.0f / (float)N;
  const HwRegTwiddle<LOGM> tw(j);
  c2 wp[U];
#pragma unroll
  for (int u = 0; u < U; ++u) wp[u] = cis(-(float)(j + u * P) / (float)N);
  float acc_k[U], acc_m[U];
#pragma unroll
  for (int u = 0; u < U; ++u) acc_k[u] = acc_m[u] = 0.0f;
  __syncthreads();
  for (int r0 = 0; r0 < we - wb; r0 += W) {
    const int w = wb + r0 + slot;
    const bool live = w < we;
    const int h = w * H;
    {
      // the analysis window x[h-N+1 .. h] * hann (-> spec) and dL/dy over
      // the window's outputs [h, h+N) (-> buf), transformed together
      c2 vx[8], vg[8];
      int op[8];
      const int t00 = h - N + 1 + 2 * j, g00 = h + 2 * j;
      if (__ballot(!live || h < N - 1 || h + N > a.T) == 0) {  // inside the signal: no bounds tests
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int off = 2 * in_off<M, pass_radix(LOGM, 0)>(e);
          const pair x = *reinterpret_cast<const pair*>(xs + t00 + off);
          const pair g = *reinterpret_cast<const pair*>(gs + g00 + off);
          vx[e] = c2{x.x * hw[e].x, x.y * hw[e].y};
          vg[e] = c2{g.x, g.y};
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int off = 2 * in_off<M, pass_radix(LOGM, 0)>(e), t0 = t00 + off, g0 = g00 + off;
          const float x0 = live && t0 >= 0 ? xs[t0] : 0.0f;
          const float x1 = live && t0 + 1 >= 0 ? xs[t0 + 1] : 0.0f;
          vx[e] = c2{x0 * hw[e].x, x1 * hw[e].y};
          vg[e] = c2{live && g0 < a.T ? gs[g0] : 0.0f, live && g0 + 1 < a.T ? gs[g0 + 1] : 0.0f};
        }
      }
      fft2<LOGM, false, WL>(spec, buf, j, vx, vg, op, tw);
      fft_store<LOGM>(spec, j, vx);
      fft_store<LOGM>(buf, j, vg);
      lds_sync<WL>();
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = j + u * P;
      if (k > M / 2) break;
      c2 Xk, Xm, Ek, Em;
      const int km = (M - k) & (M - 1);
      split_pair(spec[k], spec[km], k, wp[u], Xk, Xm);
      split_pair(buf[k], buf[km], k, wp[u], Ek, Em);
      acc_k[u] += Xk.x * Ek.x + Xk.y * Ek.y;
      acc_m[u] += Xm.x * Em.x + Xm.y * Em.y;
    }
    // the next round overwrites this slot's buffers
    lds_sync<WL>();
  }
  // every slot's reads are done before the partial rows reuse the buffers
  lds_barrier();
  // slots' partial sums -> one row: bins k (acc_k) and M-k (acc_m; bin M for k = 0)
  float* part = reinterpret_cast<float*>(L.buf);  // [W][M + 1]
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int k = j + u * P;
    if (k > M / 2) break;
    part[slot * (M + 1) + k] = acc_k[u];
    if (M - k != k) part[slot * (M + 1) + M - k] = acc_m[u];
  }
  lds_barrier();
  float* row = a.gpart + ((size_t)s * a.nblk + blk) * (M + 1);
  for (int b = tid; b <= M; b += kThreads) {
    float t = 0.0f;
    for (int q = 0; q < W; ++q) t += part[q * (M + 1) + b];
    const float ck = (b == 0 || b == M) ? 1.0f : 2.0f;
    row[b] = t * ck * invN;
  }
}

using StftKernel = void (*)(StftArgs);

StftKernel fwd_kernel(int logn) {
  switch (logn) {
    case 6: return k_stft_fwd<6>;
    case 7: return k_stft_fwd<7>;
    case 8: return k_stft_fwd<8>;
    case 9: return k_stft_fwd<9>;
    case 10: return k_stft_fwd<10>;
    case 11: return k_stft_fwd<11>;
    default: return nullptr;
  }
}

StftKernel bwd_kernel(int logn) {
  switch (logn) {
    case 6: return k_stft_bwd<6>;
    case 7: return k_stft_bwd<7>;
    case 8: return k_stft_bwd<8>;
    case 9: return k_stft_bwd<9>;
    case 10: return k_stft_bwd<10>;
    case 11: return k_stft_bwd<11>;
    default: return nullptr;
  }
}

int stft_shape(int64_t S, int64_t T, int64_t N, int64_t H, int& logn, const char* who) {
  logn = 0;
  while ((1ll << logn) < N) ++logn;
  DGEN_REQUIRE((1ll << logn) == N && logn >= 6 && logn <= 11, "%s: N %lld must be a power of two in [64, 2048]",
               who, (long long)N);
  DGEN_REQUIRE(S > 0 && S <= 65535 && T > 0 && T < (1ll << 30) && H >= 1 && H <= N,
               "%s: S %lld T %lld H %lld", who, (long long)S, (long long)T, (long long)H);
  return 0;
}

}  // namespace

int launch_stft_fwd(const Launch& L, const dgen_hip_op& op) {
  const int64_t x = op.arg[0], win = op.arg[1], gains = op.arg[2], y = op.arg[3], dy = op.arg[4], lossp = op.arg[5];
  const int64_t S = op.arg[6], T = op.arg[7], N = op.arg[8], H = op.arg[9];
  int logn;
  if (int rc = stft_shape(S, T, N, H, logn, "stft_fwd")) return rc;
  const int64_t tile = op.arg[10] ? op.arg[10] : kTile;
  DGEN_REQUIRE(tile >= kMinTile && tile <= kTile, "stft_fwd: tile %lld outside [%d, %d]", (long long)tile, kMinTile,
               kTile);
  const int64_t ntiles = (T + tile - 1) / tile;
  DGEN_CHECK_CELL(L, x, S * T, "stft_fwd.x");
  DGEN_CHECK_CELL(L, win, N, "stft_fwd.window");
  DGEN_CHECK_CELL(L, gains, N / 2 + 1, "stft_fwd.gains");
  if (y >= 0) DGEN_CHECK_CELL(L, y, S * T, "stft_fwd.y");
  if (dy >= 0) DGEN_CHECK_CELL(L, dy, S * T, "stft_fwd.dy");
  if (lossp >= 0) DGEN_CHECK_CELL(L, lossp, S * ntiles, "stft_fwd.loss_partials");
  DGEN_REQUIRE(ntiles <= (1ll << 31) - 1, "stft_fwd: too many tiles");
  if (L.dry) return 0;
  StftArgs a{};
  a.x = cell(L, x);
  a.win = cell(L, win);
  a.gains = cell(L, gains);
  a.y = y >= 0 ? cell(L, y) : nullptr;
  a.dy = dy >= 0 ? cell(L, dy) : nullptr;
  a.lossp = lossp >= 0 ? cell(L, lossp) : nullptr;
  a.S = (int)S;
  a.T = (int)T;
  a.H = (int)H;
  a.ntiles = (int)ntiles;
  a.tile = (int)tile;
  while ((H << a.logv) < N) ++a.logv;
  // (hmul H exceeds 2^hshift by less than H <= 2^(hshift - 30))
  a.hshift = 30;
  while ((1ll << (a.hshift - 30)) < H) ++a.hshift;
  a.hmul = (unsigned)(((1ll << a.hshift) + H - 1) / H);
  a.invT = 1.0f / (float)T;
  hipLaunchKernelGGL(fwd_kernel(logn), dim3((unsigned)ntiles, (unsigned)S), dim3(kThreads),
                     (unsigned)((tile + 63) / 64 * 64 * sizeof(float)), L.stream, a);
  DGEN_LAUNCH_CHECK("k_stft_fwd");
  return 0;
}

int launch_stft_bwd(const Launch& L, const dgen_hip_op& op) {
  const int64_t x = op.arg[0], win = op.arg[1], dy = op.arg[2], gpart = op.arg[3];
  const int64_t S = op.arg[4], T = op.arg[5], N = op.arg[6], H = op.arg[7];
  int logn;
  if (int rc = stft_shape(S, T, N, H, logn, "stft_bwd")) return rc;
  const int64_t nwin = (T + H - 1) / H;
  const int64_t rounds = op.arg[8] ? op.arg[8] : kRounds;
  DGEN_REQUIRE(rounds >= 1 && rounds <= kRounds, "stft_bwd: rounds %lld outside [1, %d]", (long long)rounds, kRounds);
  const int64_t wpb = rounds * (kThreads * 16 / N);
  const int64_t nblk = (nwin + wpb - 1) / wpb;
  DGEN_CHECK_CELL(L, x, S * T, "stft_bwd.x");
  DGEN_CHECK_CELL(L, win, N, "stft_bwd.window");
  DGEN_CHECK_CELL(L, dy, S * T, "stft_bwd.dy");
  DGEN_CHECK_CELL(L, gpart, S * nblk * (N / 2 + 1), "stft_bwd.grad_partials");
  if (L.dry) return 0;
  StftArgs a{};
  a.x = cell(L, x);
  a.win = cell(L, win);
  a.dyin = cell(L, dy);
  a.gpart = cell(L, gpart);
  a.S = (int)S;
  a.T = (int)T;
  a.H = (int)H;
  a.nblk = (int)nblk;
  a.rounds = (int)rounds;
  hipLaunchKernelGGL(bwd_kernel(logn), dim3((unsigned)nblk, (unsigned)S), dim3(kThreads), 0, L.stream, a);
  DGEN_LAUNCH_CHECK("k_stft_bwd");
  return 0;
}

}  // namespace dgen
