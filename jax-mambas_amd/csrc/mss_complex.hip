// Complex-SSM selective scan (forward and backward) for gfx950 (MI355X).
//
// Reference behaviour followed: the complex-state branch of S6 (mamba/mamba1.py:143-176):
// A = -exp(A_log.real) + i*A_imag (the caller applies that parameterisation),
// a_bar = exp(delta*A), Euler b_bar = delta*B (real) or ZOH b_bar = expm1(delta*A)/A*B
// (complex), an affine associative scan over complex states from a zero state, then
// y = sum_n C*Re(h) + D*u (``ys.real``, :175-198). The same fusions as the real scan run
// inside the kernels: softplus(delta + bias), the padding mask, the silu(z) gate, an
// optional initial state (zero reproduces the reference) and the last state. The reference
// runs this branch as an XLA associative scan and differentiates it with autodiff; the
// backward here is a hand-written adjoint that treats each complex state as a real
// 2-vector, so the transpose of multiplication by a_bar is multiplication by conj(a_bar).
//
// Mapping, as the real kernels: one wave per (batch, channel), a lane owns one 8-step
// segment, a wave pass covers a 512-step chunk, and segments are joined by a 64-lane
// inclusive scan of complex affine maps on DPP lane shifts. exp(delta*A) is
// exp2(delta*Re(A)*log2(e)) * (cos, sin)(delta*Im(A)), the angle taken in turns
// (delta*Im(A)/2pi) for the hardware sine and cosine.
#include "mss_common.h"

namespace mss {

constexpr int kCT = kSegSteps;     // steps per lane: one carry segment
constexpr int kCChunk = 64 * kCT;  // steps per wave pass
static_assert(kCChunk == kPartChunk, "the reduction's chunk is the scan's");
constexpr int kCFwdW = 4;          // waves (channels) per forward workgroup
constexpr int kCBwdW = 12;         // waves per backward workgroup (3 per SIMD, one per CU)
constexpr int kCMaxChan = 48;      // channels one backward workgroup walks, at most
// dB/dC accumulator rows of the backward: ceil(kCBwdW/N) copies of each state's row, so
// waves never share a row within one state iteration; the most over N <= 16 is 22 (N = 11).
constexpr int kCAccRows = 22;
constexpr float kInv2Pi = 0.15915494309189535f;

// Constants of exp(t * A) for one (channel, state).
struct CoefA {
  float ar2;    // Re(A) * log2(e)
  float airev;  // Im(A) / (2 pi)
  float ar, ai; // A
  float inv_a2; // 1 / |A|^2 (ZOH)
};

__device__ __forceinline__ CoefA coef_of(float2 a) {
  CoefA c;
  c.ar = a.x;
  c.ai = a.y;
  c.ar2 = c.ar * kLog2e;
  c.airev = c.ai * kInv2Pi;
  c.inv_a2 = 1.f / __builtin_fmaf(c.ar, c.ar, c.ai * c.ai);
  return c;
}
__device__ __forceinline__ CoefA load_coef(const float* __restrict__ A, size_t idx) {
  return coef_of(reinterpret_cast<const float2*>(A)[idx]);
}

// exp(t * A) = m * (cy + i sy), m = exp(t Re A).
struct CExp {
  float m, cy, sy;
};

// The angle t Im(A) in turns, reduced to [0, 1) by fract (exact), feeds the hardware
// sine and cosine (which take turns): measured on MI355X against float64 over [-8, 8]
// turns, their absolute error is at most 1.2e-7 (about one ulp of 1).
__device__ __forceinline__ CExp cexp_t(float t, const CoefA& c) {
  CExp e;
  e.m = fast_exp2(t * c.ar2);
  const float rev = __builtin_amdgcn_fractf(t * c.airev);
  e.cy = __builtin_amdgcn_cosf(rev);
  e.sy = __builtin_amdgcn_sinf(rev);
  return e;
}

// E = expm1(t A) / A (the ZOH b_bar without B) from exp(t A)'s parts. Re expm1(tA) =
// expm1(t Re A) cos y + (cos y - 1) with both terms <= 0 for t >= 0 (no cancellation
// between them), and cos y - 1 = -sin^2 y / (1 + cos y) where cos y > 0 (no cancellation
// near y = 0); Im expm1(tA) = exp(t Re A) sin y.
__device__ __forceinline__ void zoh_e(float t, const CoefA& c, const CExp& x, float& er, float& ei) {
  const float em1 = expm1f(t * c.ar);
  const float cm1 = x.cy > 0.f ? -x.sy * x.sy * fast_rcp(1.f + x.cy) : x.cy - 1.f;
  const float xr = __builtin_fmaf(em1, x.cy, cm1);
  const float xi = x.m * x.sy;
  er = __builtin_fmaf(xr, c.ar, xi * c.ai) * c.inv_a2;
  ei = __builtin_fmaf(xi, c.ar, -xr * c.ai) * c.inv_a2;
}

// One step of the 64-lane inclusive scan of complex affine maps x -> P x + H: the lane
// combines the map of the lane kCtrl selects (earlier in lane order, identity where there
// is none) with its own: (Pl, Hl) then (P, H) gives (Pl P, P Hl + H).
template <int kCtrl, int kRowMask>
__device__ __forceinline__ void caffine_step(float& pr, float& pi, float& hr, float& hi) {
  const float lpr = dpp_mov<kCtrl, kRowMask>(1.f, pr);
  const float lpi = dpp_mov<kCtrl, kRowMask>(0.f, pi);
  const float lhr = dpp_mov<kCtrl, kRowMask>(0.f, hr);
  const float lhi = dpp_mov<kCtrl, kRowMask>(0.f, hi);
  const float nhr = __builtin_fmaf(pr, lhr, __builtin_fmaf(-pi, lhi, hr));
  const float nhi = __builtin_fmaf(pr, lhi, __builtin_fmaf(pi, lhr, hi));
  const float npr = __builtin_fmaf(pr, lpr, -pi * lpi);
  const float npi = __builtin_fmaf(pr, lpi, pi * lpr);
  hr = nhr;
  hi = nhi;
  pr = npr;
  pi = npi;
}

__device__ __forceinline__ void wave_scan_caffine(float& pr, float& pi, float& hr, float& hi) {
  caffine_step<kRowShr1, 0xF>(pr, pi, hr, hi);
  caffine_step<kRowShr2, 0xF>(pr, pi, hr, hi);
  caffine_step<kRowShr4, 0xF>(pr, pi, hr, hi);
  caffine_step<kRowShr8, 0xF>(pr, pi, hr, hi);
  caffine_step<kRowBcast15, 0xA>(pr, pi, hr, hi);
  caffine_step<kRowBcast31, 0xC>(pr, pi, hr, hi);
}

// ---------------------------------------------------------------------------------
// Forward. Workgroup = kCFwdW waves over kCFwdW / kG channels of one batch row; kG = 1: no LDS, no
// block barriers. The running state of state n (entering the current chunk) is kept by lane n as
// (run_r, run_i). kG > 1: that many waves share a channel, each taking every kG-th state, their
// outputs added in order through LDS at the end of a chunk; the row may be split in time as well
// (FwdParams::split_map, here complex: [n_split - 1][batch][dim][dstate][P re, im, H re, im]).
template <bool kZOH, typename io_t, typename bc_t, int kRows, int kG>
__global__ __launch_bounds__(kCFwdW * 64) void cfwd_kernel(FwdParams p) {
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int b = row_longest_first(p.seq_lens, p.batch, p.seqlen, blockIdx.y);
  const int d = blockIdx.x * (kCFwdW / kG) + w / kG;
  const int grp = w % kG;
  static_assert(kG == 1 || kG == kCFwdW, "a workgroup leaves as one where it has barriers");
  __shared__ float s_y[kG > 1 ? kG : 1][kG > 1 ? kCT : 1][kG > 1 ? 65 : 1];  // partial outputs [wave][step][lane]
  if (d >= p.dim) return;
  const int L = p.seqlen;
  const int N = p.dstate;
  const int len = p.seq_lens ? min(max(p.seq_lens[b], 0), L) : L;
  const size_t chan = static_cast<size_t>(b) * p.dim + d;
  const long long row = b * p.io_sb + d * p.io_sd;
  const io_t* __restrict__ u_row = static_cast<const io_t*>(p.u) + row;
  const io_t* __restrict__ dl_row = static_cast<const io_t*>(p.delta) + row;
  io_t* __restrict__ out_row = static_cast<io_t*>(p.out) + row;
  const bc_t* __restrict__ Bb = static_cast<const bc_t*>(p.B) + b * p.bc_sb;
  const bc_t* __restrict__ Cb = static_cast<const bc_t*>(p.C) + b * p.bc_sb;
  const float Dv = p.D ? p.D[d] : 0.f;
  const float bias = p.delta_bias ? p.delta_bias[d] : 0.f;

  float run_r = 0.f, run_i = 0.f;
  if (p.x0 && lane < N) {
    run_r = p.x0[(chan * N + lane) * 2];
    run_i = p.x0[(chan * N + lane) * 2 + 1];
  }
  const int n_chunks = (L + kCChunk - 1) / kCChunk;
  const int n_live = (len + kCChunk - 1) / kCChunk;
  const int c_lo = kG > 1 ? blockIdx.z * p.chunks_per_split : 0;
  const int c_end = kG > 1 ? min(n_chunks, c_lo + p.chunks_per_split) : n_chunks;
  if constexpr (kG > 1) {
    if (lane < N) {  // the state through the splits to the left (those past the length keep it)
      const float4* map = reinterpret_cast<const float4*>(p.split_map) + chan * N + lane;
      const size_t m_ld = static_cast<size_t>(p.batch) * p.dim * N;
      const int m_end = min(static_cast<int>(blockIdx.z), (n_live + p.chunks_per_split - 1) / p.chunks_per_split);
      for (int m = 0; m < m_end; ++m) through_map(map[m * m_ld], run_r, run_i);
    }
  }
  for (int c = c_lo; c < c_end; ++c) {
    const int t0 = c * kCChunk;
    const int tl = t0 + lane * kCT;
    const bool fast = kRows == kWholeRows || t0 + kCChunk <= L;
    float y[kCT];
    if (c >= n_live) {
      // The whole chunk is past this row's length: the state is frozen, the output zero
      // (the backward reads no residual here, so y_pre is left unwritten).
#pragma unroll
      for (int j = 0; j < kCT; ++j) y[j] = 0.f;
      if (grp == 0) store_seg<kCT>(out_row, tl, L, fast, y, kRows);
      continue;
    }
    float dlt[kCT], uu[kCT];
    float ssum = 0.f;
    Seg<kCT, io_t> sd, su;
    fetch(sd, dl_row, tl, L, kRows);
    fetch(su, u_row, tl, L, kRows);
    finish(sd, tl, L, fast, dlt, kRows);
    finish(su, tl, L, fast, uu, kRows);
#pragma unroll
    for (int j = 0; j < kCT; ++j) {
      const bool valid = tl + j < len;
      const float x = dlt[j] + bias;
      const float dv = p.delta_softplus ? softplus(x) : x;
      dlt[j] = valid ? dv : 0.f;
      uu[j] = valid ? uu[j] : 0.f;
      y[j] = grp == 0 ? Dv * uu[j] : 0.f;
      ssum += dlt[j];
    }
    // B and C rows of the next state are loaded one state ahead,
    Seg<kCT, bc_t> sbn, scn;
    if (grp < N) {
      fetch(sbn, Bb + grp * p.bc_sn, tl, L, kRows);
      fetch(scn, Cb + grp * p.bc_sn, tl, L, kRows);
    }
    // and A: loaded in its own iteration, its latency preceded every state's work (measured on
    // MI355X, B=4 D=1536 L=2048 N=16 float32 262 -> 257 us, B=8 with bf16 rows 473 -> 460).
    const float2* __restrict__ Ad = reinterpret_cast<const float2*>(p.A) + static_cast<size_t>(d) * N;
    float2 an = grp < N ? Ad[grp] : make_float2(0.f, 0.f);
    for (int n = grp; n < N; n += kG) {
      const CoefA cf = coef_of(an);
      float ar[kCT], ai[kCT], br[kCT], bi[kCT];
      float bv[kCT], cv[kCT];
      finish(sbn, tl, L, fast, bv, kRows);
      finish(scn, tl, L, fast, cv, kRows);
      if (n + kG < N) {
        fetch(sbn, Bb + (n + kG) * p.bc_sn, tl, L, kRows);
        fetch(scn, Cb + (n + kG) * p.bc_sn, tl, L, kRows);
        an = Ad[n + kG];
      }
      float hr = 0.f, hi = 0.f;
      {
#pragma unroll
        for (int j = 0; j < kCT; ++j) {
          const CExp e = cexp_t(dlt[j], cf);
          const bool valid = tl + j < len;
          ar[j] = valid ? e.m * e.cy : 1.f;
          ai[j] = valid ? e.m * e.sy : 0.f;
          if constexpr (kZOH) {
            float er, ei;
            zoh_e(dlt[j], cf, e, er, ei);
            const float s = bv[j] * uu[j];
            br[j] = er * s;
            bi[j] = ei * s;
          } else {
            br[j] = dlt[j] * uu[j] * bv[j];
            bi[j] = 0.f;
          }
          const float nr = __builtin_fmaf(ar[j], hr, __builtin_fmaf(-ai[j], hi, br[j]));
          const float ni = __builtin_fmaf(ar[j], hi, __builtin_fmaf(ai[j], hr, bi[j]));
          hr = nr;
          hi = ni;
        }
      }
      // Segment map h -> P h + H, P = exp(A * sum delta); scanned over the lanes.
      const CExp pe = cexp_t(ssum, cf);
      float pr = pe.m * pe.cy, pim = pe.m * pe.sy;
      wave_scan_caffine(pr, pim, hr, hi);
      const float rr = readlane(run_r, n), ri = readlane(run_i, n);
      // State at the lane's last step, then the previous lane's as this lane's carry-in.
      const float er = __builtin_fmaf(pr, rr, __builtin_fmaf(-pim, ri, hr));
      const float ei = __builtin_fmaf(pr, ri, __builtin_fmaf(pim, rr, hi));
      float xr = dpp_mov<kWaveShr1, 0xF>(rr, er);
      float xi = dpp_mov<kWaveShr1, 0xF>(ri, ei);
      if (lane == 0) {
        xr = rr;
        xi = ri;
      }
      if (p.carries && (kRows == kWholeRows || tl < L)) {
        float2* cp = reinterpret_cast<float2*>(p.carries) + (chan * N + n) * p.n_seg + tl / kCT;
        *cp = make_float2(xr, xi);
      }
      {
#pragma unroll
        for (int j = 0; j < kCT; ++j) {
          const float nr = __builtin_fmaf(ar[j], xr, __builtin_fmaf(-ai[j], xi, br[j]));
          const float ni = __builtin_fmaf(ar[j], xi, __builtin_fmaf(ai[j], xr, bi[j]));
          xr = nr;
          xi = ni;
          y[j] = __builtin_fmaf(cv[j], xr, y[j]);
        }
      }
      const float nr = readlane(er, 63), ni = readlane(ei, 63);
      run_r = lane == n ? nr : run_r;
      run_i = lane == n ? ni : run_i;
    }
    if constexpr (kG > 1) {
      // Each wave finishes kV steps a lane: steps [grp, grp + 1) * 64 * kV of the chunk.
      constexpr int kV = kCT / kG;
      const int tc = (grp * 64 + lane) * kV;
      const int t = t0 + tc;
      float zv[kV];
      if (p.z) {
#pragma unroll
        for (int e = 0; e < kV; ++e)
          zv[e] = (kRows == kWholeRows || t + e < L) ? to_f32((static_cast<const io_t*>(p.z) + row)[t + e]) : 0.f;
      }
      __syncthreads();  // the previous chunk's partial outputs have been read
#pragma unroll
      for (int j = 0; j < kCT; ++j) s_y[grp][j][lane] = y[j];
      __syncthreads();
#pragma unroll
      for (int e = 0; e < kV; ++e) {
        float v = 0.f;
#pragma unroll
        for (int q = 0; q < kG; ++q) v += s_y[q][(tc + e) % kCT][(tc + e) / kCT];
        v = t + e < len ? v : 0.f;
        if (kRows == kWholeRows || t + e < L) {
          if (p.z) {
            if (p.y_pre) store_as(static_cast<io_t*>(p.y_pre) + row + t + e, v);
            v = t + e < len ? v * (zv[e] * sigmoid(zv[e])) : 0.f;
          }
          store_as(out_row + t + e, v);
        }
      }
      continue;
    }
    if (p.z) {
      if (p.y_pre) {
        float yp[kCT];
#pragma unroll
        for (int j = 0; j < kCT; ++j) yp[j] = (tl + j < len) ? y[j] : 0.f;
        store_seg<kCT>(static_cast<io_t*>(p.y_pre) + row, tl, L, fast, yp, kRows);
      }
      float zv[kCT];
      load_seg<kCT>(static_cast<const io_t*>(p.z) + row, tl, L, fast, zv, kRows);
#pragma unroll
      for (int j = 0; j < kCT; ++j) y[j] *= zv[j] * sigmoid(zv[j]);
    }
#pragma unroll
    for (int j = 0; j < kCT; ++j) y[j] = (tl + j < len) ? y[j] : 0.f;
    store_seg<kCT>(out_row, tl, L, fast, y, kRows);
  }
  if (p.last && lane < N && c_end == n_chunks && lane % kG == grp) {
    p.last[(chan * N + lane) * 2] = run_r;
    p.last[(chan * N + lane) * 2 + 1] = run_i;
  }
}

// The maps of a time-split forward: for every (channel, state) and every split but the last, the
// product of its a_bar and its end state from zero, as fwd_map_kernel does for real states. The
// product is taken chunk by chunk: one exponential of the whole split's delta would round its
// angle in turns once, at the split's size.
constexpr int kCMapW = 8;
constexpr int kCMapG = 4;  // waves that share a channel

template <bool kZOH, typename io_t, typename bc_t>
__global__ __launch_bounds__(kCMapW * 64) void cfwd_map_kernel(FwdParams p) {
  __shared__ float s_ph[kCMapW][kMaxN][4];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int b = blockIdx.y;
  const int d = blockIdx.x * (kCMapW / kCMapG) + w / kCMapG;
  const int grp = w % kCMapG;
  const int L = p.seqlen;
  const int N = p.dstate;
  if (d >= p.dim || grp >= N) return;  // no barrier in this kernel: idle waves may leave
  const int len = p.seq_lens ? min(max(p.seq_lens[b], 0), L) : L;
  const int c_lo = blockIdx.z * p.chunks_per_split;
  const int c_end = min((len + kCChunk - 1) / kCChunk, c_lo + p.chunks_per_split);
  if (c_lo >= c_end) return;  // no valid step: cfwd_kernel skips the split
  const size_t chan = static_cast<size_t>(b) * p.dim + d;
  const long long row = b * p.io_sb + d * p.io_sd;
  const bc_t* __restrict__ Bb = static_cast<const bc_t*>(p.B) + b * p.bc_sb;
  const float bias = p.delta_bias ? p.delta_bias[d] : 0.f;
  if (lane < N) {
    s_ph[w][lane][0] = 1.f;
    s_ph[w][lane][1] = s_ph[w][lane][2] = s_ph[w][lane][3] = 0.f;
  }
  for (int c = c_lo; c < c_end; ++c) {
    const int t0 = c * kCChunk;
    const int tl = t0 + lane * kCT;
    const bool fast = t0 + kCChunk <= L;
    float dlt[kCT], uu[kCT], bv[kCT];
    Seg<kCT, io_t> sd, su;
    Seg<kCT, bc_t> sb;
    fetch(sd, static_cast<const io_t*>(p.delta) + row, tl, L);
    fetch(su, static_cast<const io_t*>(p.u) + row, tl, L);
    fetch(sb, Bb + grp * p.bc_sn, tl, L);
    finish(sd, tl, L, fast, dlt);
    finish(su, tl, L, fast, uu);
    float ssum = 0.f;
#pragma unroll
    for (int j = 0; j < kCT; ++j) {
      const bool valid = tl + j < len;
      const float x = dlt[j] + bias;
      const float dv = p.delta_softplus ? softplus(x) : x;
      dlt[j] = valid ? dv : 0.f;
      uu[j] = valid ? uu[j] : 0.f;
      ssum += dlt[j];
    }
    for (int n = grp; n < N; n += kCMapG) {
      const CoefA cf = load_coef(p.A, static_cast<size_t>(d) * N + n);
      finish(sb, tl, L, fast, bv);
      fetch(sb, Bb + min(n + kCMapG, N - 1) * p.bc_sn, tl, L);
      float hr = 0.f, hi = 0.f;
#pragma unroll
      for (int j = 0; j < kCT; ++j) {
        const CExp e = cexp_t(dlt[j], cf);
        const bool valid = tl + j < len;
        const float ar = valid ? e.m * e.cy : 1.f, ai = valid ? e.m * e.sy : 0.f;
        float br, bi;
        if constexpr (kZOH) {
          zoh_e(dlt[j], cf, e, br, bi);
          br *= bv[j] * uu[j];
          bi *= bv[j] * uu[j];
        } else {
          br = dlt[j] * uu[j] * bv[j];
          bi = 0.f;
        }
        const float nr = __builtin_fmaf(ar, hr, __builtin_fmaf(-ai, hi, br));
        const float ni = __builtin_fmaf(ar, hi, __builtin_fmaf(ai, hr, bi));
        hr = nr;
        hi = ni;
      }
      const CExp pe = cexp_t(ssum, cf);
      float pr = pe.m * pe.cy, pi = pe.m * pe.sy;
      wave_scan_caffine(pr, pi, hr, hi);  // lane 63: the whole chunk
      if (lane == 63) {
        float* ph = s_ph[w][n];
        const float p0 = ph[0], p1 = ph[1], h0 = ph[2], h1 = ph[3];
        ph[0] = __builtin_fmaf(pr, p0, -pi * p1);
        ph[1] = __builtin_fmaf(pr, p1, pi * p0);
        ph[2] = __builtin_fmaf(pr, h0, __builtin_fmaf(-pi, h1, hr));
        ph[3] = __builtin_fmaf(pr, h1, __builtin_fmaf(pi, h0, hi));
      }
    }
  }
  if (lane < N && lane % kCMapG == grp) {
    const float* ph = s_ph[w][lane];
    reinterpret_cast<float4*>(p.split_map)[(static_cast<size_t>(blockIdx.z) * p.batch * p.dim + chan) * N + lane] =
        make_float4(ph[0], ph[1], ph[2], ph[3]);
  }
}

// The adjoint maps of a time-split backward (BwdParams::split_msg, complex as above): for every
// (channel, state) and every run of chunks_per_msg chunks right of the first split, the map
// m -> P m + Q of the adjoint entering from the right to the one the run sends left.
template <bool kHasZ, typename io_t, typename bc_t>
__global__ __launch_bounds__(kCMapW * 64) void cbwd_msg_kernel(BwdParams p) {
  __shared__ float s_pq[kCMapW][kMaxN][4];
  const int lane = threadIdx.x & 63;
  const int seg = 63 - lane;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int b = blockIdx.y;
  const int d = blockIdx.x * (kCMapW / kCMapG) + w / kCMapG;
  const int grp = w % kCMapG;
  const int L = p.seqlen;
  const int N = p.dstate;
  if (d >= p.dim || grp >= N) return;  // no barrier in this kernel: idle waves may leave
  const int len = p.seq_lens ? min(max(p.seq_lens[b], 0), L) : L;
  const int n_live = (len + kCChunk - 1) / kCChunk;
  const int c_lo = p.chunks_per_split + blockIdx.z * p.chunks_per_msg;
  const int c_hi = min(n_live, c_lo + p.chunks_per_msg);
  if (c_lo >= c_hi) return;  // no valid step: cbwd_kernel skips the run
  const size_t chan = static_cast<size_t>(b) * p.dim + d;
  const long long row = b * p.io_sb + d * p.io_sd;
  const bc_t* __restrict__ Cb = static_cast<const bc_t*>(p.C) + b * p.bc_sb;
  const float bias = p.delta_bias ? p.delta_bias[d] : 0.f;
  if (lane < N) {
    s_pq[w][lane][0] = 1.f;
    s_pq[w][lane][1] = s_pq[w][lane][2] = s_pq[w][lane][3] = 0.f;
  }
  for (int c = c_hi - 1; c >= c_lo; --c) {
    const int t0 = c * kCChunk;
    const int ts = t0 + seg * kCT;
    const bool fast = t0 + kCChunk <= L;
    float dlt[kCT], g[kCT], cv[kCT];
    Seg<kCT, io_t> sd, sg, sz_;
    Seg<kCT, bc_t> sc;
    fetch(sd, static_cast<const io_t*>(p.delta) + row, ts, L);
    fetch(sg, static_cast<const io_t*>(p.dout) + row, ts, L);
    if constexpr (kHasZ) fetch(sz_, static_cast<const io_t*>(p.z) + row, ts, L);
    fetch(sc, Cb + grp * p.bc_sn, ts, L);
    finish(sd, ts, L, fast, dlt);
    finish(sg, ts, L, fast, g);
    if constexpr (kHasZ) {
      float zv[kCT];
      finish(sz_, ts, L, fast, zv);
#pragma unroll
      for (int j = 0; j < kCT; ++j) g[j] *= zv[j] * sigmoid(zv[j]);
    }
    float ssum = 0.f;
#pragma unroll
    for (int j = 0; j < kCT; ++j) {
      const bool valid = ts + j < len;
      const float x = dlt[j] + bias;
      const float dv = p.delta_softplus ? softplus(x) : x;
      dlt[j] = valid ? dv : 0.f;
      g[j] = valid ? g[j] : 0.f;
      ssum += dlt[j];
    }
    for (int n = grp; n < N; n += kCMapG) {
      const CoefA cf = load_coef(p.A, static_cast<size_t>(d) * N + n);
      finish(sc, ts, L, fast, cv);
      fetch(sc, Cb + min(n + kCMapG, N - 1) * p.bc_sn, ts, L);
      float qr = 0.f, qi = 0.f;
#pragma unroll
      for (int j = kCT - 1; j >= 0; --j) {
        const CExp e = cexp_t(dlt[j], cf);
        const bool valid = ts + j < len;
        const float ar = valid ? e.m * e.cy : 1.f, ai = valid ? e.m * e.sy : 0.f;
        const float lr = __builtin_fmaf(cv[j], g[j], qr);
        const float li = qi;
        qr = __builtin_fmaf(ar, lr, ai * li);
        qi = __builtin_fmaf(ar, li, -ai * lr);
      }
      const CExp pe = cexp_t(ssum, cf);
      float pr = pe.m * pe.cy, pi = -pe.m * pe.sy;
      wave_scan_caffine(pr, pi, qr, qi);  // lane 63 (the chunk's first segment): the whole chunk
      if (lane == 63) {
        float* pq = s_pq[w][n];
        const float p0 = pq[0], p1 = pq[1], q0 = pq[2], q1 = pq[3];
        pq[0] = __builtin_fmaf(pr, p0, -pi * p1);
        pq[1] = __builtin_fmaf(pr, p1, pi * p0);
        pq[2] = __builtin_fmaf(pr, q0, __builtin_fmaf(-pi, q1, qr));
        pq[3] = __builtin_fmaf(pr, q1, __builtin_fmaf(pi, q0, qi));
      }
    }
  }
  if (lane < N && lane % kCMapG == grp) {
    const float* pq = s_pq[w][lane];
    reinterpret_cast<float4*>(p.split_msg)[(static_cast<size_t>(blockIdx.z) * p.batch * p.dim + chan) * N + lane] =
        make_float4(pq[0], pq[1], pq[2], pq[3]);
  }
}

// ---------------------------------------------------------------------------------
// Backward. Workgroup = kCBwdW waves walking p.chan_per_block channels of one batch row in
// rounds of kCBwdW, chunks from last to first. Within a chunk a lane owns segment
// 63 - lane, so the adjoint (which runs backwards in time) is an inclusive scan in lane
// order. Per state: re-run the forward inside the segment from the stored segment-entry
// state (carries), aggregate the segment's adjoint map from a zero seed, scan the maps
// across the lanes, then re-run the adjoint from the true seed and form the gradients.
// dB/dC of the chunk accumulate in LDS rows: at state iteration i wave w handles state
// (i + w) mod N in copy w / N of that state's row, so no two waves share a row at once and
// the sum order is fixed; a wave adds into its row once the row's previous owner has
// counted that iteration done in LDS (no workgroup barrier per iteration). After every
// chunk the rows (copies summed in order) go to this workgroup's partial rows; a second
// kernel sums the partials over workgroups in a fixed order.
template <bool kZOH, bool kHasZ, typename io_t, typename bc_t, int kRows>
__global__ __launch_bounds__(kCBwdW * 64) void cbwd_kernel(BwdParams p) {
  constexpr int W = kCBwdW;
  __shared__ __attribute__((aligned(16))) float s_acc[kCAccRows][2][kCChunk];
  __shared__ float s_mu[kCMaxChan][kMaxN][2];  // adjoint entering the chunk from the right
  __shared__ float s_dA[kCMaxChan][kMaxN][2];
  __shared__ float s_dD[kCMaxChan];
  __shared__ float s_db[kCMaxChan];
  __shared__ int s_done[W];  // state iterations of the current chunk each wave has finished

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = row_longest_first(p.seq_lens, p.batch, p.seqlen, blockIdx.y);
  const int L = p.seqlen;
  const int N = p.dstate;
  const int len = p.seq_lens ? min(max(p.seq_lens[b], 0), L) : L;
  const int cpb = p.chan_per_block;
  const int d0 = blockIdx.x * cpb;
  const int rounds = cpb / W;
  const int copies = (W + N - 1) / N;
  const int seg = 63 - lane;
  const bc_t* __restrict__ Bb = static_cast<const bc_t*>(p.B) + b * p.bc_sb;
  const bc_t* __restrict__ Cb = static_cast<const bc_t*>(p.C) + b * p.bc_sb;
  // Chunks [c_lo, c_end) of the row are this workgroup's.
  const int n_chunks = (L + kCChunk - 1) / kCChunk;
  const int n_live = (len + kCChunk - 1) / kCChunk;
  const int c_lo = blockIdx.z * p.chunks_per_split;
  const int c_end = min(n_chunks, c_lo + p.chunks_per_split);

  for (int i = tid; i < cpb * N; i += W * 64) {
    const int k = i / N, n = i - k * N;
    const int d = d0 + k;
    float mr = 0.f, mi = 0.f;
    if (p.dlast && d < p.dim) {
      const size_t o = ((static_cast<size_t>(b) * p.dim + d) * N + n) * 2;
      mr = p.dlast[o];
      mi = p.dlast[o + 1];
    }
    if (p.n_split > 1 && d < p.dim) {
      // the adjoint through the chunks to the right (those past the row's length pass it on)
      const float4* pq = reinterpret_cast<const float4*>(p.split_msg) + (static_cast<size_t>(b) * p.dim + d) * N + n;
      const size_t m_ld = static_cast<size_t>(p.batch) * p.dim * N;
      const int m_end = (n_live - p.chunks_per_split + p.chunks_per_msg - 1) / p.chunks_per_msg;
      for (int m = m_end - 1; m >= c_lo / p.chunks_per_msg; --m) through_map(pq[m * m_ld], mr, mi);
    }
    s_mu[k][n][0] = mr;
    s_mu[k][n][1] = mi;
    s_dA[k][n][0] = 0.f;
    s_dA[k][n][1] = 0.f;
  }
  for (int i = tid; i < cpb; i += W * 64) s_dD[i] = s_db[i] = 0.f;
  for (int i = tid; i < copies * N * 2 * kCChunk; i += W * 64) (&s_acc[0][0][0])[i] = 0.f;
  if (tid < W) s_done[tid] = 0;
  // The previous owner of this wave's row at chunk iteration g: the copy's next wave at
  // g - 1, or, for the copy's last wave, the copy's first wave at g - (N - w % N); every
  // wait is on an earlier iteration, so all waits resolve.
  const int wmod = w % N;
  const int copy_waves = min(N, W - (w / N) * N);
  const int pred = wmod + 1 < copy_waves ? w + 1 : w - wmod;
  const int pred_lag = wmod + 1 < copy_waves ? 1 : N - wmod;
  __syncthreads();

  for (int c = c_end - 1; c >= c_lo; --c) {
    const int t0 = c * kCChunk;
    const int ts = t0 + seg * kCT;
    const bool fast = kRows == kWholeRows || t0 + kCChunk <= L;
    const bool live = c < n_live;  // workgroup-uniform
    for (int r = 0; r < rounds; ++r) {
      const int k = r * W + w;
      const int d = d0 + k;
      const bool active = d < p.dim;
      const int dd = active ? d : p.dim - 1;
      const size_t chan = static_cast<size_t>(b) * p.dim + dd;
      const long long row = b * p.io_sb + dd * p.io_sd;
      io_t* du_row = static_cast<io_t*>(p.du) + row;
      io_t* ddl_row = static_cast<io_t*>(p.ddelta) + row;
      if (!live) {
        // Past the row's length: zero gradients; the adjoint passes through unchanged.
        if (active) {
          float zero[kCT];
#pragma unroll
          for (int j = 0; j < kCT; ++j) zero[j] = 0.f;
          store_seg<kCT>(du_row, ts, L, fast, zero, kRows);
          store_seg<kCT>(ddl_row, ts, L, fast, zero, kRows);
          if constexpr (kHasZ) store_seg<kCT>(static_cast<io_t*>(p.dz) + row, ts, L, fast, zero, kRows);
        }
        continue;
      }
      const float Dv = p.D ? p.D[dd] : 0.f;
      const float bias = p.delta_bias ? p.delta_bias[dd] : 0.f;
      float xraw[kCT], dlt[kCT], uu[kCT], g[kCT];
      Seg<kCT, io_t> sd, su, sg, sz_, sy;
      fetch(sd, static_cast<const io_t*>(p.delta) + row, ts, L, kRows);
      fetch(su, static_cast<const io_t*>(p.u) + row, ts, L, kRows);
      fetch(sg, static_cast<const io_t*>(p.dout) + row, ts, L, kRows);
      if constexpr (kHasZ) {
        fetch(sz_, static_cast<const io_t*>(p.z) + row, ts, L, kRows);
        fetch(sy, static_cast<const io_t*>(p.y_pre) + row, ts, L, kRows);
      }
      finish(sd, ts, L, fast, xraw, kRows);
      finish(su, ts, L, fast, uu, kRows);
      finish(sg, ts, L, fast, g, kRows);
      float ssum = 0.f;
#pragma unroll
      for (int j = 0; j < kCT; ++j) {
        const bool valid = ts + j < len;
        xraw[j] += bias;
        const float dv = p.delta_softplus ? softplus(xraw[j]) : xraw[j];
        dlt[j] = valid ? dv : 0.f;
        uu[j] = valid ? uu[j] : 0.f;
        g[j] = valid ? g[j] : 0.f;
        ssum += dlt[j];
      }
      if constexpr (kHasZ) {
        float zv[kCT], yp[kCT], dz[kCT];
        finish(sz_, ts, L, fast, zv, kRows);
        finish(sy, ts, L, fast, yp, kRows);
#pragma unroll
        for (int j = 0; j < kCT; ++j) {
          const float sz = sigmoid(zv[j]);
          dz[j] = g[j] * yp[j] * sz * __builtin_fmaf(zv[j], 1.f - sz, 1.f);
          g[j] = g[j] * zv[j] * sz;
        }
        if (active) store_seg<kCT>(static_cast<io_t*>(p.dz) + row, ts, L, fast, dz, kRows);
      }
      float du[kCT], ddl[kCT];
#pragma unroll
      for (int j = 0; j < kCT; ++j) {
        du[j] = Dv * g[j];
        ddl[j] = 0.f;
      }

      // B, C rows and the segment-entry state of the next state are loaded one state
      // ahead, so their latency overlaps a state's arithmetic (Euler; ZOH keeps E_t per
      // step in registers and has no room for them, so it loads each state's rows in place).
      constexpr bool kAhead = !kZOH;
      const float2* __restrict__ carry_seg = reinterpret_cast<const float2*>(p.carries) +
                                             chan * N * p.n_seg + ts / kCT;
      Seg<kCT, bc_t> sbn, scn;
      float2 hnx = make_float2(0.f, 0.f);
      if (kAhead && active) {
        const int n0 = w % N;
        fetch(sbn, Bb + n0 * p.bc_sn, ts, L, kRows);
        fetch(scn, Cb + n0 * p.bc_sn, ts, L, kRows);
        if (kRows == kWholeRows || ts < L) hnx = carry_seg[static_cast<size_t>(n0) * p.n_seg];
      }
      for (int it = 0; it < N; ++it) {
        const int n = (it + w) % N;
        const int arow = (w / N) * N + n;
        if (active) {
          const CoefA cf = load_coef(p.A, static_cast<size_t>(dd) * N + n);
          float bv[kCT], cv[kCT];
          float hinr, hini;
          if constexpr (kAhead) {
            finish(sbn, ts, L, fast, bv, kRows);
            finish(scn, ts, L, fast, cv, kRows);
            hinr = hnx.x;
            hini = hnx.y;
            if (it + 1 < N) {
              const int nn = (it + 1 + w) % N;
              fetch(sbn, Bb + nn * p.bc_sn, ts, L, kRows);
              fetch(scn, Cb + nn * p.bc_sn, ts, L, kRows);
              if (kRows == kWholeRows || ts < L) hnx = carry_seg[static_cast<size_t>(nn) * p.n_seg];
            }
          } else {
            load_seg<kCT>(Bb + n * p.bc_sn, ts, L, fast, bv, kRows);
            load_seg<kCT>(Cb + n * p.bc_sn, ts, L, fast, cv, kRows);
            const float2 h0 = kRows == kWholeRows || ts < L ? carry_seg[static_cast<size_t>(n) * p.n_seg] : make_float2(0.f, 0.f);
            hinr = h0.x;
            hini = h0.y;
          }
          // Forward re-run: a_j, the state before each step, (ZOH) E_j.
          float ar[kCT], ai[kCT], hpr[kCT], hpi[kCT], er[kCT], ei[kCT];
#pragma unroll
          for (int j = 0; j < kCT; ++j) {
            const CExp e = cexp_t(dlt[j], cf);
            const bool valid = ts + j < len;
            ar[j] = valid ? e.m * e.cy : 1.f;
            ai[j] = valid ? e.m * e.sy : 0.f;
            float brj, bij;
            if constexpr (kZOH) {
              zoh_e(dlt[j], cf, e, er[j], ei[j]);
              const float s = bv[j] * uu[j];
              brj = er[j] * s;
              bij = ei[j] * s;
            } else {
              er[j] = ei[j] = 0.f;
              brj = dlt[j] * uu[j] * bv[j];
              bij = 0.f;
            }
            hpr[j] = hinr;
            hpi[j] = hini;
            const float nr = __builtin_fmaf(ar[j], hinr, __builtin_fmaf(-ai[j], hini, brj));
            const float ni = __builtin_fmaf(ar[j], hini, __builtin_fmaf(ai[j], hinr, bij));
            hinr = nr;
            hini = ni;
          }
          // Segment adjoint map m -> Pc m + Hc (m entering at the segment end): Pc = conj of
          // the segment's product of a_bar, Hc from a zero seed.
          float hcr = 0.f, hci = 0.f;
#pragma unroll
          for (int j = kCT - 1; j >= 0; --j) {
            const float lr = __builtin_fmaf(cv[j], g[j], hcr);
            const float li = hci;
            hcr = __builtin_fmaf(ar[j], lr, ai[j] * li);
            hci = __builtin_fmaf(ar[j], li, -ai[j] * lr);
          }
          const CExp pe = cexp_t(ssum, cf);
          float pcr = pe.m * pe.cy, pci = -pe.m * pe.sy;
          wave_scan_caffine(pcr, pci, hcr, hci);
          const float mur = s_mu[k][n][0], mui = s_mu[k][n][1];
          const float oar = __builtin_fmaf(pcr, mur, __builtin_fmaf(-pci, mui, hcr));
          const float oai = __builtin_fmaf(pcr, mui, __builtin_fmaf(pci, mur, hci));
          float mr = dpp_mov<kWaveShr1, 0xF>(mur, oar);
          float mi = dpp_mov<kWaveShr1, 0xF>(mui, oai);
          if (lane == 0) {
            mr = mur;
            mi = mui;
          }
          // Lane 63 holds segment 0: its outgoing adjoint enters the previous chunk.
          if (lane == 63) {
            s_mu[k][n][0] = oar;
            s_mu[k][n][1] = oai;
          }
          float dar = 0.f, dai = 0.f;
          float accB[kCT], accC[kCT];
#pragma unroll
          for (int j = kCT - 1; j >= 0; --j) {
            const float lr = __builtin_fmaf(cv[j], g[j], mr);
            const float li = mi;
            // W = lambda * conj(a_bar h_prev): dA += delta W, ddelta += Re(W conj(A))
            const float ahr = __builtin_fmaf(ar[j], hpr[j], -ai[j] * hpi[j]);
            const float ahi = __builtin_fmaf(ar[j], hpi[j], ai[j] * hpr[j]);
            const float wr = __builtin_fmaf(lr, ahr, li * ahi);
            const float wi = __builtin_fmaf(li, ahr, -lr * ahi);
            dar = __builtin_fmaf(dlt[j], wr, dar);
            dai = __builtin_fmaf(dlt[j], wi, dai);
            ddl[j] = __builtin_fmaf(wr, cf.ar, __builtin_fmaf(wi, cf.ai, ddl[j]));
            // m = conj(a_bar) lambda: the adjoint leaving the step towards the past.
            const float nmr = __builtin_fmaf(ar[j], lr, ai[j] * li);
            const float nmi = __builtin_fmaf(ar[j], li, -ai[j] * lr);
            if constexpr (kZOH) {
              const float s = bv[j] * uu[j];
              const float ge = __builtin_fmaf(er[j], lr, ei[j] * li);  // Re(conj(E) lambda)
              du[j] = __builtin_fmaf(bv[j], ge, du[j]);
              accB[j] = uu[j] * ge;
              ddl[j] = __builtin_fmaf(s, nmr, ddl[j]);  // s Re(conj(a_bar) lambda)
              // dE/dA = (delta a_bar - E) / A
              const float xr = __builtin_fmaf(dlt[j], ar[j], -er[j]);
              const float xi = __builtin_fmaf(dlt[j], ai[j], -ei[j]);
              const float vr = __builtin_fmaf(xr, cf.ar, xi * cf.ai) * cf.inv_a2;
              const float vi = __builtin_fmaf(xi, cf.ar, -xr * cf.ai) * cf.inv_a2;
              dar = __builtin_fmaf(s, __builtin_fmaf(vr, lr, vi * li), dar);
              dai = __builtin_fmaf(s, __builtin_fmaf(vr, li, -vi * lr), dai);
              accC[j] = g[j] * __builtin_fmaf(er[j], s, ahr);
            } else {
              const float q = lr * bv[j];
              du[j] = __builtin_fmaf(dlt[j], q, du[j]);
              ddl[j] = __builtin_fmaf(uu[j], q, ddl[j]);
              const float dlu = dlt[j] * uu[j];
              accB[j] = lr * dlu;
              accC[j] = g[j] * __builtin_fmaf(dlu, bv[j], ahr);
            }
            mr = nmr;
            mi = nmi;
          }
          const float sar = wave_sum(dar), sai = wave_sum(dai);
          if (lane == 0) {
            s_dA[k][n][0] += sar;
            s_dA[k][n][1] += sai;
          }
          // This wave's rows for the iteration: accumulate the segment's dB/dC once the
          // rows' previous owner is done with them (bounded poll: it always progresses).
          {
            const int need = r * N + it - pred_lag + 1;
            if (need > 0) {
              int spins = 0;
              while (__hip_atomic_load(&s_done[pred], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < need &&
                     ++spins < (1 << 22))
                __builtin_amdgcn_s_sleep(1);
            }
            asm volatile("" ::: "memory");  // the row's reads stay below the poll
          }
          f32x4* rb = reinterpret_cast<f32x4*>(&s_acc[arow][0][seg * kCT]);
          f32x4* rc = reinterpret_cast<f32x4*>(&s_acc[arow][1][seg * kCT]);
#pragma unroll
          for (int q = 0; q < kCT / 4; ++q) {
            f32x4 vb = rb[q], vc = rc[q];
            vb.x += accB[4 * q + 0];
            vb.y += accB[4 * q + 1];
            vb.z += accB[4 * q + 2];
            vb.w += accB[4 * q + 3];
            vc.x += accC[4 * q + 0];
            vc.y += accC[4 * q + 1];
            vc.z += accC[4 * q + 2];
            vc.w += accC[4 * q + 3];
            rb[q] = vb;
            rc[q] = vc;
          }
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the row writes have landed
        } else {
          // An inactive wave owns its rows without touching them: it passes them on after
          // their previous owner.
          const int need = r * N + it - pred_lag + 1;
          if (need > 0) {
            int spins = 0;
            while (__hip_atomic_load(&s_done[pred], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < need &&
                   ++spins < (1 << 22))
              __builtin_amdgcn_s_sleep(1);
          }
        }
        if (lane == 0) __hip_atomic_store(&s_done[w], r * N + it + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
      if (active) {
        float dsum = 0.f, gsum = 0.f;
#pragma unroll
        for (int j = 0; j < kCT; ++j) {
          const bool valid = ts + j < len;
          float dx = ddl[j];
          if (p.delta_softplus) dx *= sigmoid(xraw[j]);
          dx = valid ? dx : 0.f;
          du[j] = valid ? du[j] : 0.f;
          ddl[j] = dx;
          dsum += dx;
          gsum = __builtin_fmaf(g[j], uu[j], gsum);
        }
        store_seg<kCT>(du_row, ts, L, fast, du, kRows);
        store_seg<kCT>(ddl_row, ts, L, fast, ddl, kRows);
        const float sd = wave_sum(gsum), sb = wave_sum(dsum);
        if (lane == 0) {
          s_dD[k] += sd;
          s_db[k] += sb;
        }
      }
    }
    // This chunk's dB/dC partial rows (copies summed in order), then clear the rows, after
    // every wave's last accumulation. None past the row's length: the reduction takes those
    // steps as zero (the rows stay zero).
    __syncthreads();
    if (tid < W) s_done[tid] = 0;  // (read again only after the barrier that ends the flush)
    float* part = p.part_dBC + static_cast<size_t>(blockIdx.x) * p.part_stride;
    for (int i = tid; live && i < 2 * N * kCChunk; i += W * 64) {
      const int which = i / (N * kCChunk);
      const int rem = i - which * N * kCChunk;
      const int n = rem / kCChunk;
      const int t = rem - n * kCChunk;
      float s = 0.f;
      for (int cp = 0; cp < copies; ++cp) {
        s += s_acc[cp * N + n][which][t];
        s_acc[cp * N + n][which][t] = 0.f;
      }
      if (t0 + t < L) part[(static_cast<size_t>(b) * 2 * N + which * N + n) * L + t0 + t] = s;
    }
    __syncthreads();
  }
  for (int i = tid; i < cpb * N; i += W * 64) {
    const int k = i / N, n = i - k * N;
    const int d = d0 + k;
    if (d >= p.dim) continue;
    const size_t o = ((static_cast<size_t>(b) * p.dim + d) * N + n) * 2;
    float* part_dA = p.part_dA + static_cast<size_t>(blockIdx.z) * p.batch * p.dim * N * 2;
    part_dA[o] = s_dA[k][n][0];
    part_dA[o + 1] = s_dA[k][n][1];
    if (p.dinit && c_lo == 0) {
      p.dinit[o] = s_mu[k][n][0];
      p.dinit[o + 1] = s_mu[k][n][1];
    }
  }
  for (int i = tid; i < cpb; i += W * 64) {
    const int d = d0 + i;
    if (d >= p.dim) continue;
    const size_t o = (static_cast<size_t>(blockIdx.z) * p.batch + b) * p.dim + d;
    p.part_dD[o] = s_dD[i];
    p.part_dbias[o] = s_db[i];
  }
}

// ---------------------------------------------------------------------------------
// Single-token step with complex A (S6.step's complex branch, mamba/mamba1.py:200-214):
// state [B][D][N][2] float32 (interleaved complex) updated in place, out = (sum_n C Re(h) +
// D u) * silu(z). Mapping of the real step: a 16-lane DPP row per (b, d) channel, one lane
// per state, batch fastest.
template <bool kZOH, typename io_t, typename bc_t>
__global__ __launch_bounds__(256) void cssm_step_kernel(StepParams p) {
  const long long idx = (static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x) >> 4;
  const int n = threadIdx.x & 15;
  const bool ch_ok = idx < static_cast<long long>(p.batch) * p.dim;
  const int b = ch_ok ? static_cast<int>(idx % p.batch) : 0;
  const int d = ch_ok ? static_cast<int>(idx / p.batch) : 0;
  const int N = p.dstate;
  const bool on = ch_ok && n < N;
  const long long io = b * p.io_sb + d * p.io_sd;
  float yv = 0.f, u = 0.f;
  if (ch_ok) {
    u = to_f32(static_cast<const io_t*>(p.u)[io]);
    float dt = to_f32(static_cast<const io_t*>(p.delta)[io]) + (p.delta_bias ? p.delta_bias[d] : 0.f);
    if (p.delta_softplus) dt = softplus(dt);
    if (on) {
      const CoefA cf = load_coef(p.A, static_cast<size_t>(d) * N + n);
      const CExp e = cexp_t(dt, cf);
      const float s = to_f32(static_cast<const bc_t*>(p.B)[b * p.bc_sb + n * p.bc_sn]) * u;
      float br, bi;
      if constexpr (kZOH) {
        float er, ei;
        zoh_e(dt, cf, e, er, ei);
        br = er * s;
        bi = ei * s;
      } else {
        br = dt * s;
        bi = 0.f;
      }
      float2* st = reinterpret_cast<float2*>(p.state) + (static_cast<size_t>(b) * p.dim + d) * N + n;
      const float2 h = *st;
      const float ar = e.m * e.cy, ai = e.m * e.sy;
      const float nr = __builtin_fmaf(ar, h.x, __builtin_fmaf(-ai, h.y, br));
      const float ni = __builtin_fmaf(ar, h.y, __builtin_fmaf(ai, h.x, bi));
      *st = make_float2(nr, ni);
      yv = to_f32(static_cast<const bc_t*>(p.C)[b * p.bc_sb + n * p.bc_sn]) * nr;
    }
  }
  yv += dpp_mov<kRowShr1, 0xF>(0.f, yv);
  yv += dpp_mov<kRowShr2, 0xF>(0.f, yv);
  yv += dpp_mov<kRowShr4, 0xF>(0.f, yv);
  yv += dpp_mov<kRowShr8, 0xF>(0.f, yv);
  if (ch_ok && n == 15) {
    float y = yv;
    if (p.D) y = __builtin_fmaf(p.D[d], u, y);
    if (p.z) {
      const float z = to_f32(static_cast<const io_t*>(p.z)[io]);
      y *= z * sigmoid(z);
    }
    store_as(static_cast<io_t*>(p.out) + io, y);
  }
}

hipError_t launch_cssm_step(const StepParams& p, bool zoh, bool io_bf16, bool bc_bf16, hipStream_t stream) {
  const long long n = static_cast<long long>(p.batch) * p.dim * 16;
  const dim3 grid(static_cast<unsigned>((n + 255) / 256)), block(256);
#define MSS_CSTEP(Z, IO, BC) hipLaunchKernelGGL((cssm_step_kernel<Z, IO, BC>), grid, block, 0, stream, p)
  if (zoh) {
    if (io_bf16) { if (bc_bf16) MSS_CSTEP(true, bf16_t, bf16_t); else MSS_CSTEP(true, bf16_t, float); }
    else { if (bc_bf16) MSS_CSTEP(true, float, bf16_t); else MSS_CSTEP(true, float, float); }
  } else {
    if (io_bf16) { if (bc_bf16) MSS_CSTEP(false, bf16_t, bf16_t); else MSS_CSTEP(false, bf16_t, float); }
    else { if (bc_bf16) MSS_CSTEP(false, float, bf16_t); else MSS_CSTEP(false, float, float); }
  }
#undef MSS_CSTEP
  return hipGetLastError();
}

// ---------------------------------------------------------------------------------
// Four waves share a channel where one each would leave three quarters of the GPU's waves (5 per
// SIMD) idle and there are states enough for what the four repeat: four (ZOH three), one fewer up to
// 512 channels (two waves a SIMD), two up to 256. One wave and four, B=1 L=1024 float32: D=128 N=1 5.7
// and 6.0 us, N=2 7.0 and 6.1; D=300 N=2 7.4 and 7.7, N=3 8.7 and 7.9; D=600 N=3 9.3 and 10.3, N=4 10.8
// and 10.6; D=1280 N=1 8.5 and 12.0, N=4 15.9 and 14.9. Rows are split in time where even those leave
// more than a third of the SIMDs idle (160 channels or fewer) and at least three chunks go off the
// chain (one state: four), as fwd_plan does for real states. Measured on MI355X, N=16 float32: B=1
// D=400 L=8000 356 us with a wave to a channel, 165 with four; whole and split (maps among it) B=1
// D=64 L=1536 14.4 and 14.5, L=2048 18 and 15, L=8192 67 and 30; D=160 L=4096 36 and 36, L=8192 70 and
// 64; D=200 L=4096 37 and 48, L=8192 72 and 71; D=256 L=8192 71 and 89.
constexpr int kCFwdSlots = 5 * 4 * kCUs;

static bool cfwd_groups(const FwdParams& p, bool zoh) {
  const long long waves = 4LL * p.batch * p.dim;
  if (waves > kCFwdSlots) return false;
  const int least = waves <= 4 * kCUs ? 2 : (waves <= 2 * 4 * kCUs ? 3 : 4) - (zoh ? 1 : 0);
  return p.n_split > 1 || p.dstate >= least;
}

FwdPlan cfwd_plan(int batch, int dim, int seqlen, int dstate) {
  const int n_chunks = (seqlen + kCChunk - 1) / kCChunk;
  FwdPlan plan{1, n_chunks};
  const long long waves = 4LL * batch * dim;
  if (8 * waves > kCFwdSlots) return plan;
  const int s = static_cast<int>(kCFwdSlots / waves < n_chunks ? kCFwdSlots / waves : n_chunks);
  const int per = (n_chunks + s - 1) / s;
  if (n_chunks - per < (dstate == 1 ? 4 : 3)) return plan;
  return FwdPlan{(n_chunks + per - 1) / per, per};
}

template <bool kZOH, typename io_t, typename bc_t, int kG>
static hipError_t launch_cfwd_g(const FwdParams& p, hipStream_t stream) {
  constexpr int kChan = kCFwdW / kG;
  const dim3 grid((p.dim + kChan - 1) / kChan, p.batch, kG > 1 ? p.n_split : 1);
  if constexpr (sizeof(io_t) == sizeof(bc_t)) {
    if (p.seqlen % kCChunk == 0) {
      hipLaunchKernelGGL((cfwd_kernel<kZOH, io_t, bc_t, kWholeRows, kG>), grid, dim3(kCFwdW * 64), 0, stream, p);
      return hipGetLastError();
    }
  }
  if (slots_fit<io_t>(p.seqlen) && slots_fit<bc_t>(p.seqlen))
    hipLaunchKernelGGL((cfwd_kernel<kZOH, io_t, bc_t, kSlotRows, kG>), grid, dim3(kCFwdW * 64), 0, stream, p);
  else
    hipLaunchKernelGGL((cfwd_kernel<kZOH, io_t, bc_t, kAnyRows, kG>), grid, dim3(kCFwdW * 64), 0, stream, p);
  return hipGetLastError();
}

template <bool kZOH, typename io_t, typename bc_t>
static hipError_t launch_cfwd_t(const FwdParams& p, hipStream_t stream) {
  if (!cfwd_groups(p, kZOH)) return launch_cfwd_g<kZOH, io_t, bc_t, 1>(p, stream);
  if (p.n_split > 1) {
    constexpr int kChan = kCMapW / kCMapG;
    const dim3 grid((p.dim + kChan - 1) / kChan, p.batch, p.n_split - 1);
    hipLaunchKernelGGL((cfwd_map_kernel<kZOH, io_t, bc_t>), grid, dim3(kCMapW * 64), 0, stream, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return launch_cfwd_g<kZOH, io_t, bc_t, kCFwdW>(p, stream);
}

hipError_t launch_cfwd(const FwdParams& p, int zoh, int io_bf16, int bc_bf16, hipStream_t stream) {
  if (zoh) {
    if (io_bf16) return bc_bf16 ? launch_cfwd_t<true, bf16_t, bf16_t>(p, stream)
                                : launch_cfwd_t<true, bf16_t, float>(p, stream);
    return bc_bf16 ? launch_cfwd_t<true, float, bf16_t>(p, stream)
                   : launch_cfwd_t<true, float, float>(p, stream);
  }
  if (io_bf16) return bc_bf16 ? launch_cfwd_t<false, bf16_t, bf16_t>(p, stream)
                              : launch_cfwd_t<false, bf16_t, float>(p, stream);
  return bc_bf16 ? launch_cfwd_t<false, float, bf16_t>(p, stream)
                 : launch_cfwd_t<false, float, float>(p, stream);
}

BwdPlan cbwd_plan(int batch, int dim, int seqlen, bool split) {
  // One workgroup per CU (registers: 3 waves per SIMD); take the fewest channel rounds K
  // with batch * ceil(dim / (kW*K)) <= 256, at most kCMaxChan channels.
  const long long per_row = (dim + kCBwdW - 1) / kCBwdW;
  long long k = 1;
  while (k < per_row && k * kCBwdW < kCMaxChan &&
         static_cast<long long>(batch) * ((per_row + k - 1) / k) > kCUs)
    ++k;
  const int n_chunks = (seqlen + kCChunk - 1) / kCChunk;
  BwdPlan plan{kCBwdW, static_cast<int>(k) * kCBwdW, 1, n_chunks, 0, 1};
  // Rows split in time where that leaves half the CUs or more idle, as bwd_split_plan does for
  // real states; a chunk of a round takes about 60 us, its adjoint map an eighth of that. Measured
  // on MI355X, B=1 D=400 L=8000 N=16 float32: 996 us whole, 271 in six splits
  // (maps 62); D=1536 L=2048 241 and 166 in two.
  const long long grid = static_cast<long long>(batch) * ((per_row + k - 1) / k);
  if (split && 2 * grid <= kCUs && n_chunks > 1) {
    const int s = static_cast<int>(kCUs / grid < n_chunks ? kCUs / grid : n_chunks);
    plan.chunks_per_split = (n_chunks + s - 1) / s;
    // Maps as long as they can be with 16 waves (four to a channel) for every CU.
    const long long map_chunks = static_cast<long long>(batch) * dim * kCMapG * (n_chunks - plan.chunks_per_split);
    const long long want = map_chunks / (16LL * kCUs) > 1 ? map_chunks / (16LL * kCUs) : 1;
    const int per_split = static_cast<int>((plan.chunks_per_split + want - 1) / want);
    plan.chunks_per_msg = (plan.chunks_per_split + per_split - 1) / per_split;
    plan.chunks_per_split = plan.chunks_per_msg * per_split;
    plan.n_split = (n_chunks + plan.chunks_per_split - 1) / plan.chunks_per_split;
    if (plan.n_split > 1)
      plan.n_msg = (n_chunks - plan.chunks_per_split + plan.chunks_per_msg - 1) / plan.chunks_per_msg;
  }
  return plan;
}

template <bool kZOH, bool kHasZ, typename io_t, typename bc_t>
static hipError_t launch_cbwd_t(const BwdParams& p, hipStream_t stream) {
  dim3 grid(p.n_blocks_d, p.batch, p.n_split);
  if constexpr (sizeof(io_t) == sizeof(bc_t)) {
    if (p.seqlen % kCChunk == 0) {
      hipLaunchKernelGGL((cbwd_kernel<kZOH, kHasZ, io_t, bc_t, kWholeRows>), grid, dim3(kCBwdW * 64), 0, stream, p);
      return hipGetLastError();
    }
  }
  if (slots_fit<io_t>(p.seqlen) && slots_fit<bc_t>(p.seqlen))
    hipLaunchKernelGGL((cbwd_kernel<kZOH, kHasZ, io_t, bc_t, kSlotRows>), grid, dim3(kCBwdW * 64), 0, stream, p);
  else
    hipLaunchKernelGGL((cbwd_kernel<kZOH, kHasZ, io_t, bc_t, kAnyRows>), grid, dim3(kCBwdW * 64), 0, stream, p);
  return hipGetLastError();
}

template <typename io_t, typename bc_t>
static hipError_t launch_cbwd_io(const BwdParams& p, int zoh, hipStream_t stream) {
  const bool hz = p.z != nullptr;
  if (p.n_split > 1) {
    constexpr int kChan = kCMapW / kCMapG;
    const dim3 grid((p.dim + kChan - 1) / kChan, p.batch, p.n_msg);
    hipLaunchKernelGGL((hz ? cbwd_msg_kernel<true, io_t, bc_t> : cbwd_msg_kernel<false, io_t, bc_t>), grid,
                       dim3(kCMapW * 64), 0, stream, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if (zoh) return hz ? launch_cbwd_t<true, true, io_t, bc_t>(p, stream)
                     : launch_cbwd_t<true, false, io_t, bc_t>(p, stream);
  return hz ? launch_cbwd_t<false, true, io_t, bc_t>(p, stream)
            : launch_cbwd_t<false, false, io_t, bc_t>(p, stream);
}

hipError_t launch_cbwd_scan(const BwdParams& p, int zoh, int io_bf16, int bc_bf16, hipStream_t stream) {
  if (io_bf16) return bc_bf16 ? launch_cbwd_io<bf16_t, bf16_t>(p, zoh, stream)
                              : launch_cbwd_io<bf16_t, float>(p, zoh, stream);
  return bc_bf16 ? launch_cbwd_io<float, bf16_t>(p, zoh, stream)
                 : launch_cbwd_io<float, float>(p, zoh, stream);
}

}  // namespace mss
