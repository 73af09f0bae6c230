// Forward selective-scan kernel for gfx950 (MI355X): the kernel template and its launch
// shapes, shared by the translation units that instantiate it (mss_fwd.hip: float32 I/O and
// the dispatcher; mss_fwd_bf16.hip: bf16 I/O, compiled with another machine-scheduler
// strategy). Algorithm and mapping: see the comment at the top of mss_fwd.hip.
#pragma once
#include "mss_common.h"


// Launch shapes. A "wide" shape (16 steps per lane, 4 waves per SIMD) for bf16 grids that
// fill the GPU several times over, and a "narrow" one (8 steps per lane, 6 waves per SIMD:
// 50% more resident workgroups) for float32 rows and for grids that fit in one pass of it,
// where the wide shape would leave a half-occupied tail pass. Waves per workgroup and states per staging round
// are shared; all are overridable at build time for tuning sweeps.
#ifndef MSS_FWD_W
#define MSS_FWD_W 8
#endif
#ifndef MSS_FWD_NB
#define MSS_FWD_NB 4
#endif
#ifndef MSS_FWD_T_WIDE
#define MSS_FWD_T_WIDE 16
#endif
#ifndef MSS_FWD_OCC_WIDE
#define MSS_FWD_OCC_WIDE 4
#endif
#ifndef MSS_FWD_T_NARROW
#define MSS_FWD_T_NARROW 8
#endif
#ifndef MSS_FWD_OCC_NARROW
#define MSS_FWD_OCC_NARROW 6
#endif


namespace mss {

// Resident workgroups of the narrow shape: 256 CUs * kOcc waves per SIMD * 4 SIMDs / kW.
constexpr long long kFwdNarrowSlots = 256LL * MSS_FWD_OCC_NARROW * 4 / MSS_FWD_W;
constexpr int kFwdG = 4;  // waves that share a channel where the channels alone leave it idle

// Stage elements [t0, t0 + 64*kT) of `nrows` rows (B rows of states n0.., then C rows)
// into dst[row][slot] (64*kT elements of bc_t per row), spread over all threads.
// Row k of B (C) starts at Bb (Cb) + (n0 + k) * sn.
// dma: rows are 16-byte aligned and L is a multiple of the slot width, so each slot is
// either fully inside [0, L) or fully past it; past-the-end slots re-read the last valid
// slot (finite values; they only meet zero coefficients).
template <int kT, int kW, int kNB, typename bc_t>
__device__ __forceinline__ void stage_round(const bc_t* __restrict__ Bb, const bc_t* __restrict__ Cb,
                                            int n0, int nb, int t0, int L, long long sn, bool dma,
                                            uint4 (*dst)[2][64 * kT * sizeof(bc_t) / 16], int tid) {
  constexpr int kE = BcStage<bc_t>::kElemsPerSlot;
  constexpr int kQ = kT / kE;
  constexpr int kSlots = 64 * kQ;  // per row
  const int total = nb * 2 * kSlots;
  if (dma) {
    const int lane = tid & 63;
    const int w = tid >> 6;
    // Lane's source offset inside a row for slot s0 + lane: the same for every row.
    for (int f0 = w * 64; f0 < total; f0 += kW * 64) {
      const int rowi = f0 / kSlots;  // uniform: kSlots is a multiple of 64
      const int k = rowi >> 1;
      const int which = rowi & 1;
      const int s0 = f0 - rowi * kSlots;
      const int s = s0 + lane;
      const int i = s / kQ;  // kQ is a power of two
      const int q = (s % kQ) ^ slot_swz<kQ>(i);
      int e = t0 + i * kT + q * kE;
      e = e < L ? e : L - kE;
      const bc_t* src = (which ? Cb : Bb) + (n0 + k) * sn + e;
      __builtin_amdgcn_global_load_lds((gbl_void_t)src, (lds_void_t)(&dst[k][which][s0]), 16, 0, 0);
    }
  } else {
    const bool fast = t0 + 64 * kT <= L;
    for (int f = tid; f < total; f += kW * 64) {
      const int rowi = f / kSlots;
      const int k = rowi >> 1;
      const int which = rowi & 1;
      const int s = f - rowi * kSlots;
      const int i = s / kQ;
      const int q = (s % kQ) ^ slot_swz<kQ>(i);
      dst[k][which][s] = load_slot((which ? Cb : Bb) + (n0 + k) * sn, t0 + i * kT + q * kE, L, fast);
    }
  }
}

// kMaxS: the per-wave state tables' size (kMaxN, or kMaxNWide for float32 scans with more
// states). kRows: kWholeRows, L is a multiple of the chunk and the B/C rows can be copied to LDS
// directly, so no lane ever meets the row's end (the paths that handle it spill registers: B=8 D=2560
// L=4096 float32 with lengths 306 us, the general instance 351); kSlotRows, the same B/C rows and L a
// multiple of 16 bytes of activations (B=8 D=2048 L=4032 N=16 float32: 482 us, the general instance
// 517; more than 16 states and rows of two types have no whole-row instance); kAnyRows, the general
// one: B=3 D=1000 L=2051 bf16 in 92 us; element-wise accesses to such rows took 146.
// kG: waves that share a channel, each taking every kG-th state of a staging round; their partial
// outputs are added in order through LDS at the end of a chunk. 1 where the channels alone fill
// the GPU (the waves of a channel repeat its delta and u loads and the softplus).
template <int kT, int kW, int kNB, int kOcc, bool kZOH, typename io_t, typename bc_t, int kMaxS, int kRows, int kG>
__global__ __launch_bounds__(kW * 64) __attribute__((amdgpu_waves_per_eu(kOcc, kOcc)))
void fwd_kernel(FwdParams p) {
  constexpr int kChunk = 64 * kT;
  static_assert(kT % kSegSteps == 0, "lane segments must hold whole carry segments");
  constexpr int kRowSlots = kChunk * static_cast<int>(sizeof(bc_t)) / 16;
  // Two stage buffers as distinct objects, selected statically (rounds run in pairs), so
  // the compiler can tell the in-flight copy into one from the reads of the other.
  __shared__ uint4 stage0[kNB][2][kRowSlots];  // [state][B|C][slot]
  __shared__ uint4 stage1[kNB][2][kRowSlots];
  __shared__ float s_run[kW][kMaxS];
  __shared__ float s_a2[kW][kMaxS];
  __shared__ float s_a[kW][kMaxS];
  // 16-step lanes: each wave's z row for the current chunk, copied from global memory at the
  // chunk start (direct-to-LDS) so its latency passes under the state loop instead of after
  // it; lane i's q-th 16-byte slot at [q * 64 + i]. (Measured on MI355X, c3 forward 414 ->
  // 406 us, a c5 layer's 162 -> 158; with the 8-step float32 shape, whose three workgroups
  // per CU it would take 16 KB of LDS each, c2 102 -> 111, so that shape keeps the load.)
  constexpr bool kZLds = kT == 16;
  constexpr int kZq = kT * static_cast<int>(sizeof(io_t)) / 16;
  __shared__ uint4 s_z[kW][kZLds ? kZq * 64 : 1];
  static_assert(kG == 1 || (kT == kSegSteps && kNB % kG == 0 && kT % kG == 0), "state groups share rounds evenly");
  __shared__ float s_y[kG > 1 ? kW : 1][kG > 1 ? kT : 1][kG > 1 ? 65 : 1];  // partial outputs [wave][step][lane]

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = row_longest_first(p.seq_lens, p.batch, p.seqlen, blockIdx.y);
  const int d_raw = blockIdx.x * (kW / kG) + w / kG;
  const int grp = w % kG;
  auto own = [&](int n) { return (n % kNB) % kG == grp; };  // the states this wave runs
  const bool active = d_raw < p.dim;
  const int d = active ? d_raw : p.dim - 1;
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

  const int n_chunks = (L + kChunk - 1) / kChunk;
  const int n_active_chunks = (len + kChunk - 1) / kChunk;
  // Chunks [c_lo, c_end) of the row are this workgroup's.
  const int c_lo = kG > 1 ? blockIdx.z * p.chunks_per_split : 0;
  const int c_end = kG > 1 ? min(n_chunks, c_lo + p.chunks_per_split) : n_chunks;

  for (int n = lane; n < N; n += 64) {
    float h0 = p.x0 ? p.x0[chan * N + n] : 0.f;
    if constexpr (kG > 1) {
      // the state through the splits to the left (those past the row's length keep it)
      const size_t m_ld = static_cast<size_t>(p.batch) * p.dim * N * 2;
      const float* map = p.split_map + (chan * N + n) * 2;
      const int m_end = min(static_cast<int>(blockIdx.z), (n_active_chunks + p.chunks_per_split - 1) / p.chunks_per_split);
#pragma unroll 4
      for (int m = 0; m < m_end; ++m) h0 = through_map(map[m * m_ld], map[m * m_ld + 1], h0);
    }
    s_run[w][n] = h0;
    const float an = p.A[static_cast<size_t>(d) * N + n];
    s_a[w][n] = an;
    s_a2[w][n] = an * kLog2e;
  }
  const float Dv = p.D ? p.D[d] : 0.f;
  const float bias = p.delta_bias ? p.delta_bias[d] : 0.f;
  const bool dma = kRows != kAnyRows || p.vec_bc != 0;
  float dsum_total = 0.f;  // sum of delta over all finished steps (reference residual)

  // Rounds of kNB states per chunk, padded to an even count so round g of every chunk
  // uses buffer g & 1.
  const int rounds = ((N + kNB - 1) / kNB + 1) & ~1;
  auto issue_round = [&](int r, uint4 (*buf)[2][kRowSlots]) {
    const int c = r / rounds;
    const int n0 = (r - c * rounds) * kNB;
    const int nb = min(kNB, N - n0);
    if (nb > 0) stage_round<kT, kW, kNB, bc_t>(Bb, Cb, n0, nb, c * kChunk, L, p.bc_sn, dma, buf, tid);
  };
  const int c_live = min(n_active_chunks, c_end);
  if (c_live > c_lo) issue_round(c_lo * rounds, stage0);

  for (int c = c_lo; c < c_end; ++c) {
    const int t0 = c * kChunk;
    const int tl = t0 + lane * kT;
    const bool fast = kRows == kWholeRows || t0 + kChunk <= L;  // wave-uniform
    // Reference residual slot written at this chunk's end (2048-step boundary or end of
    // the sequence), -1 if none.
    const int chunk_end = t0 + kChunk;
    const int ref_idx = (chunk_end % kRefChunk == 0 || c == n_chunks - 1)
                            ? min((chunk_end + kRefChunk - 1) / kRefChunk, p.n_ref) - 1
                            : -1;

    if (c >= n_active_chunks) {
      // Entire chunk is past this row's length: state frozen, output zero. The backward's
      // residuals (carries, y_pre) are not written here: it never reads them.
      if (active) {
        float zero[kT];
#pragma unroll
        for (int j = 0; j < kT; ++j) zero[j] = 0.f;
        if (p.out && grp == 0) store_seg<kT>(out_row, tl, L, fast, zero, kRows);
        if (p.ref_states && lane == 63 && ref_idx >= 0) {
          for (int n = 0; n < N; ++n) {
            if (!own(n)) continue;
            float* rs = p.ref_states + ((chan * p.n_ref + ref_idx) * N + n) * 2;
            rs[0] = fast_exp2(s_a2[w][n] * dsum_total);
            rs[1] = s_run[w][n];
          }
        }
        if (p.last && c == n_chunks - 1)
          for (int n = lane; n < N; n += 64)
            if (own(n)) p.last[chan * N + n] = s_run[w][n];
      }
      continue;
    }

    float dlt[kT], dlu[kT], y[kT];
    float ssum = 0.f;
    // z through LDS for whole chunks of aligned rows (wave-uniform); the first round barrier's
    // wait covers the copies.
    const bool z_lds = kZLds && active && fast && p.vec_z && p.z != nullptr && p.out != nullptr;
    if (active) {
      Seg<kT, io_t> sd, su;
      fetch(sd, dl_row, tl, L, kRows);
      fetch(su, u_row, tl, L, kRows);
      if (kZLds && z_lds) {
        const io_t* zsrc = static_cast<const io_t*>(p.z) + row + tl;
#pragma unroll
        for (int q = 0; q < kZq; ++q)
          __builtin_amdgcn_global_load_lds((gbl_void_t)(zsrc + q * (16 / static_cast<int>(sizeof(io_t)))),
                                           (lds_void_t)(&s_z[w][q * 64]), 16, 0, 0);
      }
      finish(sd, tl, L, fast, dlt, kRows);
      finish(su, tl, L, fast, y, kRows);
#pragma unroll
      for (int j = 0; j < kT; ++j) {
        const bool valid = tl + j < len;
        const float x = dlt[j] + bias;
        float dv = p.delta_softplus ? softplus(x) : x;
        dv = valid ? dv : 0.f;
        const float uu = valid ? y[j] : 0.f;
        dlt[j] = dv;
        dlu[j] = kZOH ? uu : dv * uu;  // ZOH keeps u; Euler keeps delta*u
        y[j] = grp == 0 ? Dv * uu : 0.f;
        ssum += dv;
      }
    } else {
#pragma unroll
      for (int j = 0; j < kT; ++j) dlt[j] = dlu[j] = y[j] = 0.f;
    }
    if (p.ref_states) dsum_total += wave_sum(ssum);

    auto compute_round = [&](int g, uint4 (*buf)[2][kRowSlots]) {
      const int n0 = g * kNB;
      const int nb = min(kNB, N - n0);
      for (int k = grp; k < nb; k += kG) {
        const int n = n0 + k;
        const float a2 = s_a2[w][n];
        const float run = s_run[w][n];  // read early: its wait would otherwise follow the scan
        float a[kT], bu[kT];
        float H = 0.f;
        {
          float bv[kT];
          read_staged<kT, bc_t>(buf[k][0], lane, bv);
#pragma unroll
          for (int j = 0; j < kT; ++j) {
            a[j] = fast_exp2(dlt[j] * a2);
            if constexpr (kZOH) {
              const float An = s_a[w][n];
              bu[j] = (expm1f(dlt[j] * An) * fast_rcp(An)) * bv[j] * dlu[j];
            } else {
              bu[j] = dlu[j] * bv[j];
            }
            H = __builtin_fmaf(a[j], H, bu[j]);
          }
        }
        float P = fast_exp2(a2 * ssum);
        wave_scan_affine_fwd(P, H);
        const float hend = __builtin_fmaf(P, run, H);  // true state at the lane's last step
        float h = dpp_mov<kWaveShr1, 0xF>(run, hend);   // carry-in (lane 0: running state)
        {
          float cv[kT];
          float hseg[kT / kSegSteps];  // state before each kSegSteps-step sub-segment
          read_staged<kT, bc_t>(buf[k][1], lane, cv);
#pragma unroll
          for (int j = 0; j < kT; ++j) {
            if (j % kSegSteps == 0) hseg[j / kSegSteps] = h;
            h = __builtin_fmaf(a[j], h, bu[j]);
            y[j] = __builtin_fmaf(cv[j], h, y[j]);
          }
          // Residual for the backward: the state entering every kSegSteps-step segment.
          if (p.carries) {
            float* crow = p.carries + (chan * N + n) * p.n_seg + tl / kSegSteps;
#pragma unroll
            for (int q = 0; q < kT / kSegSteps; ++q)
              if (kRows == kWholeRows || tl / kSegSteps + q < p.n_seg) crow[q] = hseg[q];
          }
        }
        const float run_new = readlane(hend, 63);
        if (lane == 0) s_run[w][n] = run_new;
        // Reference residual: (prod, h) at 2048-step chunk ends.
        if (p.ref_states && lane == 63 && ref_idx >= 0) {
          float* rs = p.ref_states + ((chan * p.n_ref + ref_idx) * N + n) * 2;
          rs[0] = fast_exp2(a2 * dsum_total);
          rs[1] = hend;
        }
        if (p.last && c == n_chunks - 1 && lane == 63) p.last[chan * N + n] = hend;
      }
    };
    const int last_round = c_live * rounds;
    for (int g = 0; g < rounds; g += 2) {
      const int r = c * rounds + g;
      wait_vmem_all();   // this thread's copies for round r have landed in LDS
      __syncthreads();   // ... and everyone's; round r-1's readers are done
      if (r + 1 < last_round) issue_round(r + 1, stage1);
      if (active) compute_round(g, stage0);
      wait_vmem_all();
      __syncthreads();
      if (r + 2 < last_round) issue_round(r + 2, stage0);
      if (active) compute_round(g + 1, stage1);
    }

    if constexpr (kG > 1) {
      // The waves of a channel finish kT / kG steps a lane each: steps [grp, grp + 1) * 64 * kV of
      // the chunk.
      constexpr int kV = kT / kG;
      const int tc = (grp * 64 + lane) * kV;  // first step within the chunk
      const int t = t0 + tc;
      float zv[kV];
      if (active && p.z) {
#pragma unroll
        for (int e = 0; e < kV; ++e)
          zv[e] = (kRows == kWholeRows || t + e < L) ? to_f32((static_cast<const io_t*>(p.z) + row)[t + e]) : 0.f;
      }
#pragma unroll
      for (int j = 0; j < kT; ++j) s_y[w][j][lane] = y[j];
      __syncthreads();  // (the next chunk's writes come after its round barriers)
      if (active && p.out) {
#pragma unroll
        for (int e = 0; e < kV; ++e) {
          float v = 0.f;
#pragma unroll
          for (int q = 0; q < kG; ++q) v += s_y[w - grp + q][(tc + e) % kT][(tc + e) / kT];
          if (p.z) {
            if (p.y_pre && t + e < len && __builtin_fabsf(zv[e]) < kZTiny)
              store_as(static_cast<io_t*>(p.y_pre) + row + t + e, v);
            v *= zv[e] * sigmoid(zv[e]);
          }
          if (kRows == kWholeRows || t + e < L) store_as(out_row + t + e, t + e < len ? v : 0.f);
        }
      }
    } else if (active && p.out) {
      if (p.z) {
        float zv[kT];
        if (kZLds && z_lds) {
          // the wave's own copies, completed at the first round barrier
          if constexpr (sizeof(io_t) == 4) {
#pragma unroll
            for (int q = 0; q < kZq; ++q) {
              const uint4 x = s_z[w][q * 64 + lane];
              zv[4 * q + 0] = __uint_as_float(x.x);
              zv[4 * q + 1] = __uint_as_float(x.y);
              zv[4 * q + 2] = __uint_as_float(x.z);
              zv[4 * q + 3] = __uint_as_float(x.w);
            }
          } else {
#pragma unroll
            for (int q = 0; q < kZq; ++q) {
              const uint4 x = s_z[w][q * 64 + lane];
              const uint32_t wd[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
              for (int k = 0; k < 4; ++k) {
                zv[8 * q + 2 * k + 0] = __uint_as_float(wd[k] << 16);
                zv[8 * q + 2 * k + 1] = __uint_as_float(wd[k] & 0xffff0000u);
              }
            }
          }
        } else {
          load_seg<kT>(static_cast<const io_t*>(p.z) + row, tl, L, fast, zv, kRows);
        }
        if (p.y_pre) {
          // The backward takes y sigma(z) from out / z; y itself is kept only where z is too
          // small for that (rare: nothing else of the row is written).
          io_t* __restrict__ yrow = static_cast<io_t*>(p.y_pre) + row;
#pragma unroll
          for (int j = 0; j < kT; ++j)
            if (tl + j < len && __builtin_fabsf(zv[j]) < kZTiny) store_as(yrow + tl + j, y[j]);
        }
#pragma unroll
        for (int j = 0; j < kT; ++j) y[j] *= zv[j] * sigmoid(zv[j]);
      }
#pragma unroll
      for (int j = 0; j < kT; ++j) y[j] = (tl + j < len) ? y[j] : 0.f;
      store_seg<kT>(out_row, tl, L, fast, y, kRows);
    }
  }
}

// The maps of a time-split forward (FwdParams::split_map): for every (channel, state) and every
// split but the last, (P, H) with P the product of the split's a_bar and H its end state from
// zero. kMapG waves share a (channel, split), each taking every kMapG-th state; lane = 8 steps.
// B rows straight from memory, the next state's fetched while this one computes. It runs only
// where most of the GPU would idle, so its time is its own latency: short chains, few states a
// wave.
constexpr int kMapW = 8;
constexpr int kMapG = 4;

template <bool kZOH, typename io_t, typename bc_t>
__global__ __launch_bounds__(kMapW * 64) void fwd_map_kernel(FwdParams p) {
  constexpr int kT = kSegSteps;
  constexpr int kChunk = 64 * kT;
  __shared__ float s_h[kMapW][kMaxN];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int b = blockIdx.y;
  const int d = blockIdx.x * (kMapW / kMapG) + w / kMapG;
  const int grp = w % kMapG;
  if (d >= p.dim || grp >= p.dstate) return;  // no barrier in this kernel: idle waves may leave
  const int L = p.seqlen;
  const int N = p.dstate;
  const int len = p.seq_lens ? min(max(p.seq_lens[b], 0), L) : L;
  const int c_lo = blockIdx.z * p.chunks_per_split;
  const int c_end = min((len + kChunk - 1) / kChunk, c_lo + p.chunks_per_split);
  if (c_lo >= c_end) return;  // no valid step: fwd_kernel skips the split
  const size_t chan = static_cast<size_t>(b) * p.dim + d;
  const long long row = b * p.io_sb + d * p.io_sd;
  const bc_t* __restrict__ Bb = static_cast<const bc_t*>(p.B) + b * p.bc_sb;
  const float* __restrict__ Ad = p.A + static_cast<size_t>(d) * N;
  const float bias = p.delta_bias ? p.delta_bias[d] : 0.f;
  if (lane < N) s_h[w][lane] = 0.f;
  float dsum = 0.f;  // sum of delta over the split
  for (int c = c_lo; c < c_end; ++c) {
    const int t0 = c * kChunk;
    const int tl = t0 + lane * kT;
    const bool fast = t0 + kChunk <= L;  // wave-uniform
    float dlt[kT], dlu[kT], bv[kT];
    Seg<kT, io_t> sd, su;
    Seg<kT, bc_t> sb;
    fetch(sd, static_cast<const io_t*>(p.delta) + row, tl, L);
    fetch(su, static_cast<const io_t*>(p.u) + row, tl, L);
    fetch(sb, Bb + grp * p.bc_sn, tl, L);
    finish(sd, tl, L, fast, dlt);
    finish(su, tl, L, fast, dlu);
    float ssum = 0.f;
#pragma unroll
    for (int j = 0; j < kT; ++j) {
      const bool valid = tl + j < len;
      const float x = dlt[j] + bias;
      const float dv = p.delta_softplus ? softplus(x) : x;
      const float uu = valid ? dlu[j] : 0.f;
      dlt[j] = valid ? dv : 0.f;
      dlu[j] = kZOH ? uu : dlt[j] * uu;
      ssum += dlt[j];
    }
    dsum += wave_sum(ssum);
    for (int n = grp; n < N; n += kMapG) {
      const float An = Ad[n];
      const float a2 = An * kLog2e;
      const float h_in = s_h[w][n];
      finish(sb, tl, L, fast, bv);
      fetch(sb, Bb + min(n + kMapG, N - 1) * p.bc_sn, tl, L);
      float H = 0.f;
#pragma unroll
      for (int j = 0; j < kT; ++j) {
        const float bu = kZOH ? (expm1f(dlt[j] * An) * fast_rcp(An)) * bv[j] * dlu[j] : dlu[j] * bv[j];
        H = __builtin_fmaf(fast_exp2(dlt[j] * a2), H, bu);
      }
      float P = fast_exp2(a2 * ssum);
      wave_scan_affine_fwd(P, H);  // lane 63: the whole chunk
      if (lane == 63) s_h[w][n] = __builtin_fmaf(P, h_in, H);
    }
  }
  for (int n = lane; n < N; n += 64) {
    if (n % kMapG != grp) continue;
    float* map = p.split_map + ((static_cast<size_t>(blockIdx.z) * p.batch * p.dim + chan) * N + n) * 2;
    map[0] = fast_exp2(Ad[n] * kLog2e * dsum);
    map[1] = s_h[w][n];
  }
}

template <int kT, int kW, int kNB, int kOcc, bool kZOH, typename io_t, typename bc_t, int kMaxS = kMaxN, int kG = 1>
static hipError_t launch_fwd_t(const FwdParams& p, hipStream_t stream) {
  constexpr int kChan = kW / kG;  // channels of a workgroup
  const dim3 grid((p.dim + kChan - 1) / kChan, p.batch, kG > 1 ? p.n_split : 1);
  if constexpr (kG > 1) {
    if (p.n_split > 1) {
      constexpr int kMapChan = kMapW / kMapG;
      const dim3 maps((p.dim + kMapChan - 1) / kMapChan, p.batch, p.n_split - 1);
      hipLaunchKernelGGL((fwd_map_kernel<kZOH, io_t, bc_t>), maps, dim3(kMapW * 64), 0, stream, p);
      const hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
    }
  }
  if constexpr (kMaxS == kMaxN && sizeof(io_t) == sizeof(bc_t)) {
    if (p.vec_bc && p.seqlen % (64 * kT) == 0) {
      hipLaunchKernelGGL((fwd_kernel<kT, kW, kNB, kOcc, kZOH, io_t, bc_t, kMaxS, kWholeRows, kG>), grid, dim3(kW * 64),
                         0, stream, p);
      return hipGetLastError();
    }
  }
  if (p.vec_bc && slots_fit<io_t>(p.seqlen))
    hipLaunchKernelGGL((fwd_kernel<kT, kW, kNB, kOcc, kZOH, io_t, bc_t, kMaxS, kSlotRows, kG>), grid, dim3(kW * 64), 0,
                       stream, p);
  else
    hipLaunchKernelGGL((fwd_kernel<kT, kW, kNB, kOcc, kZOH, io_t, bc_t, kMaxS, kAnyRows, kG>), grid, dim3(kW * 64), 0,
                       stream, p);
  return hipGetLastError();
}

// Whether four waves share a channel (`groups` workgroups with one wave each): where the grid still
// fits one pass of the narrow shape, and each wave's states outweigh the delta and u rows, softplus
// and output exchange that the four repeat. That takes more states the more workgroups a CU holds
// already (one, two, three), fewer for ZOH and for bf16 rows. Measured on MI355X, B=1 L=4096, one wave
// and four: D=400 (L=2048) float32 N=1 12.9 and 14.0 us, N=4 17.7 and 15.2; D=768 float32 N=6 42 and
// 44, N=8 47 and 44, ZOH N=2 38 and 41, N=3 46 and 42, bf16 N=3 32 and 32, N=8 50 and 39; D=1536 float32
// N=4 37 and 48, N=16 80 and 79 (L=1024 22 and 24; L=4097, the general instance, 113 and 106), ZOH N=6
// 73 and 71 (L=1024 20 and 22), N=8 88 and 75, bf16 N=11 65 and 63 (L=1024 18 and 20), N=16 81 and 72.
template <typename io_t>
static bool fwd_shares_channels(const FwdParams& p, long long groups, bool zoh) {
  const long long wgs = kFwdG * groups;
  if (wgs > kFwdNarrowSlots) return false;
  if (p.n_split > 1) return true;
  constexpr bool kHalf = sizeof(io_t) == 2;
  const bool general = !p.vec_bc || !slots_fit<io_t>(p.seqlen);
  int least;
  if (wgs <= kCUs)
    least = zoh ? 1 : 2;
  else if (wgs <= 2 * kCUs)
    least = kHalf ? (zoh ? 2 : 4) : (zoh ? 3 : 8);
  else
    least = kHalf ? (zoh ? 4 : 12) : zoh ? 7 : general ? 16 : kMaxN + 1;
  return p.dstate >= least;
}

template <bool kZOH, typename io_t, typename bc_t>
static hipError_t launch_fwd_z(const FwdParams& p, hipStream_t stream) {
  if (p.dstate > kMaxN) {
    // Wider state (float32 only): 24 KB of state tables per workgroup, two workgroups of
    // the narrow shape per CU (4 waves per SIMD).
    if constexpr (sizeof(io_t) == 4 && sizeof(bc_t) == 4) {
      if (p.dstate > kMaxNWide) return hipErrorInvalidValue;
      return launch_fwd_t<MSS_FWD_T_NARROW, MSS_FWD_W, MSS_FWD_NB, 4, kZOH, io_t, bc_t, kMaxNWide>(p, stream);
    } else {
      return hipErrorInvalidValue;
    }
  }
  // Float32 rows take the narrow shape at every grid size (measured on MI355X: B=16 D=2560
  // L=8192 with variable lengths 1.69 -> 1.39 ms, B=8 D=2048 L=4096 0.54 -> 0.48 ms); bf16
  // rows take it only when the grid fits one pass of it (B=8 D=2048 L=4096 428 vs 436 us,
  // B=8 D=1536 L=2048 167 vs 175 us wide vs narrow). Four waves to a channel: B=1 D=1536 L=16384
  // bf16 333 -> 275 us (two waves: 311; eight over rounds of eight states: 364). Over two passes
  // they lose: a B=3 D=1000 L=2051 bf16 training call takes 249 us with one wave, 268 with four.
  const long long groups = static_cast<long long>(p.batch) * ((p.dim + MSS_FWD_W - 1) / MSS_FWD_W);
  if constexpr (sizeof(io_t) == 2) {
    if (groups > kFwdNarrowSlots)
      return launch_fwd_t<MSS_FWD_T_WIDE, MSS_FWD_W, MSS_FWD_NB, MSS_FWD_OCC_WIDE, kZOH, io_t, bc_t>(p, stream);
  }
  if (fwd_shares_channels<io_t>(p, groups, kZOH))
    return launch_fwd_t<MSS_FWD_T_NARROW, MSS_FWD_W, MSS_FWD_NB, MSS_FWD_OCC_NARROW, kZOH, io_t, bc_t, kMaxN, kFwdG>(
        p, stream);
  return launch_fwd_t<MSS_FWD_T_NARROW, MSS_FWD_W, MSS_FWD_NB, MSS_FWD_OCC_NARROW, kZOH, io_t, bc_t>(p, stream);
}

}  // namespace mss
