// Implicit GEMM (gfx950, 16x16x32 bf16/fp16 MFMA -> fp32) for the forward convolution and
// for the stride phases of the input gradient.
//
//   * A workgroup owns a box of output positions (any extents whose product fits its tiles)
//     and a group of output channels. Its W waves (4 or 8) are arranged WM along the channels and
//     W/WM along the positions; each wave accumulates MB x NB fragments of 16 x 16.
//   * The GEMM input is staged per call into octet-major planes (8 channels = 16 bytes per
//     position). The region the box reads through every tap (the halo) is copied once per
//     channel chunk into LDS: one plane per octet of 8 channels, 16 bytes per position,
//     zero outside the tensor, with host-chosen pitches that keep every 16-lane B-fragment
//     read on distinct bank slots. Every tap then reuses the same LDS bytes.
//   * K is ordered (channel chunk, tap, channel). A B fragment is one 16-byte LDS read at
//     pos[q] + tap[k]; A fragments (weights) are packed per call in MFMA lane order and read
//     from global memory (L2 resident, 16 bytes per lane).
//   * The geometry (tap offsets, halo rows, box positions and per-box origins and bounds)
//     comes from small tables that the prologue launch writes once per call, so the kernel
//     has no per-axis code: its setup is a few table reads and its epilogue one store per
//     fragment for boxes inside the output.
// The input gradient of a strided convolution is split into stride phases: output
// coordinate x = r + s*j (r the phase residue); the taps that reach phase r are those with
// (r + pad - t*d) divisible by s, each at the shifted input e(t) = (r + pad - t*d) / s.
// Every phase is then a stride-1 convolution with per-tap offsets e(t), which the same
// kernel runs (blockIdx.z covers batch x phase).

#include <type_traits>

#include "convnd_geometry.h"
#include "convnd_internal.h"
#include "convnd_types.h"

namespace convnd {
namespace {

// ---- main kernel ---------------------------------------------------------------------

// Register budget: two waves per SIMD (256 VGPR+AGPR per wave) for tiles up to 16
// fragments, one wave per SIMD above. The planner's occupancy model (igemm_reg_waves in
// the host code) must match.
template <int MB, int NB>
constexpr int igemm_waves = MB * NB >= 32 ? 1 : 2;

// 16 bytes per lane from the buffer straight into LDS: lane l writes dst + 16 l (dst the same
// for every lane). Outside a lambda: the builtin's address-space cast inside one leaves the
// kernel's host stub undefined.
__device__ __forceinline__ void stage_lds16(__amdgpu_buffer_rsrc_t r, unsigned char* dst,
                                            unsigned voff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      r, (__attribute__((address_space(3))) void*)(dst), 16, voff, 0, 0, 0);
}

// body(std::integral_constant<int, 0>) .. <N - 1>.
template <int N, typename F, int I = 0>
__device__ __forceinline__ void unrolled(F&& body) {
  if constexpr (I < N) {
    body(std::integral_constant<int, I>{});
    unrolled<N, F, I + 1>(static_cast<F&&>(body));
  }
}

// The part products of one K32 step, smallest first: position parts b, weight parts a. Six of them
// into one accumulator; with NP = 8 all but the one below 2^-30 of the product, the seven cross
// products in an accumulator of their own, so that neither a truncated part nor a small product
// added to a large sum is lost.
template <typename M, int MB, int NB, int NP>
__device__ __forceinline__ void part_products(const typename M::frag (*b)[NB],
                                              const typename M::frag (*a)[MB],
                                              f32x4 (&acc)[MB][NB], f32x4 (&cross)[MB][NB]) {
  constexpr int kData[8] = {1, 2, 1, 2, 0, 1, 0, 0};
  constexpr int kOther[8] = {2, 1, 1, 0, 2, 0, 1, 0};
#pragma unroll
  for (int q = 8 - NP; q < 8; ++q) {
    f32x4(&sum)[MB][NB] = NP == 8 && q < 7 ? cross : acc;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
        sum[mb][nb] = M::run(b[kData[q]][nb], a[kOther[q]][mb], sum[mb][nb]);
  }
}

// T: GEMM operand type; O: output and bias type (T, or float for split-precision fp32).
// P: bf16 parts of split-precision fp32 staged and packed once each (3), else 1; NP: products of
// two parts that a K step adds (see part_products).
// Every per-axis quantity comes from the geometry tables (IgemmArgs::tables), so the
// kernel body is the same for every rank.
template <typename T, typename O, int MB, int NB, int WM, bool DS, int W, int P = 1, int NP = 6>
__global__ __launch_bounds__(64 * W)
__attribute__((amdgpu_waves_per_eu(igemm_waves<MB, NB>, igemm_waves<MB, NB>)))
void igemm_kernel(IgemmArgs A) {
  constexpr int kWT = 64 * W;  // threads of the workgroup
  using M = Mfma16<T>;
  using frag = typename M::frag;
  extern __shared__ __align__(16) unsigned char lds[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave % WM;
  const int wn = wave / WM;
  const int lg = lane >> 4;
  // Phases phase .. phase + plen - 1 (plen 1 unless the octet-major halo is shared by several).
  const int plen = DS ? 1 : A.plen;
  const int phase_groups = DS ? A.nphase : A.nphase / plen;
  const int n = blockIdx.z / phase_groups;
  int phase = (blockIdx.z % phase_groups) * plen;
  const int g = blockIdx.y / A.mgroups;
  const int mg = blockIdx.y % A.mgroups;

  // Consecutive workgroup ids go round-robin to the eight XCDs; give each XCD a
  // contiguous run of boxes so neighbouring halos share its L2.
  int bx = blockIdx.x;
  {
    const int nbx = gridDim.x;
    if (nbx >= 8) {
      const int q = nbx >> 3, rem = nbx & 7, x = bx & 7, idx = bx >> 3;
      bx = x * q + (x < rem ? x : rem) + idx;
    }
  }
  const char* tab = static_cast<const char*>(A.tables);
  const IgemmBox* boxp = reinterpret_cast<const IgemmBox*>(tab + A.tab_box) + phase * A.boxes + bx;
  // Uniform over the workgroup (phase with a shorter j extent; the first of a group has the
  // longest).
  if (boxp->flags & 1) return;
  const IgemmBox& box = *boxp;  // the halo: the same for every phase of the group
  int KC = box.kc;
  int KF = box.kf;

  // LDS: [octet planes (DS: nbuf sets, alternating per channel chunk) | rows: input offset
  // (-1 outside the input), with DS also LDS position offset | output offset of every box position (read
  // by the epilogue; kept out of registers during the main loop) | the phases' tap offsets,
  // 4 lane groups x tap_row each].
  int* rowin = reinterpret_cast<int*>(lds + (DS ? A.nbuf : 1) * A.halo_bytes);
  const int rows4 = (A.rows + 3) & ~3;
  int* rowlds = rowin + rows4;  // (direct staging)
  int* posout = DS ? rowlds + rows4 : rowlds;
  int* ltaps = posout + ((A.box_vol + 3) & ~3);
  const int4* pt = reinterpret_cast<const int4*>(tab + A.tab_pos);
  for (int q = tid; q < A.box_vol; q += kWT) posout[q] = pt[q].y;
  {
    const int* gt = reinterpret_cast<const int*>(tab + A.tab_taps) + phase * 4 * A.tap_row;
    for (int i = tid; i < plen * 4 * A.tap_row; i += kWT) ltaps[i] = gt[i];
  }
  // Input offset of every halo row, for split tap tc: its shift moves the origin and the bounds
  // along the split axes.
  auto fill_rows = [&](int tc) {
    const int4* rt = reinterpret_cast<const int4*>(tab + A.tab_rows);
    unsigned long long lo = box.lo, hi = box.hi;
    int in_base = box.in_base;
    if (!DS && A.tsplit > 0) {
      const int2 e = reinterpret_cast<const int2*>(tab + A.tab_split)[tc];
      const int vol0 = A.in_vol / A.in_size[0];
      in_base += e.x * vol0;
      auto bound = [&](int a, int h) {
        const int lo_a = h >= 0 ? 0 : (-h < A.hext[a] ? -h : A.hext[a]);
        int hi_a = A.in_size[a] - h;
        hi_a = hi_a < 0 ? 0 : (hi_a < A.hext[a] ? hi_a : A.hext[a]);
        const unsigned long long keep = ~(0xffull << (8 * a));
        lo = (lo & keep) | (static_cast<unsigned long long>(lo_a) << (8 * a));
        hi = (hi & keep) | (static_cast<unsigned long long>(hi_a) << (8 * a));
      };
      bound(0, box.org[0] + e.x);
      if (A.tsplit > 1) {
        in_base += e.y * (vol0 / A.in_size[1]);
        bound(1, box.org[1] + e.y);
      }
    }
    for (int r = tid; r < A.rows; r += kWT) {
      const int4 e = rt[r];
      const unsigned long long h =
          static_cast<unsigned>(e.z) | (static_cast<unsigned long long>(static_cast<unsigned>(e.w)) << 32);
      const bool ok = swar_all_ge(h, lo, kGuard8) && swar_all_less(h, hi, kGuard8, kOnes8);
      rowin[r] = ok ? in_base + e.y : -1;
      if constexpr (DS) rowlds[r] = e.x;
    }
  };
  fill_rows(0);
  // Per lane and position block: LDS byte offset of the lane's B-fragment position.
  int pbase[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) pbase[nb] = pt[(wn * NB + nb) * 16 + (lane & 15)].x;
  // Tap offsets of this lane group (LDS, read in pairs of steps ahead of use); the partial
  // last step separately.
  const int* tp = ltaps + lg * A.tap_row;
  int tail_tap = reinterpret_cast<const int*>(tab + A.tab_tail)[phase * 4 + lg];
  // Bias of this wave's output channels, loaded now so its latency hides behind the loop.
  const int mt0 = (mg * WM + wm) * MB;  // first m-tile of this wave
  // The MFMAs run with the positions as the A operand, so D = (W X)^T: lane l holds output
  // channel (l % 16) of its m-tile at four consecutive box positions 4*(l/16) .. +3.
  float bias_v[MB];
  {
    const O* bias = static_cast<const O*>(A.bias);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const int m = (mt0 + mb) * 16 + (lane & 15);
      bias_v[mb] =
          (bias != nullptr && m < A.cout_g) ? static_cast<float>(bias[g * A.cout_g + m]) : 0.f;
    }
  }

  const int hlast = A.hlast;
  const int corg = box.corg;
  const int last_size = A.last_size;
  const int noct = A.noct;
  const T* in = static_cast<const T*>(A.in);
  const frag* wp = static_cast<const frag*>(A.wpk);
  f32x4 acc[MB][NB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
  // Sums of the cross products (P == 3, NP == 8; unused otherwise).
  f32x4 cross[MB][NB];
  auto clear_cross = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) cross[mb][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  clear_cross();

  const size_t wpart = (size_t)A.mtiles_padded * 64;  // fragments per part of a K32 step
  const size_t wstep = P * wpart;                     // fragments per K32 step
  constexpr unsigned kPast = 0xffffffe0u;  // past every staged tensor (planner: < kPast bytes)
  const __amdgpu_buffer_rsrc_t srsrc =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(in), 0, A.in_bytes, 0x00020000);

  // MFMAs of chunk ck (split tap, channel chunk) over the halo planes at hb. `issue` runs once, after the first
  // weight fragments and B fragments are requested and before the loop (the next chunk's
  // staging loads go there, behind this chunk's first weight loads in the load queue).
  auto mma_chunk = [&](int ck, const unsigned char* hb, auto&& issue) __attribute__((always_inline)) {
    const frag* wck = wp +
                      ((size_t)((phase * A.groups + g) * A.tcount * A.nchunk + ck) * A.kc_max) * wstep +
                      (size_t)mt0 * 64 + lane;
    if constexpr (P == 3) {
      // Split-precision fp32, each K32 step from the three parts of both operands: 3 MB weight
      // and 3 NB position fragments feed 6 MB NB MFMAs, half the operand traffic per MFMA of
      // six copies along K (which a small tile is bound by: the weights through the vector L1
      // at 64 B per clock, the positions through LDS). Weights kRing - 1 steps ahead (ring),
      // position fragments one step ahead, tap offsets kUnroll at a time one iteration ahead.
      // 48 -> 24 channels, 3^4 taps, [2,.,13,11,10,15] (input gradient): 111 -> 78 us.
      constexpr int kRing = MB * NB <= 2 ? 8 : (MB == 1 ? 4 : 2);
      constexpr int kUnroll = kRing < 4 ? 4 : kRing;
      static_assert(kUnroll <= kTapPad && kUnroll % kRing == 0 && kUnroll % 4 == 0, "tap prefetch");
      const int ppitch = noct * A.plane_bytes;  // LDS bytes from one part's planes to the next
      if (KF > 0) {
        const int last = KF - 1;
        auto wstep_at = [&](int k) { return (size_t)(k < last ? k : last) * wstep; };
        frag ar[kRing][3][MB], br[2][3][NB];
        auto load_w = [&](frag (*a)[MB], int k) {
          const size_t at = wstep_at(k);
#pragma unroll
          for (int p = 0; p < 3; ++p)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) a[p][mb] = wck[at + p * wpart + mb * 64];
        };
        auto load_b = [&](frag (*b)[NB], int tap) {
#pragma unroll
          for (int p = 0; p < 3; ++p)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
              b[p][nb] = *reinterpret_cast<const frag*>(hb + pbase[nb] + tap + p * ppitch);
        };
        int4 tq[kUnroll / 4];
        auto tap_of = [](const int4* q, int j) {
          const int4 v = q[j >> 2];
          return (j & 3) == 0 ? v.x : (j & 3) == 1 ? v.y : (j & 3) == 2 ? v.z : v.w;
        };
#pragma unroll
        for (int j = 0; j < kRing - 1; ++j) load_w(ar[j], j);
#pragma unroll
        for (int j = 0; j < kUnroll / 4; ++j) tq[j] = *reinterpret_cast<const int4*>(tp + 4 * j);
        load_b(br[0], tap_of(tq, 0));
        __builtin_amdgcn_sched_barrier(0);
        issue();
        // Step i of an iteration at kc; tb: tap offset of the step after it.
        auto step = [&](auto ic, int kc, int tb) {
          constexpr int i = decltype(ic)::value;
          load_b(br[(i + 1) & 1], tb);
          load_w(ar[(i + kRing - 1) % kRing], kc + i + kRing - 1);
          __builtin_amdgcn_sched_barrier(0);
          part_products<M, MB, NB, NP>(br[i & 1], ar[i % kRing], acc, cross);
          __builtin_amdgcn_sched_barrier(0);
        };
        int kc = 0;
        for (; kc + kUnroll <= KF; kc += kUnroll) {
          int4 tn[kUnroll / 4];
#pragma unroll
          for (int j = 0; j < kUnroll / 4; ++j)
            tn[j] = *reinterpret_cast<const int4*>(tp + kc + kUnroll + 4 * j);
          unrolled<kUnroll>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            step(ic, kc, i + 1 < kUnroll ? tap_of(tq, i + 1) : tap_of(tn, i + 1 - kUnroll));
          });
#pragma unroll
          for (int j = 0; j < kUnroll / 4; ++j) tq[j] = tn[j];
        }
        const int left = KF - kc;  // 0 to kUnroll - 1 whole steps remain
        unrolled<kUnroll - 1>([&](auto ic) {
          constexpr int i = decltype(ic)::value;
          if (i < left) step(ic, kc, tap_of(tq, i + 1));
        });
      } else {
        issue();
      }
      if (KC > KF) {
        // The partial last step: zero position fragments past the phase's last tap.
        frag at[3][MB], bt[3][NB];
#pragma unroll
        for (int p = 0; p < 3; ++p) {
#pragma unroll
          for (int mb = 0; mb < MB; ++mb) at[p][mb] = wck[(size_t)KF * wstep + p * wpart + mb * 64];
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) {
            u32x4 v = *reinterpret_cast<const u32x4*>(hb + pbase[nb] + (tail_tap < 0 ? 0 : tail_tap) +
                                                      p * ppitch);
            if (tail_tap < 0) v = u32x4{0u, 0u, 0u, 0u};
            bt[p][nb] = __builtin_bit_cast(frag, v);
          }
        }
        part_products<M, MB, NB, NP>(bt, at, acc, cross);
      }
      return;
    }
    if (KF > 0 && MB * NB <= 4 && std::is_same<O, float>::value) {
      // Small tiles (at most 4 MFMAs per K step) of split-precision fp32: their packed weights
      // (six part products per channel) mostly come from beyond L2, and a step's MFMAs take
      // far less than that round trip. The weights are therefore loaded kRing - 1 steps ahead
      // into a ring of kRing fragment sets (16 for one M tile, 8 for two, within the register
      // budget) and the B fragments 3 steps ahead into a ring of 4, kRing steps per
      // iteration. Tap offsets come kRing at a time, one iteration ahead (the table repeats
      // the last whole step for kTapPad entries past the end, so every prefetch stays inside
      // the halo). Measured: C4 fp32 step 3.40 -> 2.94 ms; with 16-bit data, whose weights
      // stay in L2, no gain on C4 and 7 % slower on C5's short K loops.
      constexpr int kRing = MB == 1 ? 16 : 8;
      static_assert(kRing <= kTapPad && kRing % 4 == 0, "tap prefetch inside the tap table");
      const int last = KF - 1;
      auto wstep_at = [&](int k) { return (size_t)(k < last ? k : last) * wstep; };
      frag ar[kRing][MB], br[4][NB];
#pragma unroll
      for (int j = 0; j < kRing - 1; ++j)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) ar[j][mb] = wck[wstep_at(j) + mb * 64];
      int4 tq[kRing / 4];
#pragma unroll
      for (int j = 0; j < kRing / 4; ++j) tq[j] = *reinterpret_cast<const int4*>(tp + 4 * j);
      auto tap_of = [](const int4* q, int j) {
        const int4 v = q[j >> 2];
        return (j & 3) == 0 ? v.x : (j & 3) == 1 ? v.y : (j & 3) == 2 ? v.z : v.w;
      };
#pragma unroll
      for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
          br[j][nb] = *reinterpret_cast<const frag*>(hb + pbase[nb] + tap_of(tq, j));
      __builtin_amdgcn_sched_barrier(0);
      issue();
      __builtin_amdgcn_sched_barrier(0);
      int kc = 0;
      for (; kc + kRing - 1 < KF; kc += kRing) {
        int4 tn[kRing / 4];
#pragma unroll
        for (int j = 0; j < kRing / 4; ++j)
          tn[j] = *reinterpret_cast<const int4*>(tp + kc + kRing + 4 * j);
#pragma unroll
        for (int i = 0; i < kRing; ++i) {
          const int tb = i + 3 < kRing ? tap_of(tq, i + 3) : tap_of(tn, i + 3 - kRing);
#pragma unroll
          for (int nb = 0; nb < NB; ++nb)
            br[(i + 3) & 3][nb] = *reinterpret_cast<const frag*>(hb + pbase[nb] + tb);
          const size_t ws = wstep_at(kc + i + kRing - 1);
#pragma unroll
          for (int mb = 0; mb < MB; ++mb) ar[(i + kRing - 1) % kRing][mb] = wck[ws + mb * 64];
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
              acc[mb][nb] = M::run(br[i & 3][nb], ar[i][mb], acc[mb][nb]);
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int j = 0; j < kRing / 4; ++j) tq[j] = tn[j];
      }
      // 0 to kRing - 1 whole steps remain: weights of step kc + i in ar[i], B fragments of the
      // first three in br[0..2].
      const int left = KF - kc;
#pragma unroll
      for (int i = 0; i < kRing - 1; ++i) {
        if (i < left) {
          if (i + 3 < left) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
              br[(i + 3) & 3][nb] =
                  *reinterpret_cast<const frag*>(hb + pbase[nb] + tap_of(tq, i + 3));
          }
#pragma unroll
          for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
              acc[mb][nb] = M::run(br[i & 3][nb], ar[i][mb], acc[mb][nb]);
        }
      }
    } else if (KF > 0) {
      // Software pipeline over the whole steps, four steps per iteration: weights three
      // K32 steps ahead (global, L2-resident; four fragment sets in flight), B fragments
      // one step ahead (LDS), tap offsets four at a time a full iteration ahead (LDS; the
      // table repeats the last whole step past the end, so every prefetch is unconditional
      // and stays inside the halo). The scheduling fences keep each step's loads ahead of
      // the MFMAs they overlap (left alone, the scheduler sinks every load next to its
      // first use and the prefetch distance collapses).
      const int last = KF - 1;
      auto wstep_at = [&](int k) { return (size_t)(k < last ? k : last) * wstep; };
      frag a0[MB], a1[MB], a2[MB], a3[MB], b0[NB], b1[NB];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) a0[mb] = wck[mb * 64];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) a1[mb] = wck[wstep_at(1) + mb * 64];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) a2[mb] = wck[wstep_at(2) + mb * 64];
      int4 t = *reinterpret_cast<const int4*>(tp);
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
        b0[nb] = *reinterpret_cast<const frag*>(hb + pbase[nb] + t.x);
      __builtin_amdgcn_sched_barrier(0);
      issue();
      __builtin_amdgcn_sched_barrier(0);
      // One step: B fragments of the next step into bn (tap offset tn), weights of step
      // ks into al, MFMAs of the current step (bc, ac).
      auto step = [&](frag* bn, int tn, frag* al, int ks, const frag* bc, const frag* ac) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
          bn[nb] = *reinterpret_cast<const frag*>(hb + pbase[nb] + tn);
        const size_t ws = wstep_at(ks);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) al[mb] = wck[ws + mb * 64];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = M::run(bc[nb], ac[mb], acc[mb][nb]);
        __builtin_amdgcn_sched_barrier(0);
      };
      int kc = 0;
      for (; kc + 3 < KF; kc += 4) {
        const int4 tn = *reinterpret_cast<const int4*>(tp + kc + 4);
        step(b1, t.y, a3, kc + 3, b0, a0);
        step(b0, t.z, a0, kc + 4, b1, a1);
        step(b1, t.w, a1, kc + 5, b0, a2);
        step(b0, tn.x, a2, kc + 6, b1, a3);
        t = tn;
      }
      // 0 to 3 whole steps remain: B of step kc is in b0, weights of kc .. kc+2 in a0..a2.
      const int left = KF - kc;
      if (left >= 1) {
        if (left >= 2) {
#pragma unroll
          for (int nb = 0; nb < NB; ++nb)
            b1[nb] = *reinterpret_cast<const frag*>(hb + pbase[nb] + t.y);
        }
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = M::run(b0[nb], a0[mb], acc[mb][nb]);
      }
      if (left >= 2) {
        if (left >= 3) {
#pragma unroll
          for (int nb = 0; nb < NB; ++nb)
            b0[nb] = *reinterpret_cast<const frag*>(hb + pbase[nb] + t.z);
        }
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = M::run(b1[nb], a1[mb], acc[mb][nb]);
      }
      if (left >= 3) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = M::run(b0[nb], a2[mb], acc[mb][nb]);
      }
    } else {
      issue();
    }
    if (KC > KF) {
      // The partial last step holds k-groups past the phase's last tap (offset -1): their
      // B fragments are zero, so padding never multiplies a zero weight by a non-finite
      // input.
      frag at[MB], bt[NB];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) at[mb] = wck[(size_t)KF * wstep + mb * 64];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        u32x4 v = *reinterpret_cast<const u32x4*>(hb + pbase[nb] + (tail_tap < 0 ? 0 : tail_tap));
        if (tail_tap < 0) v = u32x4{0u, 0u, 0u, 0u};
        bt[nb] = __builtin_bit_cast(frag, v);
      }
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = M::run(bt[nb], at[mb], acc[mb][nb]);
    }
  };

  // Epilogue: straight from the accumulators. A lane's four values are box positions
  // 4*lg .. 4*lg+3 of its position block. In a box inside the output whose rows have whole runs
  // of 4 positions on a unit output step they are adjacent: one 8-byte store for 16-bit
  // O, 16 bytes for float. Otherwise every position has its own offset and bounds check, and a
  // lane whose four positions are all inside and adjacent still stores them at once.
  // The activation is a compile-time constant of each epilogue copy, dispatched once: every
  // copy's code is contiguous (a launch starts on a cold instruction cache, and per-element
  // branches over the activations' code would spread the executed instructions over many
  // more cache lines).
  auto store4 = [](O* dst, const O* v) {
    if constexpr (sizeof(O) == 2) {
      uint2 w;
      w.x = __builtin_bit_cast(unsigned short, v[0]) |
            ((unsigned)__builtin_bit_cast(unsigned short, v[1]) << 16);
      w.y = __builtin_bit_cast(unsigned short, v[2]) |
            ((unsigned)__builtin_bit_cast(unsigned short, v[3]) << 16);
      *reinterpret_cast<uint2*>(dst) = w;
    } else {
      *reinterpret_cast<f32x4*>(dst) = f32x4{v[0], v[1], v[2], v[3]};
    }
  };
  // (Inlined by force: left out of line for the largest tile, it put the accumulators in scratch.)
  auto epilogue = [&](auto act_c) __attribute__((always_inline)) {
    constexpr int kAct = decltype(act_c)::value;
    const int flags = boxp->flags;
    O* out = static_cast<O*>(A.out);
    const size_t chan0 = (size_t)n * A.cout_total + (size_t)g * A.cout_g;
    O* obox = out + boxp->out_origin;
    if (A.out_cl) {
      // Channels-last output: output channel m of position q at
      // ((n*out_vol + q)*cout_total + g*cout_g + m); sixteen lanes write one position's 16
      // consecutive channels.
      const size_t ostride = static_cast<size_t>(A.cout_total);
      O* ocl = out + ((size_t)n * A.out_vol + boxp->out_origin) * ostride + (size_t)g * A.cout_g;
      const bool inside = A.packed_ok && (flags & 2);
      int off[NB][4];
      {
        const unsigned long long lim = boxp->lim;
        const unsigned long long guard = A.coord_bits == 16 ? kGuard16 : kGuard8;
        const unsigned long long ones = A.coord_bits == 16 ? kOnes16 : kOnes8;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int q = (wn * NB + nb) * 16 + 4 * lg + i;
            if (inside) {
              off[nb][i] = posout[q];
            } else {
              const int4 e = pt[q];
              const unsigned long long c = static_cast<unsigned>(e.z) |
                                           (static_cast<unsigned long long>(static_cast<unsigned>(e.w)) << 32);
              off[nb][i] = swar_all_less(c, lim, guard, ones) ? e.y : -1;
            }
          }
        }
      }
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        const int m = (mt0 + mb) * 16 + (lane & 15);
        if (m >= A.cout_g) continue;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (off[nb][i] >= 0)
              ocl[(size_t)off[nb][i] * ostride + m] =
                  static_cast<O>(epilogue_act(acc[mb][nb][i] + bias_v[mb], kAct));
        }
      }
    } else if (A.packed_ok && (flags & 2)) {
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        const int m = (mt0 + mb) * 16 + (lane & 15);
        if (m >= A.cout_g) continue;
        O* orow = obox + (chan0 + m) * A.out_vol;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          O v[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = static_cast<O>(epilogue_act(acc[mb][nb][i] + bias_v[mb], kAct));
          store4(orow + posout[(wn * NB + nb) * 16 + 4 * lg], v);
        }
      }
    } else {
      const unsigned long long lim = boxp->lim;
      const unsigned long long guard = A.coord_bits == 16 ? kGuard16 : kGuard8;
      const unsigned long long ones = A.coord_bits == 16 ? kOnes16 : kOnes8;
      int off[NB][4];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int4 e = pt[(wn * NB + nb) * 16 + 4 * lg + i];
          const unsigned long long c =
              static_cast<unsigned>(e.z) | (static_cast<unsigned long long>(static_cast<unsigned>(e.w)) << 32);
          off[nb][i] = swar_all_less(c, lim, guard, ones) ? e.y : -1;
        }
      }
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        const int m = (mt0 + mb) * 16 + (lane & 15);
        if (m >= A.cout_g) continue;
        O* orow = obox + (chan0 + m) * A.out_vol;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          O v[4];
#pragma unroll
          for (int i = 0; i < 4; ++i)
            v[i] = static_cast<O>(epilogue_act(acc[mb][nb][i] + bias_v[mb], kAct));
          const int o0 = off[nb][0];
          if (o0 >= 0 && off[nb][1] == o0 + 1 && off[nb][2] == o0 + 2 && off[nb][3] == o0 + 3) {
            store4(orow + o0, v);
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (off[nb][i] >= 0) orow[off[nb][i]] = v[i];
          }
        }
      }
    }
  };
  auto store_outputs = [&]() __attribute__((always_inline)) {
    if constexpr (P == 3 && NP == 8) {
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[mb][nb] += cross[mb][nb];
    }
    switch (A.act) {
      case CONVND_HIP_ACT_RELU:
        epilogue(std::integral_constant<int, CONVND_HIP_ACT_RELU>{});
        break;
      case CONVND_HIP_ACT_GELU:
        epilogue(std::integral_constant<int, CONVND_HIP_ACT_GELU>{});
        break;
      case CONVND_HIP_ACT_GELU_TANH:
        epilogue(std::integral_constant<int, CONVND_HIP_ACT_GELU_TANH>{});
        break;
      default:
        epilogue(std::integral_constant<int, CONVND_HIP_ACT_NONE>{});
    }
  };

  if constexpr (DS) {
    // Halo staged straight from the channels-first operand [N][cin_total][in_vol]. A task
    // (halo row r, run jj, octet o; octet fastest) loads the run of 8 consecutive last-axis
    // elements starting at input column 8*(jlo + jj) for the octet's 8 channels (eight
    // 16-byte loads, zero past the tensor or for rows outside it), transposes the 8 x 8
    // block in registers (v_perm) and writes each column inside the halo and the input as
    // one 16-byte position of the octet plane. Halo columns outside the input's last axis
    // are never written by a task: they are cleared once, in every buffer. With two buffers
    // they alternate per chunk: the next chunk's loads are issued inside this chunk's MFMA loop
    // setup and written after it, so staging overlaps the MFMAs (nbuf 2; with nbuf 1 the
    // loads still overlap, the writes wait for the chunk's last reads).
    constexpr int kPf = MB * NB >= 32 ? 2 : 1;  // tasks per thread held in registers
    const int nrun = A.nrun;
    const int ntask = A.rows * nrun * A.noct;
    const int jlo = corg > 0 ? (corg >> 3) : 0;
    const int clast = (corg + hlast < last_size ? corg + hlast : last_size) - 1;
    const int nrun_box = clast >= jlo * 8 ? (clast >> 3) - jlo + 1 : 0;
    const unsigned img_chan = static_cast<unsigned>(n * A.cin_total + g * A.cin_g);
    const unsigned in_vol = static_cast<unsigned>(A.in_vol);
    const unsigned in_bytes = static_cast<unsigned>(A.in_bytes);
    // Channels-last: element (n, position, channel) at (n*in_vol + position)*cin_total + channel;
    // load i of a task is position i of the run (its 8 channels), not channel i.
    const bool in_cl = A.in_cl != 0;
    const unsigned cl_img = static_cast<unsigned>(n) * in_vol;
    const unsigned cl_stride = static_cast<unsigned>(A.cin_total);
    auto task_load = [&](int ck, int t, u32x4* v) {
      const int rt = fast_div(t, A.div_noct);
      const int o = t - rt * noct;
      const int r = rt / nrun;
      const int jj = rt - r * nrun;
      const int ro = (t < ntask && jj < nrun_box) ? rowin[r] : -1;
      const unsigned chan = img_chan + static_cast<unsigned>(ck * A.cc + o * 8);
      const unsigned pos = static_cast<unsigned>(ro + (jlo + jj) * 8);
      const unsigned cl_chan = static_cast<unsigned>(g * A.cin_g + ck * A.cc + o * 8);
      unsigned offs[8];
      bool straddle = false;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const unsigned off =
            ro < 0 ? kPast
                   : (in_cl ? ((cl_img + pos + i) * cl_stride + cl_chan) * 2u
                            : ((chan + i) * in_vol + pos) * 2u);
        offs[i] = off;
        v[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(srsrc, off, 0, 0));
        straddle = straddle || (off < in_bytes && off + 16u > in_bytes);
      }
      // The buffer's range check is per dword: a dword straddling the tensor's end reads
      // zero, valid half included. A run that crosses the end loads element by element (one
      // rarely taken branch per task, so the common path's code stays contiguous).
      if (straddle) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const unsigned off = offs[i];
          if (off < in_bytes && off + 16u > in_bytes) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              const unsigned lo = __builtin_amdgcn_raw_buffer_load_b16(srsrc, off + 4u * k, 0, 0);
              const unsigned hi =
                  __builtin_amdgcn_raw_buffer_load_b16(srsrc, off + 4u * k + 2u, 0, 0);
              v[i][k] = lo | (hi << 16);
            }
          }
        }
      }
    };
    auto task_store = [&](int t, const u32x4* v, unsigned char* buf) {
      const int rt = fast_div(t, A.div_noct);
      const int o = t - rt * noct;
      const int r = rt / nrun;
      const int jj = rt - r * nrun;
      if (t >= ntask || jj >= nrun_box) return;
      const int c0 = (jlo + jj) * 8;
      unsigned char* rowp = buf + o * A.plane_bytes + (rowlds[r] - corg) * 16;
      if (in_cl) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int c = c0 + e;
          if (c >= corg && c <= clast) *reinterpret_cast<u32x4*>(rowp + c * 16) = v[e];
        }
        return;
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int c = c0 + e;
        if (c >= corg && c <= clast) {
          const unsigned sel = (e & 1) ? 0x07060302u : 0x05040100u;
          const int d = e >> 1;
          u32x4 w;
          w.x = __builtin_amdgcn_perm(v[1][d], v[0][d], sel);
          w.y = __builtin_amdgcn_perm(v[3][d], v[2][d], sel);
          w.z = __builtin_amdgcn_perm(v[5][d], v[4][d], sel);
          w.w = __builtin_amdgcn_perm(v[7][d], v[6][d], sel);
          *reinterpret_cast<u32x4*>(rowp + c * 16) = w;
        }
      }
    };
    // Tasks past the ones held in registers: loaded and written in place (not overlapped).
    auto stage_rest = [&](int ck, unsigned char* buf) {
      // Two tasks per pass, both tasks' loads in flight before the stores.
      for (int t = tid + kPf * kWT; t < ntask; t += 2 * kWT) {
        u32x4 v0[8], v1[8];
        task_load(ck, t, v0);
        task_load(ck, t + kWT, v1);
        task_store(t, v0, buf);
        task_store(t + kWT, v1, buf);
      }
    };
    __syncthreads();  // row tables in LDS
    {
      const int zl = corg < 0 ? (-corg < hlast ? -corg : hlast) : 0;
      const int rstart = last_size - corg > zl ? last_size - corg : zl;  // first right column
      const int zr = hlast > rstart ? hlast - rstart : 0;
      const int zc = zl + zr;
      const int nz = A.nbuf * A.noct * A.rows * zc;
      for (int i = tid; i < nz; i += kWT) {
        const int col = i % zc;
        const int rest = i / zc;
        const int r = rest % A.rows;
        const int bo = rest / A.rows;  // buffer * noct + octet
        const int hp = col < zl ? col : rstart + (col - zl);
        *reinterpret_cast<u32x4*>(lds + bo * A.plane_bytes + (rowlds[r] + hp) * 16) =
            u32x4{0u, 0u, 0u, 0u};
      }
    }
    u32x4 pf[kPf][8];
#pragma unroll
    for (int q = 0; q < kPf; ++q) task_load(0, tid + q * kWT, pf[q]);
#pragma unroll
    for (int q = 0; q < kPf; ++q) task_store(tid + q * kWT, pf[q], lds);
    stage_rest(0, lds);
    __syncthreads();
    // nbuf 2: chunk ck reads buffer ck & 1 while the next chunk goes to the other one;
    // nbuf 1: one buffer, rewritten after every wave is done with it.
    const int alt = A.nbuf == 2 ? A.halo_bytes : 0;
    for (int ck = 0; ck < A.nchunk; ++ck) {
      unsigned char* cur = lds + (ck & 1) * alt;
      unsigned char* nxt = lds + ((ck + 1) & 1) * alt;
      const bool more = ck + 1 < A.nchunk;
      mma_chunk(ck, cur, [&]() {
        if (more) {
#pragma unroll
          for (int q = 0; q < kPf; ++q) task_load(ck + 1, tid + q * kWT, pf[q]);
        }
      });
      if (more) {
        if (A.nbuf == 1) __syncthreads();  // every wave is done reading the buffer
#pragma unroll
        for (int q = 0; q < kPf; ++q) task_store(tid + q * kWT, pf[q], nxt);
        stage_rest(ck + 1, nxt);
        __syncthreads();  // next chunk's halo written
      }
    }
    store_outputs();
  } else {
    // Halo staged straight to LDS from the octet-major copy, every load in flight at once: a
    // wave's load writes 64 consecutive LDS positions of a plane (1 KB), each lane reading the
    // position's source (slot table: halo row and column; zero past the staged tensor for
    // padding and for positions outside the input), the same positions of all planes in turn.
    // With split taps the halo is restaged per tap of the outer axes: at rank 6 (3^6 taps) it is
    // what lets a box of 256 positions, or all three parts of fp32, fit LDS. [1,8,8^6] -> 16
    // channels, forward / input gradient: fp32 696 / 1417 -> 266 / 503 us, bf16 154 / 274 ->
    // 105 / 131 us.
    const int plane_pos = A.plane_bytes >> 4;  // a multiple of 64
    // Octet planes of this image and group: [cin_total/8][in_vol][8], addressed in bytes from
    // the staged tensor's base.
    const unsigned img_base =
        static_cast<unsigned>(((size_t)n * (A.cin_total >> 3) + (size_t)(g * (A.cin_g >> 3))) *
                              A.in_vol * 16);
    const int* slots = reinterpret_cast<const int*>(tab + A.tab_slots);
    const unsigned plane_step = static_cast<unsigned>(A.in_vol) * 16u;
    auto stage = [&](int ck) {
      const unsigned cbase = img_base + static_cast<unsigned>(ck * noct) * plane_step;
      for (int i0 = __builtin_amdgcn_readfirstlane(wave) * 64; i0 < plane_pos; i0 += kWT) {
        const int e = slots[i0 + lane];
        const int ro = e >= 0 ? rowin[e >> 8] : -1;
        const int cl = corg + (e & 0xff);
        const bool ok = ro >= 0 && cl >= 0 && cl < last_size;
        unsigned off = ok ? cbase + static_cast<unsigned>(ro + cl) * 16u : kPast;
        unsigned char* dst = lds + i0 * 16;
#pragma unroll 1
        for (int p = 0; p < P; ++p) {
          unsigned po = off;
#pragma unroll 1
          for (int o = 0; o < noct; ++o) {
            stage_lds16(srsrc, dst, po);
            dst += A.plane_bytes;
            if (ok) po += plane_step;
          }
          if (ok) off += static_cast<unsigned>(A.part_octs) * plane_step;
        }
      }
    };
    // The phases of the group (one, unless plen > 1) from one halo: with several there is one
    // chunk, staged for the first. Half of a strided input gradient's workgroup was staging the
    // halo that its phases share: 128 <- 64 channels in 4 groups, stride 2 on three axes, 24^3 x 12,
    // 103 -> 79 us.
    const bool taps_inner = P == 1 && std::is_same<O, float>::value && A.taps_inner;
    for (int q = 0;;) {
      for (int tc = 0, ck = 0, last = 0;;) {
        // Every wave is past the staging that read the rows (the last chunk's barrier).
        if (tc != last) fill_rows(tc);
        last = tc;
        if (q == 0) {
          // Row table written, and every wave done reading the chunk before.
          __syncthreads();
          stage(ck);
          __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wave's loads have landed in LDS
          __syncthreads();
        }
        mma_chunk(tc * A.nchunk + ck, lds, []() {});
        // Chunks of a split tap, then the next tap; or the taps of a chunk (IgemmArgs::taps_inner).
        if (taps_inner ? ++tc == A.tcount : ++ck == A.nchunk) {
          if (taps_inner ? ++ck == A.nchunk : ++tc == A.tcount) break;
          (taps_inner ? tc : ck) = 0;
        }
      }
      store_outputs();
      do {
        if (++q == plen) return;
        ++phase;
        boxp += A.boxes;
      } while (boxp->flags & 1);
      KC = boxp->kc;
      KF = boxp->kf;
      tp = ltaps + (q * 4 + lg) * A.tap_row;
      tail_tap = reinterpret_cast<const int*>(tab + A.tab_tail)[phase * 4 + lg];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
      clear_cross();
    }
  }
}

// The compiled implicit-GEMM tiles: (MB, NB, WM) with four waves per workgroup, and the
// eight-wave ones (direct staging, 16-bit data): one workgroup of two waves per SIMD per CU,
// whose waves are issued evenly where two four-wave workgroups sharing a CU are not (the
// older one's waves run ahead and the other finishes alone).
#define CONVND_IGEMM_TILES(X)                                                             \
  X(1, 2, 1) X(1, 4, 1) X(1, 8, 1) X(2, 2, 1) X(2, 4, 1) X(2, 8, 1) X(4, 2, 1) X(4, 4, 1) \
  X(4, 8, 1) X(1, 4, 2) X(1, 8, 2) X(2, 4, 2) X(2, 8, 2) X(1, 4, 4) X(1, 8, 4)
#define CONVND_IGEMM_TILES8(X) \
  X(4, 4, 1) X(2, 4, 1) X(4, 2, 1) X(2, 8, 1) X(1, 8, 1) X(1, 4, 1) X(1, 2, 1) X(2, 2, 1)

// Split precision from three parts (two waves per SIMD, 256 registers each); with the second
// accumulators of eight products, the tiles that fit them without scratch.
#define CONVND_IGEMM_TILES_P3X8(X) \
  X(1, 2, 1) X(1, 4, 1) X(2, 2, 1) X(1, 4, 2) X(2, 2, 2) X(1, 4, 4)
#define CONVND_IGEMM_TILES_P3(X) \
  CONVND_IGEMM_TILES_P3X8(X) X(2, 4, 1) X(2, 4, 2) X(4, 2, 1)

hipError_t igemm_dispatch_p3(int mb, int nb, const IgemmArgs& a, size_t lds, hipStream_t s) {
  const dim3 grid(a.boxes, a.groups * a.mgroups, a.batch * (a.nphase / a.plen));
#define CONVND_IGEMM_CASE_NP(MBV, NBV, WMV, NPV)                                               \
  if (mb == MBV && nb == NBV && a.wm == WMV && a.waves == 4 && a.products == NPV) {            \
    auto fn = igemm_kernel<__bf16, float, MBV, NBV, WMV, false, 4, 3, NPV>;                    \
    hipError_t err =                                                                           \
        ensure_dynamic_lds<igemm_kernel<__bf16, float, MBV, NBV, WMV, false, 4, 3, NPV>>(lds); \
    if (err != hipSuccess) return err;                                                         \
    hipLaunchKernelGGL(fn, grid, dim3(256), lds, s, a);                                        \
    return hipGetLastError();                                                                  \
  }
#define CONVND_IGEMM_CASE(MBV, NBV, WMV) CONVND_IGEMM_CASE_NP(MBV, NBV, WMV, 6)
#define CONVND_IGEMM_CASE_X8(MBV, NBV, WMV) CONVND_IGEMM_CASE_NP(MBV, NBV, WMV, 8)
  CONVND_IGEMM_TILES_P3(CONVND_IGEMM_CASE)
  CONVND_IGEMM_TILES_P3X8(CONVND_IGEMM_CASE_X8)
#undef CONVND_IGEMM_CASE_X8
#undef CONVND_IGEMM_CASE
#undef CONVND_IGEMM_CASE_NP
  return hipErrorInvalidValue;
}

template <typename T, typename O, bool DS>
hipError_t igemm_dispatch(int mb, int nb, const IgemmArgs& a, size_t lds, hipStream_t s) {
  const dim3 grid(a.boxes, a.groups * a.mgroups, a.batch * (a.nphase / a.plen));
#define CONVND_IGEMM_CASE(MBV, NBV, WMV)                                                 \
  if (mb == MBV && nb == NBV && a.wm == WMV && a.waves == 4) {                           \
    auto fn = igemm_kernel<T, O, MBV, NBV, WMV, DS, 4>;                                  \
    hipError_t err = ensure_dynamic_lds<igemm_kernel<T, O, MBV, NBV, WMV, DS, 4>>(lds);  \
    if (err != hipSuccess) return err;                                                   \
    hipLaunchKernelGGL(fn, grid, dim3(256), lds, s, a);                                  \
    return hipGetLastError();                                                            \
  }
  CONVND_IGEMM_TILES(CONVND_IGEMM_CASE)
#undef CONVND_IGEMM_CASE
  if constexpr (DS) {
#define CONVND_IGEMM_CASE8(MBV, NBV, WMV)                                                \
  if (mb == MBV && nb == NBV && a.wm == WMV && a.waves == 8) {                           \
    auto fn = igemm_kernel<T, O, MBV, NBV, WMV, DS, 8>;                                  \
    hipError_t err = ensure_dynamic_lds<igemm_kernel<T, O, MBV, NBV, WMV, DS, 8>>(lds);  \
    if (err != hipSuccess) return err;                                                   \
    hipLaunchKernelGGL(fn, grid, dim3(512), lds, s, a);                                  \
    return hipGetLastError();                                                            \
  }
    CONVND_IGEMM_TILES8(CONVND_IGEMM_CASE8)
#undef CONVND_IGEMM_CASE8
  }
  return hipErrorInvalidValue;
}

}  // namespace

bool igemm_tile_supported(int mb, int nb, int wm, int waves, int parts, int products) {
#define CONVND_IGEMM_HAS(MBV, NBV, WMV) \
  if (mb == MBV && nb == NBV && wm == WMV) return true;
  if (parts == 3) {
    if (waves == 4 && products == 8) {
      CONVND_IGEMM_TILES_P3X8(CONVND_IGEMM_HAS)
    } else if (waves == 4) {
      CONVND_IGEMM_TILES_P3(CONVND_IGEMM_HAS)
    }
    return false;
  }
  if (waves == 4) {
    CONVND_IGEMM_TILES(CONVND_IGEMM_HAS)
  } else if (waves == 8) {
    CONVND_IGEMM_TILES8(CONVND_IGEMM_HAS)
  }
#undef CONVND_IGEMM_HAS
  return false;
}

hipError_t launch_igemm(convnd_hip_dtype dtype, int mb, int nb, const IgemmArgs& a,
                        size_t lds_bytes, hipStream_t stream) {
  if (a.boxes == 0 || a.batch == 0) return hipSuccess;
  if (dtype == CONVND_HIP_BFLOAT16)
    return a.direct ? igemm_dispatch<__bf16, __bf16, true>(mb, nb, a, lds_bytes, stream)
                    : igemm_dispatch<__bf16, __bf16, false>(mb, nb, a, lds_bytes, stream);
  if (dtype == CONVND_HIP_FLOAT16)
    return a.direct ? igemm_dispatch<_Float16, _Float16, true>(mb, nb, a, lds_bytes, stream)
                    : igemm_dispatch<_Float16, _Float16, false>(mb, nb, a, lds_bytes, stream);
  if (dtype == CONVND_HIP_FLOAT32 && a.split_c > 0 && !a.direct && a.parts == 3)
    return igemm_dispatch_p3(mb, nb, a, lds_bytes, stream);
  if (dtype == CONVND_HIP_FLOAT32 && a.split_c > 0 && !a.direct)
    return igemm_dispatch<__bf16, float, false>(mb, nb, a, lds_bytes, stream);
  return hipErrorInvalidValue;
}

}  // namespace convnd
