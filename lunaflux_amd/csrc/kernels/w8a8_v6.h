// w8a8_v6.h - e4m3 x e4m3 MFMA main loop whose scales change with every
// 128-deep k-tile (128 x 128 block-scaled weights, activations scaled per
// token and 128-column group).
//
// One v_mfma_scale_f32_16x16x128_f8f6f4 (unit scales) covers a whole k-tile
// of a 16 x 16 fragment, so its products leave the matrix pipe once per
// k-tile, into four fresh registers, and are folded into the sums with one
// v_fma each: acc += part * (sa[row][kt] * sw[block][kt]). Nothing on the
// accumulators' path waits for the vector unit (a loop that multiplies the
// accumulators themselves by the ratio of successive scales between MFMAs
// does), and no table or carried scale is needed: a zero scale gives zero.
// The factor sa * sw is one fp32 product, so it loses bits where it is below
// 2^-126 (rows of 1e-35 under block scales of 1e-6: relative error 6e-3 of bf16
// outputs; 2e-3 from 1e-34 on), and the sums are plain fp32 sums, so a partial
// sum past the fp32 range stays infinite.
// The fold is 64 v_fma against 16 MFMAs (512 matrix cycles) per wave and
// k-tile; two waves per SIMD overlap the two pipes.
//
// Block: 8 waves, each a 128 x 64 or 64 x 64 wave tile; NS stages of BM x 128 activation
// bytes and BN / 16 packed weight tiles, filled by global_load_lds (the
// layout, swizzle and k order of w8a8_v3.h). The MFMAs take the weight
// fragment first, so a lane holds one activation row (lane % 16) and four
// consecutive columns per fragment: one row scale per lane and fragment row.
//
// Order inside a k-tile (kFM fragment rows of kFN MFMAs): kRing activation
// fragments and the kFN weight fragments are in registers, each refilled
// from LDS right after its last use; each MFMA is preceded by the fold of the
// product register it overwrites (the row before's). Once the last
// fragments of this k-tile have been requested, a row's MFMAs run, then the
// wave waits for its loads of the next stage and joins the block barrier:
// every wave has its current fragments in registers, so the current stage's
// slot is free, and the matrix pipe is busy meanwhile. The rows after that
// read the next k-tile and issue the loads of stage kt + NS, spread over
// them.
#pragma once

#include "w8a8_v3.h"

namespace w8a8v6 {

template <int BM, int BN, int WGM, int WGN, int NS>
struct Tile {
  static constexpr int kBM = BM, kBN = BN, kStages = NS;
  static constexpr int kWgm = WGM, kWgn = WGN;
  static constexpr int kWaves = WGM * WGN, kThreads = 64 * kWaves;
  static constexpr int kWaveM = BM / WGM, kWaveN = BN / WGN;
  static constexpr int kFM = kWaveM / 16, kFN = kWaveN / 16;
  static constexpr int kABytes = BM * 128, kBBytes = BN * 128;
  static constexpr int kStage = kABytes + kBBytes;
  static constexpr int kSmem = NS * kStage;
  // activation fragments held in registers; slots of the scale window (the
  // scales of k-tile kt are read after stage kt + NS is issued)
  static constexpr int kRing = kFM < 4 ? kFM : 4, kScaleSlots = NS + 1;
  static constexpr int kAIns = BM / (8 * kWaves), kBIns = BN / (8 * kWaves);
  static_assert(kAIns * 8 * kWaves == BM && kBIns * 8 * kWaves == BN, "load split");
  static_assert(kFM >= 2 && kFN % 2 == 0 && kWaveN <= 128, "wave tile");
  static_assert(NS >= 2, "ring");
};

template <class T>
struct Plan {
  // Loads as wave-uniform bases and 32-bit lane offsets: activation
  // instruction q of k-tile kt reads a_base + a_off[q] + 128 kt, weight
  // instruction q b_base[q] + 2048 kt + b_lane.
  const uint8_t *a_base;
  uint32_t a_off[T::kAIns];
  const uint8_t *b_base[T::kBIns];
  uint32_t b_lane;
};

// SCALES (the block's scales):
//   kFold: false where the scales do not change with k (per-channel weights,
//     per-token activations): the MFMAs then accumulate into acc, and the
//     rest of SCALES is not used
//   kIns: side loads per wave and stage; issue(kt): issues stage kt's
//   row(kt, i): the scale of this lane's row of fragment row i (an LDS read)
//   block(kt, p): the weight scale of part p (wave-uniform); p = 1: the up
//     fragments of a gate/up block (kParts == 2: j >= kFN / 2)
// The scales of k-tile kt are read after the barrier that publishes its stage
// (scales an issue() loads land with it) and until its last fragment row, when
// stage kt + NS may already be landing.
// LIVE: the wave's fragment rows that hold a live row (the others' sums stay
// zero and are never stored); its loads and barriers are those of every wave.
template <class T, class SCALES, int LIVE = T::kFM>
LF_DEVICE void mainloop(const Plan<T> &plan, int KT, uint8_t *smem, f32x4 (&acc)[T::kFM][T::kFN],
                        const SCALES &scales) {
  constexpr int NS = T::kStages, FM = T::kFM, FN = T::kFN, R = T::kRing, P = SCALES::kParts;
  constexpr int kBarrierRow = FM - R;
  constexpr int kIns = T::kAIns + T::kBIns + SCALES::kIns;
  constexpr bool FOLD = SCALES::kFold;
  // the row at which the next k-tile's first row scale is read: the last live
  // row, or the barrier's (after it) where the live rows end before that
  constexpr int kNextScaleRow = LIVE - 1 > kBarrierRow ? LIVE - 1 : kBarrierRow;
  static_assert((NS - 1) * kIns < 64, "vmcnt range");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  const int wm = wave / T::kWgn, wn = wave % T::kWgn;
  const int g = lane >> 4, r = lane & 15;
  const uint32_t smem_base = __builtin_amdgcn_readfirstlane(w8a8v3::lds_offset_of(smem));

  // Part p of parts of stage kt's loads.
  auto issue = [&](int kt, int p, int parts) {
    const uint32_t a = smem_base + (kt % NS) * T::kStage;
    const uint8_t *ab = plan.a_base + static_cast<uint64_t>(kt) * 128;
#pragma unroll
    for (int q = 0; q < T::kAIns + T::kBIns; ++q) {
      if (q % parts != p) continue;
      if (q < T::kAIns) {
        w8a8v3::dma16(ab, plan.a_off[q], a + (wave * T::kAIns + q) * 1024);
      } else {
        const int qb = q - T::kAIns;
        w8a8v3::dma16(plan.b_base[qb] + static_cast<uint64_t>(kt) * kTileBytes, plan.b_lane,
                      a + T::kABytes + (wave * T::kBIns + qb) * 1024);
      }
    }
    if (p == parts - 1) scales.issue(kt);
  };
  const int a_row = wm * T::kWaveM + r;
  const int a_lo = w8a8v3::a_chunk_offset(a_row, 2 * g), a_hi = w8a8v3::a_chunk_offset(a_row, 2 * g + 1);
  const int b_at = T::kABytes + wn * FN * kTileBytes + lane * 16;
  auto read_a = [&](int kt, int i, w8a8::Frag8 &f) {
    // (16 rows further down keep the swizzle: it depends on row mod 8)
    const uint8_t *a = smem + (kt % NS) * T::kStage + i * 16 * 128;
    f.h[0] = *reinterpret_cast<const uint4 *>(a + a_lo);
    f.h[1] = *reinterpret_cast<const uint4 *>(a + a_hi);
  };
  auto read_b = [&](int kt, int j, w8a8::Frag8 &f) {
    const uint8_t *b = smem + (kt % NS) * T::kStage + b_at + j * kTileBytes;
    f.h[0] = *reinterpret_cast<const uint4 *>(b);
    f.h[1] = *reinterpret_cast<const uint4 *>(b + 1024);
  };

#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < NS - 1 && s < KT; ++s) issue(s, 0, 1);
  if (NS - 1 <= KT) {
    w8a8v3::wait_vmcnt<(NS - 2) * kIns>();
  } else {
    w8a8v3::wait_vmcnt<0>();
  }
  __syncthreads();
  if (NS - 1 < KT) issue(NS - 1, 0, 1);

  w8a8::Frag8 a[R], b[FN];
  f32x4 part[FN];      // products of the row before, not folded yet
  float f[P];          // their factors
  float sa, sw[P];     // the next row's scale, this k-tile's block scales
#pragma unroll
  for (int i = 0; i < (R < LIVE ? R : LIVE); ++i) read_a(0, i, a[i]);
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    if (LIVE > 0) read_b(0, j, b[j]);
    part[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  if constexpr (FOLD) {
    sa = scales.row(0, 0);
#pragma unroll
    for (int p = 0; p < P; ++p) {
      sw[p] = scales.block(0, p);
      f[p] = 0.0f;
    }
  }
  auto fold = [&](int i, int j) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      acc[i][j][e] = __builtin_fmaf(part[j][e], f[P == 2 && j >= FN / 2 ? 1 : 0], acc[i][j][e]);
    }
  };
  // K-tile kt. MORE: kt + NS < KT; NEXT: kt + 1 < KT. No branch inside: one
  // would let the compiler sink the MFMAs of several rows behind it, past
  // the registers.
  auto step = [&](int kt, auto more_tag, auto next_tag) {
    constexpr bool MORE = decltype(more_tag)::value, NEXT = decltype(next_tag)::value;
    float nsw[P];
    static_for<FM>([&](auto ii) {
      constexpr int i = decltype(ii)::value;
      [[maybe_unused]] const float sa_row = sa;
      if constexpr (FOLD && i < LIVE) {
        if constexpr (i + 1 < LIVE) {
          sa = scales.row(kt, i + 1);
        } else if constexpr (NEXT && i == kNextScaleRow && i > kBarrierRow) {
          sa = scales.row(kt + 1, 0);
        }
      }
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        if constexpr (FOLD && i < LIVE) {
          fold((i + LIVE - 1) % LIVE, j);
          part[j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(b[j].v, a[i % R].v, f32x4{0.f, 0.f, 0.f, 0.f}, 0,
                                                                     0, 0, 127, 0, 127);
        } else if constexpr (i < LIVE) {
          acc[i][j] =
              __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(b[j].v, a[i % R].v, acc[i][j], 0, 0, 0, 127, 0, 127);
        }
        if constexpr (LIVE > 0 && NEXT && i == FM - 1) read_b(kt + 1, j, b[j]);
      }
      if constexpr (FOLD && i < LIVE) {
#pragma unroll
        for (int p = 0; p < P; ++p) f[p] = sa_row * sw[p];
      }
      if constexpr (NEXT && i == kBarrierRow) {
        __builtin_amdgcn_sched_barrier(0);
        // stage kt + 1 visible (at most the NS - 2 stages after it are
        // outstanding); this wave's reads of stage kt are done, so its slot
        // may be refilled
        if constexpr (MORE) {
          w8a8v3::wait_vmcnt<(NS - 2) * kIns>();
        } else {
          w8a8v3::wait_vmcnt<0>();
        }
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (FOLD) {
          if constexpr (LIVE > 0 && i == kNextScaleRow) sa = scales.row(kt + 1, 0);
#pragma unroll
          for (int p = 0; p < P; ++p) nsw[p] = scales.block(kt + 1, p);
        }
      }
      if constexpr (MORE && i > kBarrierRow) issue(kt + NS, i - kBarrierRow - 1, R - 1);
      if constexpr (i < kBarrierRow) {
        if constexpr (i + R < LIVE) read_a(kt, i + R, a[i % R]);
      } else if constexpr (NEXT && i - kBarrierRow < LIVE) {
        read_a(kt + 1, i - kBarrierRow, a[i % R]);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (FOLD && NEXT) {
#pragma unroll
      for (int p = 0; p < P; ++p) sw[p] = nsw[p];
    }
  };
  int kt = 0;
  for (; kt + NS < KT; ++kt) step(kt, std::true_type{}, std::true_type{});
  for (; kt + 1 < KT; ++kt) step(kt, std::false_type{}, std::true_type{});
  step(kt, std::false_type{}, std::false_type{});
  if constexpr (FOLD && LIVE > 0) {
#pragma unroll
    for (int j = 0; j < FN; ++j) fold(LIVE - 1, j);
  }
}

// The main loop of a wave with live_fm live fragment rows (wave-uniform).
template <class T, class SCALES>
LF_DEVICE void mainloop_live(const Plan<T> &plan, int KT, uint8_t *smem, f32x4 (&acc)[T::kFM][T::kFN],
                             const SCALES &scales, int live_fm) {
  const int live = __builtin_amdgcn_readfirstlane(live_fm);
  if (live <= 0) {
    mainloop<T, SCALES, 0>(plan, KT, smem, acc, scales);
  } else if (live == 1) {
    mainloop<T, SCALES, 1>(plan, KT, smem, acc, scales);
  } else if (live == 2) {
    mainloop<T, SCALES, 2>(plan, KT, smem, acc, scales);
  } else {
    mainloop<T, SCALES>(plan, KT, smem, acc, scales);
  }
}

// Scales that do not change with k.
struct NoScales {
  static constexpr bool kFold = false;
  static constexpr int kIns = 0, kParts = 1;
  LF_DEVICE void issue(int) const {}
  LF_DEVICE float row(int, int) const { return 1.0f; }
  LF_DEVICE float block(int, int) const { return 1.0f; }
};

// Row scales of a dense tile, k-tile-major in memory ([K / 128][cap], the
// tile's at base): each stage side-loads its k-tile's BM scales into a slot
// of an LDS window. Wave w loads rows 64 (w mod BM / 64) .. + 63, one dword
// per lane (waves with equal w mod BM / 64 write the same bytes, so every
// wave has the same loads to count). The block scales are scalar loads.
template <class T, int PARTS>
struct DenseScales {
  static constexpr bool kFold = true;
  static constexpr int kIns = 1, kParts = PARTS;
  const uint8_t *base;     // scales_t + m0 (wave-uniform)
  uint64_t stride;         // bytes per k-tile
  uint32_t win_offset;     // LDS offset of the window [kScaleSlots][BM]
  const float *win;        // the window
  const float *sw[PARTS];  // this wave's block scales [KT] (wave-uniform)
  int row0;                // this lane's row of fragment 0
  LF_DEVICE void issue(int kt) const {
    const int lane = threadIdx.x & 63;
    const int part = (static_cast<int>(threadIdx.x) >> 6) & (T::kBM / 64 - 1);
    w8a8v3::dma4(w8a8v3::uniform_ptr(base + static_cast<uint64_t>(kt) * stride),
                 static_cast<uint32_t>(64 * part + lane) * 4,
                 win_offset + static_cast<uint32_t>(kt % T::kScaleSlots * T::kBM + 64 * part) * 4);
  }
  LF_DEVICE float row(int kt, int i) const {
    typedef const __attribute__((address_space(3))) float *lds_ptr;
    return ((lds_ptr)win)[kt % T::kScaleSlots * T::kBM + row0 + 16 * i];
  }
  LF_DEVICE float block(int kt, int p) const { return sload(sw[p], kt); }
};

}  // namespace w8a8v6
