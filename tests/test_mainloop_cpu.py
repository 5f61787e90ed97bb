"""The order of the folding W8A8 main loop (csrc/kernels/w8a8_v6.h), run on the
CPU: the header is compiled for the host with the device builtins replaced by
recorders, and the events of one wave (loads of a stage, waits, block barriers,
reads of a row or block scale) are checked against what makes them safe:

* stage kt is visible after block barrier kt + 1 (the first barrier publishes
  stage 0), and at that barrier at most the NS - 2 stages after it are
  outstanding, so a scale of k-tile kt may be read from then on;
* a scale slot of k-tile kt is reused by stage kt + NS + 1, whose loads must
  not be issued before the block barrier that follows the last read.

For every wave tile the kernels use and every number of live fragment rows.
"""
import os
import subprocess

import pytest

from lunaflux_amd import build as native_build

CLANG = "/opt/rocm/llvm/bin/clang++"
HEADER = os.path.join(native_build.CSRC, "kernels", "w8a8_v6.h")

pytestmark = pytest.mark.skipif(not os.path.exists(CLANG), reason="needs the ROCm clang")

STUB = r"""
#pragma once
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <type_traits>
#include <utility>
#define LF_DEVICE inline
struct uint4 { uint32_t x, y, z, w; };
typedef float f32x4 __attribute__((vector_size(16)));
typedef int i32x8 __attribute__((vector_size(32)));
struct Dim { unsigned x; };
static Dim threadIdx{0};
constexpr int kTileBytes = 2048;
struct Model { int barriers = 0, issued = 0, outstanding = 0, last_read[4096] = {}, rows = 0, blocks = 0; };
static Model model;
static int g_ns, g_ins, g_kt;
static void fail(const char *what, int kt, int i) {
  std::printf("FAIL %s k-tile %d row %d barriers %d\n", what, kt, i, model.barriers);
  std::exit(1);
}
static void barrier() { ++model.barriers; }
static void __syncthreads() { barrier(); }
#define __builtin_amdgcn_readfirstlane(v) (v)
#define __builtin_amdgcn_sched_barrier(v)
#define __builtin_amdgcn_s_waitcnt(v)
#define __builtin_amdgcn_s_barrier() barrier()
#define __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(...) (f32x4{})
namespace w8a8 { union Frag8 { uint4 h[2]; i32x8 v; }; }
template <class F, int... I>
inline void static_for_impl(F &&f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, class F>
inline void static_for(F &&f) { static_for_impl(f, std::make_integer_sequence<int, N>{}); }
inline float sload(const float *p, int i) { return p[i]; }
namespace w8a8v3 {
inline uint32_t lds_offset_of(const uint8_t *) { return 0; }
inline int a_chunk_offset(int row, int chunk) { return row * 128 + chunk * 16; }
inline void dma16(const uint8_t *, uint32_t, uint32_t) { ++model.outstanding; }
inline void dma4(const uint8_t *, uint32_t, uint32_t) {}
inline const uint8_t *uniform_ptr(const uint8_t *p) { return p; }
// all but the N most recent loads have landed
template <int N>
inline void wait_vmcnt() {
  if (model.outstanding > N) model.outstanding = N;
  // the barrier after this wait publishes stage model.barriers: every load of
  // it must have landed, so at most those of the stages issued after it remain
  const int later = (model.issued - 1 - model.barriers) * g_ins;
  if (model.outstanding > later) fail("stage published before its loads landed", model.barriers, 0);
}
}  // namespace w8a8v3
"""

PROBE = r"""
#include "w8a8_v6.h"
template <int NS, bool FOLD, int PARTS>
struct Scales {
  static constexpr bool kFold = FOLD;
  static constexpr int kIns = FOLD ? 1 : 0, kParts = PARTS;
  void issue(int kt) const {
    if (kt != model.issued) fail("stages issued out of order", kt, 0);
    ++model.issued;
    model.outstanding += kIns;
    // the slot of k-tile kt - (NS + 1): its last read is behind a barrier
    const int old = kt - (NS + 1);
    if (FOLD && old >= 0 && model.last_read[old] >= model.barriers) fail("slot refilled under a read", old, 0);
  }
  void seen(int kt, int i) const {
    if (kt < 0 || kt >= g_kt) fail("no such k-tile", kt, i);
    if (model.barriers < kt + 1) fail("scale read before its stage is visible", kt, i);
    model.last_read[kt] = model.barriers;
  }
  float row(int kt, int i) const { ++model.rows; seen(kt, i); return 1.0f; }
  float block(int kt, int) const { ++model.blocks; seen(kt, -1); return 1.0f; }
};
template <int BM, int BN, int WGM, int WGN, int NS, bool FOLD, int PARTS, int LIVE>
void check(uint8_t *smem, const uint8_t *src) {
  using T = w8a8v6::Tile<BM, BN, WGM, WGN, NS>;
  using S = Scales<NS, FOLD, PARTS>;
  w8a8v6::Plan<T> plan{};
  plan.a_base = src;
  for (int q = 0; q < T::kBIns; ++q) plan.b_base[q] = src;
  for (int kt : {1, 2, 3, 4, 5, 9}) {
    model = Model{};
    g_ns = NS; g_kt = kt; g_ins = T::kAIns + T::kBIns + S::kIns;
    f32x4 acc[T::kFM][T::kFN];
    w8a8v6::mainloop<T, S, LIVE>(plan, kt, smem, acc, S{});
    if (model.issued != kt) fail("stages issued", model.issued, kt);
    if (FOLD && LIVE > 0 && model.rows != kt * LIVE) fail("row scales read", model.rows, kt * LIVE);
    if (FOLD && model.blocks != kt * PARTS) fail("block scales read", model.blocks, kt * PARTS);
  }
  std::printf("ok %dx%d ns%d fold%d parts%d live%d\n", BM, BN, NS, FOLD, PARTS, LIVE);
}
int main() {
  uint8_t *smem = static_cast<uint8_t *>(std::aligned_alloc(1024, 1 << 20));
  for (int i = 0; i < 1 << 20; ++i) smem[i] = 0;
  CHECKS
  return 0;
}
"""

# (BM, BN, WGM, WGN, NS): 256 x 256 and 256 x 128 dense, 128 x 256 split and grouped
TILES = [(256, 256, 2, 4, 2), (256, 128, 4, 2, 3), (128, 256, 2, 4, 3)]


@pytest.mark.parametrize("fold", [True, False])
@pytest.mark.parametrize("tile", TILES)
def test_mainloop_order(tmp_path, tile, fold):
    (tmp_path / "w8a8_v3.h").write_text(STUB)
    with open(HEADER) as f:
        (tmp_path / "w8a8_v6.h").write_text(f.read())
    frag_rows = tile[0] // tile[2] // 16
    args = ", ".join(map(str, tile))
    checks = "\n".join(f"  check<{args}, {str(fold).lower()}, {parts}, {live}>(smem, smem);"
                       for parts in ((1, 2) if fold else (1,)) for live in range(frag_rows + 1))
    (tmp_path / "probe.cpp").write_text(PROBE.replace("CHECKS", checks))
    exe = str(tmp_path / "probe")
    subprocess.run([CLANG, "-std=c++17", "-O1", "-w", str(tmp_path / "probe.cpp"), "-o", exe], check=True)
    done = subprocess.run([exe], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout
