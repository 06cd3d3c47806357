// launch_rules.hpp — how the host sizes launches whose work it can split in several ways.
//
// Host-only (no HIP): pure functions of counts and forms.
#pragma once
#include <stdint.h>

#include <algorithm>

#include "../../include/vgi.h"

namespace vgi {

// Wavefronts that share a 64-pixel block's cones (k_trace), for a launch of `blocks` such
// blocks. With few blocks a third wavefront shortens the launch, until the specular cone
// alone sets its length (room, 9 + 1 cones, FP16 x-pair: 96 x 54 pixels 104 us with one, 60
// with two, 47 with three, 48 with five; 640 x 360 147 / 125 / 116; 1280 x 720 359 / 344 /
// 345). With many, two suffice and the third only costs its setup (4 + 1 cones at 1080p,
// FP32: 481 us with two, 530 with three). But a block's results take 1 KB of LDS per
// diffuse cone, and seven wavefronts a SIMD must fit beside them: two a block up to 10
// cones, four beyond (16 + 1 cones at 1080p, FP32: 1.71 ms with two, 1.37 with three, 1.29
// with four). Sorted pixels take four too: their footprints are scattered, and the fewer
// blocks a CU holds the more of them its L1 keeps (a frame of 16 scenes in Morton order,
// FP16: 3.69 ms with two, 3.63 with three, 3.54 with four; 3.61 with a wavefront each).
//
// From kOneTraceBlocks up to ten diffuse cones a wavefront takes a block alone again
// (k_trace_one), but for FP32. There sharing is worth little to a camera's G-buffer and costs
// scattered pixels in tile order (room and soup, 1636 x 1504, 4 + 1 cones, one / two
// wavefronts: BF16 618 / 628 us and 4.62 / 4.93 ms, FP16 601 / 599 and 4.60 / 4.77, x-pair
// 500 / 509 and 4.82 / 5.14; room, 1920 x 1080, 9 + 1: 910 / 905, 891 / 874, 726 / 720),
// while at 1280 x 720 it is worth 5% (BF16 454 / 433). FP32 gains more by it (whole calls, a
// room at 1080p, 9 + 1 cones, 892 / 802; 1636 x 1504, 4 + 1, 606 / 561), and loses up to 6% on
// scattered pixels (soup, 256^3, 1636 x 1504, 4 + 1 cones, 2000 triangles 7.05 / 7.45 ms, 20000
// 10.45 / 10.69; 9 + 1, 20000, 16.73 / 16.68): what kind a G-buffer is the launch does not know.
constexpr uint64_t kOneTraceBlocks = 24000;
constexpr uint64_t kManyTraceBlocks = 12000;
// From here a launch fills the chip (k_trace's registers: trace_waves).
constexpr uint64_t kFullTraceBlocks = 5000;
// Work-items of a launch: HIP refuses 2^32 and more. A block's wavefronts are lowered to stay
// below, so that what one wavefront a block could launch launches.
constexpr uint64_t kMaxLaunchItems = 0xFFFFFFFFull;
inline uint32_t trace_wavefronts(uint64_t blocks, uint32_t cones, uint32_t diffuse, bool sorted, uint32_t prec) {
  if (!sorted && prec != VGI_PREC_FP32 && diffuse <= 10 && blocks >= kOneTraceBlocks) return 1u;
  const uint32_t w = sorted || diffuse > 10 ? 4u : blocks < kManyTraceBlocks ? 3u : 2u;
  const uint64_t fit = blocks ? std::max<uint64_t>(1, kMaxLaunchItems / (64u * blocks)) : w;
  return std::max(1u, (uint32_t)std::min<uint64_t>(std::min(w, cones), fit));
}

// Up to here a launch leaves most of each CU's wavefront slots empty, its length is that of
// the specular cone's chain of samples, and a block's wavefronts march that cone together
// (k_trace SHARED): twelve of them, for FP32, whose footprints keep L1 busier, eight (room, 9
// + 1 cones: 96 x 54 pixels FP16 x-pair 44.7 us dealt, 37.2 / 31.5 / 31.3 with 8 / 12 / 16,
// FP16 47.6 / 39.4 / 32.2 / 32.3, FP32 53.9 / 51.1 / 49.4 / 48.7; 256 x 144, 576 blocks:
// 54.8 / 55.6 / 45.9 / 60.4 and FP32 89.1 / 79.7 / 81.2; 256 x 256, 1024 blocks: 58.9 /
// 65.0 / 60.4, FP32 94.9 / 94.7 / 112.5).
constexpr uint64_t kSharedTraceBlocks = 600;
inline uint32_t shared_wavefronts(uint32_t prec, uint32_t cones, uint32_t diffuse) {
  const uint32_t w = prec == VGI_PREC_FP32 ? 8u : 12u;
  return cones > diffuse ? w : std::max(1u, std::min(w, diffuse));  // (no specular cone: one each)
}

// Workgroups of k_voxelize: one a work unit as far as earlier calls of the stream tell (an
// eighth more and 64, or eight a CU without any), at most the units that the call's scratch
// holds. Never fewer than one a CU: in a call whose pairs overflow, these workgroups share the
// whole batch's triangles, whatever small scenes the stream has seen (4000 grid-wide triangles
// at 256^3 after scenes of a few units: 35.1 ms with 65 workgroups, 23.4 with 256; 20.2 since the
// pass keeps its triangle in scalar registers).
inline uint32_t voxelize_workgroups(uint64_t units_seen, uint64_t work_cap, uint64_t cus) {
  const uint64_t want = units_seen ? units_seen + units_seen / 8 + 64 : cus * 8;
  return (uint32_t)std::max<uint64_t>(cus, std::min<uint64_t>(want, work_cap));
}

}  // namespace vgi
