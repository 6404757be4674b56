// Which common-case Gauss-Newton kernel takes a pass over square subsets and the
// LDS that it asks for; the cell size of VSG radius windows.  Host arithmetic only,
// so that it can be tested without a GPU.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstddef>

namespace dice_hip {

// Per-subset constants of the BATCHED fast Gauss-Newton pass at the end of a
// wave's slot: the 6 x 6 matrix sum(phi phi^T), sum(phi), sum(F) and the pixel
// count (44 doubles), then the sums of the current pass, sum(gmf phi) and
// sum(G) (7 doubles), and one double of padding.
constexpr int kPersistFloats = 104;

// The most dynamic LDS that the kernels below are launched with.
constexpr size_t kMaxLaunchLds = 64 * 1024 - 2048;
// correlate_trans_kernel and its crew hold a column of the subset per lane.
constexpr int kTransMaxSide = 64;
// rows after which the translation walk's six row sums are back in their places
constexpr int kTransChunk = 6;

// The side of the square subsets of size S (DICe_Subset.cpp:90-92): odd, so
// that an even S means S + 1 pixels.
constexpr int square_side(int S) { return 2 * (S / 2) + 1; }

// The window of a translated square subset: side + 6 pixels at most (the taps
// and a fractional shift), side + 11 and side + 12 with the ring and the odd
// pitch; a multiple of four floats.
constexpr int trans_window_floats(int side, int cap) {
  const int w = ((side + 12) * (side + 11) + 3) & ~3;
  return w < cap ? w : cap & ~3;
}

// LDS floats of a wave of correlate_trans_kernel and of a crew: the slot (the
// window and the per-subset constants), gtab, and a crew's reference tables.
constexpr int trans_lds_floats(int S, int slot, bool crew) {
  const int side = square_side(S);
  if (crew) return slot + 4 * side * side;
  return trans_window_floats(side, slot - kPersistFloats) + kPersistFloats + 4 * kTransChunk * side;
}

enum class CommonKernel { kNone, kLean, kTrans, kCrew };

// What the choice depends on.
struct CommonPass {
  int n, S;          // subsets and their size
  bool affine;       // all six parameters, or translation only
  int slot;          // LDS floats per wave
  bool keys;         // Keys fourth-order interpolation, or bilinear
  bool uncertainty;  // the uncertainty fields are formed
  bool listed;       // a part of the subsets, from a list (rounds of neighbour initialization)
  int border;        // the sides of the image, 1 left, 2 right, 4 top and 8 bottom, at which a subset's
                     // box reaches the pixels that are dropped there
  int num_cus;
};

// The ends, 1 low and 2 high, at which centres in [x0, x1] with half width hw
// reach the 4 px along the border of an image of w pixels whose first has
// coordinate o, where warped pixels are dropped.
constexpr int reaches_border(int x0, int x1, int hw, int o, int w) {
  return ((long long)x0 - hw < (long long)o + 4 ? 1 : 0) | ((long long)x1 + hw >= (long long)o + w - 4 ? 2 : 0);
}

// Can a subset that is translated by a fraction of a pixel be finished in the
// slot?  The solve stages the side and its taps (5 px more, bilinear 1), the
// uncertainty fields the Keys taps (5), in the translation kernels with the
// margin that the general kernel's test has (7).  Where they do not fit, every
// subset would be set up there only to be handed over: 14,910 subsets of 43 x 43
// (default parameters) 2.71 ms with that launch, 2.34 ms without.
inline bool common_window_fits(const CommonPass &p) {
  const int taps = p.keys ? 5 : 1, unc = p.affine ? 5 : 7;
  const long long w = square_side(p.S) + (p.uncertainty && unc > taps ? unc : taps);
  return w * w <= p.slot - kPersistFloats;
}

// The most subsets that a crew of four waves each is taken for.  A CU holds three
// crews at a time, and the lean kernel, with four waves per SIMD, takes a
// wave's latency for all that fit: 768 six-parameter subsets of 21 x 21, 31 x 31
// and 43 x 43 take 71, 78 and 111 us there and 65, 69 and 86 us in crews, 1,024
// of them 71, 80 and 114 us against 84, 94 and 118 us.  Small subsets give a crew
// little to share: 9 x 9 px, 256 subsets 102 against 94 us, 384 104 against 108 us;
// 11 x 11 px, 300 subsets 109 against 101 us, 768 110 against 109 us.
// With translation only the kernel for many subsets has the longer wave: crews
// win up to 1,024 at 9 to 41 px.  A list holds few of its subsets.
inline int crew_max_subsets(const CommonPass &p) {
  if (!p.affine || p.listed) return 4 * p.num_cus;
  return (square_side(p.S) >= 11 ? 3 : 1) * p.num_cus;
}

// Translation only, subsets at the border: they lose pixels, need many steps and
// go to the general kernel, whose launch then takes at least a subset's time
// after the translation kernel's, while the general kernel alone works on them
// beside the others.  That is the faster way up to about 20 subsets per CU with
// Keys and 40 with bilinear interpolation: a full grid of 35 x 35 px (8 bits), 961
// subsets 175 against 232 us, 3,969 271 against 308, 5,929 361 against 340;
// bilinear 3,969 221 against 300, 10,000 604 against 669, 12,100 488 against 468.
// A round of neighbour initialization has a few subsets, and what counts is whether
// nearly every round has one at the border, as where both ends of the columns that
// the chain runs along do (361 points of 27 x 27 px, general kernel and crews: no
// border 3.96 and 2.29 ms; left 4.38 and 3.67; left and right 4.45 and 3.83; top
// and bottom 5.28 and 6.22; all four 5.35 and 6.32; three sides without the bottom
// 5.06 and 4.81, 21 x 21 px 3.26 and 3.57, 35 x 35 px 3.65 and 3.73).
inline bool general_for_border(const CommonPass &p) {
  if (!p.border || p.affine) return false;
  const bool x = (p.border & 3) == 3, y = (p.border & 12) == 12;
  if (p.listed) return y || (x && (p.border & 12) != 0);
  return p.n <= (p.keys ? 20 : 40) * p.num_cus;
}

// All six parameters: the lean kernel; translation only: its own kernel; few
// subsets of either kind: four waves each.  (The lean kernel also where a plain
// translation does not fit: subsets that shrink may.)
inline CommonKernel common_kernel(const CommonPass &p) {
  if (general_for_border(p)) return CommonKernel::kNone;
  const bool window = common_window_fits(p);
  auto fits = [&](bool crew) {
    return window && square_side(p.S) <= kTransMaxSide &&
           trans_lds_floats(p.S, p.slot, crew) * sizeof(float) <= kMaxLaunchLds;
  };
  if (p.n <= crew_max_subsets(p) && fits(true)) return CommonKernel::kCrew;
  if (p.affine) return CommonKernel::kLean;
  return fits(false) ? CommonKernel::kTrans : CommonKernel::kNone;
}

// The cell side of VSG radius windows: at least r / kVsgRings, so that every
// neighbour lies in the kVsgRings rings of cells around a subset (slack: what the
// rounding of the float centres and distances may add), and of about one subset
// on average, but no more than the radius.  Where subsets are dense in a part of
// their bounds only, the average says little: 400 at a step of 5 px in a square of
// 100 px and 4 far away, window 41, 192 us per call without that limit, 82 with it.
constexpr int kVsgRings = 4;
inline double vsg_radius_cell(double radius, double slack, double area, int n) {
  return std::max((radius + 4.0 * slack) / kVsgRings, std::min(radius, std::sqrt(area / n)));
}

}  // namespace dice_hip
