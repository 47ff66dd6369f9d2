// BC7 (BPTC) block encoder for gfx950.
//
// Reproduces FasTC's scalar BC7 search (BPTCEncoder/src/Compressor.cpp,
// RGBAEndpoints.{h,cpp}) bit for bit at quality 0, and its simulated
// annealing (Compressor.cpp:538-630) with a counter-based random stream at
// quality > 0.
//
// The search runs as a pipeline of kernels, each shaped so that the lanes of
// a wavefront execute the same code:
//   select  one wave per four blocks: classify (solid / transparent / search)
//           and run BoxSelection (Compressor.cpp:1670-1750) with lane i scoring
//           two- and three-subset shape i; a wave argmin with lowest-index ties
//           picks the shapes.  Each block's candidates (one per mode and shape
//           entry of CompressClusters, :1752-1817, with the rotation modes split
//           per rotation and index mode) are appended to per-mode queues.
//   setup   persistent, one lane per subset of a candidate, queue by queue, so a
//           wave runs one mode: principal axis, k-means, least squares and grid
//           clamp (CompressCluster, :921-1094), and the alpha fit of the rotation
//           modes (:632-919).  Small jobs run every mode in one launch.
//   anneal  each step advances every still-annealing subset of a candidate and
//           scores all 16 pixels in one pass, each against its subset's endpoints.
//           Large lists run one lane per candidate, lanes that finish refilling
//           from the work list, and hand the last few candidates of each wave
//           over; those, and short lists from the start (spread_list), run one
//           lane per pixel, 16 lanes a candidate, where few candidates are left
//           looking several steps ahead.
//   pack    one lane per block: sum the subset errors per mode in the
//           reference's mode order, keep the first strict minimum and write the
//           128-bit block (CompressionMode::Pack, :1096-1298); solid blocks get
//           the watermark entry from an exclusive scan of solid-block flags.
//
// Under the uniform error metric all errors are exact integers (< 2^24), so
// they are kept in uint32 and equal the reference's float/double sums; the
// nonuniform metric's floats are described above qerr_nu.
#include <float.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "../../include/fasthip.h"
#include "bc7_block_decode.h"
#include "bc7_index.h"
#include "ranker_tile.h"
#include "internal.h"

namespace fh {
namespace bc7 {

enum { PB_SHARED = 0, PB_NOTSHARED = 1, PB_NONE = 2 };

struct ModeAttr {
  int8_t part_bits, subsets, idx_bits, alpha_idx_bits, color_prec, alpha_prec, has_rot,
      has_idx_mode, pbit_type;
};

// Compressor.cpp:170-203
__constant__ ModeAttr kModes[8] = {
    {4, 3, 3, 0, 4, 0, 0, 0, PB_NOTSHARED}, {6, 2, 3, 0, 6, 0, 0, 0, PB_SHARED},
    {6, 3, 2, 0, 5, 0, 0, 0, PB_NONE},      {6, 2, 2, 0, 7, 0, 0, 0, PB_NOTSHARED},
    {0, 1, 2, 3, 5, 6, 1, 1, PB_NONE},      {0, 1, 2, 2, 7, 8, 1, 0, PB_NONE},
    {0, 1, 4, 0, 7, 7, 0, 0, PB_NOTSHARED}, {6, 2, 2, 0, 5, 5, 0, 0, PB_NOTSHARED}};

// The same attributes for compile-time specialisation of per-mode kernels.
constexpr ModeAttr kModeTab[8] = {
    {4, 3, 3, 0, 4, 0, 0, 0, PB_NOTSHARED}, {6, 2, 3, 0, 6, 0, 0, 0, PB_SHARED},
    {6, 3, 2, 0, 5, 0, 0, 0, PB_NONE},      {6, 2, 2, 0, 7, 0, 0, 0, PB_NOTSHARED},
    {0, 1, 2, 3, 5, 6, 1, 1, PB_NONE},      {0, 1, 2, 2, 7, 8, 1, 0, PB_NONE},
    {0, 1, 4, 0, 7, 7, 0, 0, PB_NOTSHARED}, {6, 2, 2, 0, 5, 5, 0, 0, PB_NOTSHARED}};

// BC7 partition tables (same values as BPTCEncoder/include/FasTC/Shapes.h:24-53).
__constant__ uint16_t kShape2[64] = {
    0xcccc, 0x8888, 0xeeee, 0xecc8, 0xc880, 0xfeec, 0xfec8, 0xec80, 0xc800, 0xffec, 0xfe80,
    0xe800, 0xffe8, 0xff00, 0xfff0, 0xf000, 0xf710, 0x008e, 0x7100, 0x08ce, 0x008c, 0x7310,
    0x3100, 0x8cce, 0x088c, 0x3110, 0x6666, 0x366c, 0x17e8, 0x0ff0, 0x718e, 0x399c, 0xaaaa,
    0xf0f0, 0x5a5a, 0x33cc, 0x3c3c, 0x55aa, 0x9696, 0xa55a, 0x73ce, 0x13c8, 0x324c, 0x3bdc,
    0x6996, 0xc33c, 0x9966, 0x0660, 0x0272, 0x04e4, 0x4e40, 0x2720, 0xc936, 0x936c, 0x39c6,
    0x639c, 0x9336, 0x9cc6, 0x817e, 0xe718, 0xccf0, 0x0fcc, 0x7744, 0xee22};
__constant__ uint16_t kShape3[64][2] = {
    {0xfecc, 0xf600}, {0xffc8, 0x7300}, {0xff90, 0x3310}, {0xecce, 0x00ce}, {0xff00, 0xcc00},
    {0xcccc, 0xcc00}, {0xffcc, 0x00cc}, {0xffcc, 0x3300}, {0xff00, 0xf000}, {0xfff0, 0xf000},
    {0xfff0, 0xff00}, {0xcccc, 0x8888}, {0xeeee, 0x8888}, {0xeeee, 0xcccc}, {0xffec, 0xec80},
    {0x739c, 0x7310}, {0xfec8, 0xc800}, {0x39ce, 0x3100}, {0xfff0, 0xccc0}, {0xfccc, 0x0ccc},
    {0xeeee, 0xee00}, {0xff88, 0x7700}, {0xeec0, 0xcc00}, {0x7730, 0x3300}, {0x0cee, 0x00cc},
    {0xffcc, 0xfc88}, {0x6ff6, 0x0660}, {0xff60, 0x6600}, {0xcbbc, 0xc88c}, {0xf966, 0xf900},
    {0xceec, 0x0cc0}, {0xff10, 0x7310}, {0xff80, 0xec80}, {0xccce, 0x08ce}, {0xeccc, 0xec80},
    {0x6666, 0x4444}, {0x0ff0, 0x0f00}, {0x6db6, 0x4924}, {0x6bd6, 0x4294}, {0xcf3c, 0x0c30},
    {0xc3fc, 0x03c0}, {0xffaa, 0xff00}, {0xff00, 0x5500}, {0xfcfc, 0xcccc}, {0xcccc, 0x0c0c},
    {0xf6f6, 0x6666}, {0xaffa, 0x0ff0}, {0xfff0, 0x5550}, {0xfaaa, 0xf000}, {0xeeee, 0x0e0e},
    {0xf8f8, 0x8888}, {0xfff0, 0x9990}, {0xeeee, 0xe00e}, {0x8ff8, 0x8888}, {0xf666, 0xf000},
    {0xff00, 0x9900}, {0xff66, 0xff00}, {0xcccc, 0xc00c}, {0xcffc, 0xcccc}, {0xf000, 0x9000},
    {0x8888, 0x0808}, {0xfefe, 0xeeee}, {0xfffa, 0xfff0}, {0x7bde, 0x7310}};
// Anchor (fix-up) pixels (BPTCEncoder/src/AnchorTables.h:22-51).
__constant__ uint8_t kAnchor2[64] = {
    15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 2,  8,  2,  2, 8,
    8,  15, 2,  8,  2,  2,  8,  8,  2,  2,  15, 15, 6,  8,  2,  8,  15, 15, 2,  8,  2, 2,
    2,  15, 15, 6,  6,  2,  6,  8,  15, 15, 2,  2,  15, 15, 15, 15, 15, 2,  2,  15};
__constant__ uint8_t kAnchor3[2][64] = {
    {3,  3, 15, 15, 8, 3,  15, 15, 8,  8,  6,  6,  6,  5,  3,  3,  3,  3,  8, 15, 3,  3,
     6,  10, 5, 8,  8, 6,  8,  5,  15, 15, 8,  15, 3,  5,  6,  10, 8,  15, 15, 3, 15, 5,
     15, 15, 15, 15, 3, 15, 5,  5,  5,  8,  5,  10, 5,  10, 8,  13, 15, 12, 3,  3},
    {15, 8,  8,  3,  15, 15, 3,  8,  15, 15, 15, 15, 15, 15, 15, 8,  15, 8,  15, 3,  15, 8,
     15, 8,  3,  15, 6,  10, 15, 15, 10, 8,  15, 3,  15, 10, 10, 8,  9,  10, 6,  15, 8,  15,
     3,  6,  6,  8,  15, 3,  15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 3,  15, 15, 8}};
// Weight of the second endpoint for 1..4-bit indices (Compressor.cpp:159-168);
// the first endpoint's weight is 64 minus it.
__constant__ uint8_t kW[4][16] = {
    {0, 31, 64},
    {0, 21, 43, 64},
    {0, 9, 18, 27, 37, 46, 55, 64},
    {0, 4, 9, 13, 17, 21, 26, 30, 34, 38, 43, 47, 51, 55, 60, 64}};
// Solid-block alpha-index watermark (Compressor.cpp:135-138).
__constant__ uint32_t kWM[9] = {0x32b92180, 0x32ba3080, 0x31103200, 0x28103c80, 0x32bb3080,
                                0x25903600, 0x3530b900, 0x3b32b180, 0x34b5b98};
__constant__ uint8_t kMode5Tab[256][2];
// CompressClusters' mode order (Compressor.cpp:1757).
__constant__ int kOrder[8] = {0, 2, 1, 3, 7, 4, 5, 6};
__constant__ uint8_t kDxt6Tab[256][2][3];
// 1 / n in double for the k-means means (index n = 1..16)
__constant__ double kInvCount[17] = {0.0,        1.0,        1.0 / 2,  1.0 / 3,  1.0 / 4,
                                     1.0 / 5,    1.0 / 6,    1.0 / 7,  1.0 / 8,  1.0 / 9,
                                     1.0 / 10,   1.0 / 11,   1.0 / 12, 1.0 / 13, 1.0 / 14,
                                     1.0 / 15,   1.0 / 16};

__device__ __forceinline__ uint32_t chan(uint32_t p, int k) { return (p >> (8 * k)) & 0xFFu; }

__device__ __forceinline__ uint32_t subset_mask(int shape, int ns, int s) {
  if (ns == 2) {
    const uint32_t m = kShape2[shape];
    return s ? m : (~m & 0xFFFFu);
  }
  if (ns == 3) {
    const uint32_t m0 = kShape3[shape][0], m1 = kShape3[shape][1];
    if (s == 0) return ~m0 & 0xFFFFu;
    if (s == 1) return m0 & ~m1 & 0xFFFFu;
    return m0 & m1;
  }
  return 0xFFFFu;
}

__device__ __forceinline__ int anchor_of(int s, int shape, int ns) {
  if (s == 1) return ns == 2 ? kAnchor2[shape] : kAnchor3[0][shape];
  if (s == 2) return kAnchor3[1][shape];
  return 0;
}

// Point seen by the RGB fit.  ptmode 0: the pixel.  ptmode 1..4: rotation
// r = ptmode-1 of the alpha variant: channel r-1 swapped with A, then A = 255
// (Compressor.cpp:668-692).
__device__ __forceinline__ uint32_t point_of(uint32_t pix, int ptmode) {
  if (ptmode == 0) return pix;
  const uint32_t r = (uint32_t)ptmode - 1;
  uint32_t p = pix | 0xFF000000u;
  if (r >= 1) {
    const uint32_t sh = 8 * (r - 1);
    p = (p & ~(0xFFu << sh)) | ((pix >> 24) << sh);
  }
  return p;
}

// QuantizeChannel (RGBAEndpoints.cpp:126-165).
__host__ __device__ __forceinline__ uint32_t quant_channel(uint32_t val, uint32_t mask, int pbit) {
  if (mask == 0xFFu) return val;
  if (mask == 0u) return 0xFFu;
  uint32_t prec = (uint32_t)__builtin_popcount(mask);
  const uint32_t step = 1u << (8 - prec);
  uint32_t lval = val & mask;
  uint32_t hval = lval + step;
  if (pbit >= 0) {
    prec++;
    lval |= (uint32_t)pbit << (8 - prec);
    hval |= (uint32_t)pbit << (8 - prec);
  }
  if (lval > val) {
    lval -= step;
    hval -= step;
  }
  lval |= lval >> prec;
  hval |= hval >> prec;
  const uint32_t l8 = lval & 0xFFu, h8 = hval & 0xFFu;
  const uint32_t dl = val > l8 ? val - l8 : l8 - val;
  const uint32_t dh = val > h8 ? val - h8 : h8 - val;
  return dl < dh ? l8 : h8;
}

// quant_channel of every byte for each channel precision (the number of
// bits of the channel's mask, which keeps the top bits: 0..8) and p-bit
// (-1, 0, 1), at [(bits * 3 + pbit + 1) * 256 + byte]; built on the host
// from quant_channel itself.
__constant__ uint8_t kQuant[9 * 3 * 256];

// quant_channel(val, the channel mask byte, pbit) for a top-aligned mask
__device__ __forceinline__ uint32_t quant_tab(uint32_t val, uint32_t mask_byte, int pbit) {
  return kQuant[(uint32_t)__builtin_popcount(mask_byte) * 768u + (uint32_t)(pbit + 1) * 256u + val];
}

// ToPixel on integer-valued endpoints (uint32(c + 0.5) is then c).
__device__ __forceinline__ uint32_t to_pixel_int(uint32_t p, uint32_t mask, int pbit) {
  uint32_t r = 0;
#pragma unroll
  for (int k = 0; k < 4; k++) r |= quant_tab(chan(p, k), chan(mask, k), pbit) << (8 * k);
  return r;
}

// uint32(c + 0.5) with the add in double (RGBAEndpoints.cpp:169-172), exactly,
// for c in [0, 255].
__device__ __forceinline__ uint32_t round_half_up(float c) {
  const float f = floorf(c);
  return (uint32_t)f + ((c - f) >= 0.5f ? 1u : 0u);
}


__device__ __forceinline__ uint32_t to_pixel_f(const float p[4], uint32_t mask, int pbit) {
  uint32_t r = 0;
#pragma unroll
  for (int k = 0; k < 4; k++)
    r |= quant_tab(round_half_up(p[k]) & 0xFFu, chan(mask, k), pbit) << (8 * k);
  return r;
}

__device__ __forceinline__ float dot4(const float a[4], const float b[4]) {
  float s = 0.0f;
#pragma unroll
  for (int k = 0; k < 4; k++) s += a[k] * b[k];
  return s;
}

// VectorBase::Length: sqrt in long double rounded to float equals the
// correctly rounded single-precision sqrt (the double rounding is innocuous
// since 64 >= 2*24+2).
__device__ __forceinline__ float len4(const float a[4]) { return sqrtf(dot4(a, a)); }

__device__ __forceinline__ void normalize4(float a[4]) {
  const float l = len4(a);
#pragma unroll
  for (int k = 0; k < 4; k++) a[k] /= l;
}

// Packed 16-bit lanes: channels 0 and 2 of a pixel are (pix & 0x00FF00FF),
// channels 1 and 3 are ((pix >> 8) & 0x00FF00FF); every quantity of the
// index search fits 16 bits (interpolation sums within +-16352, channel
// differences within +-255), so v_pk_* and v_dot2 give the exact integers.
typedef short s16x2 __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ u16x2 as_u16x2(uint32_t v) { return __builtin_bit_cast(u16x2, v); }
__device__ __forceinline__ s16x2 as_s16x2(uint32_t v) { return __builtin_bit_cast(s16x2, v); }
__device__ __forceinline__ s16x2 as_s16x2(u16x2 v) { return __builtin_bit_cast(s16x2, v); }

// A texel as the pixel pass reads it: 64 times its channel pairs (each 16-bit
// lane at most 64 * 255 = 16320).  The interpolated value of an index weight
// w is (e1 (64 - w) + e2 w + 32) >> 6 = (64 e1 + 32 + (e2 - e1) w) >> 6, so
// with the texel scaled by 64 its difference to the texel is one shift of
// one sum, and the texel's projection is 64 times the integer one.
__device__ __forceinline__ uint32_t pair02x64(uint32_t pix) { return (pix & 0x00FF00FFu) << 6; }
__device__ __forceinline__ uint32_t pair13x64(uint32_t pix) {
  return ((pix >> 8) & 0x00FF00FFu) << 6;
}

// a . b + c in the three-operand form of the instruction: asked to saturate
// (every sum here is far from the 32-bit range) the compiler cannot take the
// accumulating two-operand form, which needs its start value moved into place
// first (three moves per pixel in the pixel pass).
__device__ __forceinline__ int dot2(s16x2 a, s16x2 b, int c) {
  return __builtin_amdgcn_sdot2(a, b, c, true);
}

// Per-subset constants of one annealing step.
struct SubConst {
  uint32_t a02, a13;  // 64 * endpoint 1 + 32, channel pairs
  uint32_t d02, d13;  // endpoint 2 - endpoint 1 (signed pairs)
  uint32_t q02, q13;  // the projection axis (d, or d seen through a rotation)
  int ad;             // -64 * endpoint 1 . (endpoint 2 - endpoint 1)
  float rl;           // 1 / (64 l), l the squared endpoint distance (see pixel_bounds)
};

__device__ __forceinline__ SubConst sub_const(uint32_t e1, uint32_t e2) {
  SubConst c;
  const uint32_t a02 = e1 & 0x00FF00FFu, a13 = (e1 >> 8) & 0x00FF00FFu;
  const uint32_t b02 = e2 & 0x00FF00FFu, b13 = (e2 >> 8) & 0x00FF00FFu;
  c.d02 = __builtin_bit_cast(uint32_t, as_s16x2(b02) - as_s16x2(a02));
  c.d13 = __builtin_bit_cast(uint32_t, as_s16x2(b13) - as_s16x2(a13));
  c.q02 = c.d02;
  c.q13 = c.d13;
  // each 16-bit lane: 64 a + 32 <= 16352
  c.a02 = (a02 << 6) + 0x00200020u;
  c.a13 = (a13 << 6) + 0x00200020u;
  // endpoint 1's projection on the axis, subtracted from each pixel's
  c.ad = -64 * dot2(as_s16x2(a02), as_s16x2(c.d02), dot2(as_s16x2(a13), as_s16x2(c.d13), 0));
  const int l = dot2(as_s16x2(c.d02), as_s16x2(c.d02), dot2(as_s16x2(c.d13), as_s16x2(c.d13), 0));
  // equal endpoints give d = 0 for every pixel, so l = 1 yields index 0
  c.rl = scaled_rcp(l > 0 ? l : 1);
  return c;
}

// The projection axis of a rotation mode (ptmode = rotation + 1).  Its
// points are the texels with channel r - 1 replaced by alpha (r > 0) and
// alpha 255 (point_of), so a point's projection is the texel's on a permuted
// axis (alpha taking channel r - 1's component, that channel none) plus
// 255 times the axis' alpha component.  sel02 / sel13: v_perm_b32 selectors
// over (d02, d13), identity without a rotation.
__device__ __forceinline__ void rotation_selectors(int ptmode, uint32_t &sel02, uint32_t &sel13) {
  // bytes 0-3 of the selector index d13, 4-7 d02, 0x0c a zero byte
  sel02 = 0x07060504u;
  sel13 = 0x03020100u;
  if (ptmode == 1) sel13 = 0x0c0c0100u;
  if (ptmode == 2) {
    sel02 = 0x07060c0cu;
    sel13 = 0x05040100u;
  }
  if (ptmode == 3) sel13 = 0x01000c0cu;
  if (ptmode == 4) {
    sel02 = 0x0c0c0504u;
    sel13 = 0x07060100u;
  }
}
__device__ __forceinline__ void rotate_axis(SubConst &c, int ptmode, uint32_t sel02,
                                            uint32_t sel13) {
  c.q02 = __builtin_amdgcn_perm(c.d02, c.d13, sel02);
  c.q13 = __builtin_amdgcn_perm(c.d02, c.d13, sel13);
  const int da = (int)c.d13 >> 16;
  c.ad += ptmode ? 64 * 255 * da : 0;
}

// Difference of the pixel pairs (64 p) to the interpolant of index weight
// word ww, (64 e1 + 32 - 64 p + (e2 - e1) w) >> 6 = interpolant - p: z holds
// 64 e1 + 32 - 64 p, and the sum lies within +-16352, so signed 16-bit lanes
// hold it exactly.
__device__ __forceinline__ s16x2 interp_diff(s16x2 z, uint32_t d, uint32_t ww) {
  const s16x2 w = as_s16x2(ww);
  const s16x2 W = {w.y, w.y};
  const s16x2 S = {6, 6};
  return (as_s16x2(d) * W + z) >> S;
}

// The neighbouring indices of a pixel (index_bounds).  The pass is bound by VALU
// issue: an integer quotient corrected with the exact remainder took 17
// instructions per pixel where this takes 9; with the texels kept as scaled
// pairs (no unpacking, one subtraction per pair) and the rotation folded into
// the axis (no separate point) the pass went from about 54 instructions per
// pixel to 33, and the 4096 x 4096 annealing from 46.0 to 34.3 ms (reference
// search) and 5.2 to 4.1 ms (learned).
__device__ __forceinline__ void pixel_bounds(uint32_t p02, uint32_t p13, const SubConst &c,
                                             float kf, uint32_t &j1, uint32_t &j2) {
  const int d = dot2(as_s16x2(p02), as_s16x2(c.q02), dot2(as_s16x2(p13), as_s16x2(c.q13), c.ad));
  index_bounds(d, c.rl, kf, j1, j2);
}

// The per-pixel index search without branches: both neighbouring indices
// are scored and the second kept only when strictly better (where the two
// are the same index the errors are equal).  Returns the error, the index in
// *best.  p02, p13: the texel's pairs times 64.
__device__ __forceinline__ uint32_t pixel_err(uint32_t p02, uint32_t p13, const SubConst &c,
                                              float kf, WeightFn wf, uint32_t *best) {
  uint32_t j1, j2;
  pixel_bounds(p02, p13, c, kf, j1, j2);
  const s16x2 z02 = as_s16x2(c.a02) - as_s16x2(p02), z13 = as_s16x2(c.a13) - as_s16x2(p13);
  const uint32_t w1 = weight_word(wf, j1), w2 = weight_word(wf, j2);
  const s16x2 x02 = interp_diff(z02, c.d02, w1), x13 = interp_diff(z13, c.d13, w1);
  const s16x2 y02 = interp_diff(z02, c.d02, w2), y13 = interp_diff(z13, c.d13, w2);
  const uint32_t e1 = (uint32_t)dot2(x02, x02, dot2(x13, x13, 0));
  const uint32_t e2 = (uint32_t)dot2(y02, y02, dot2(y13, y13, 0));
  *best = e2 < e1 ? j2 : j1;
  return e2 < e1 ? e2 : e1;
}

// QuantizedError with endpoints already quantised to qp1/qp2
// (RGBAEndpoints.cpp:190-310, uniform metric) by the pixel pass above.
// Indices are written at pixel positions (4 bits each) for the pixels in
// smask.  (With the reference's float quotient and the weights from their
// table, two divisions and four dependent loads a pixel, this took about a
// tenth of a fit.)
__device__ __forceinline__ uint32_t qerr(const uint32_t px[16], uint32_t smask, int ptmode,
                                         uint32_t qp1, uint32_t qp2, int nb, uint64_t &idx) {
  uint32_t sel02, sel13;
  rotation_selectors(ptmode, sel02, sel13);
  SubConst c = sub_const(qp1, qp2);
  rotate_axis(c, ptmode, sel02, sel13);
  const WeightFn wf = weight_fn(nb);
  const float kf = (float)(nb - 1);
  idx = 0;
  uint32_t total = 0;
#pragma unroll 1
  for (int i = 0; i < 16; i++) {
    if (!((smask >> i) & 1)) continue;
    const uint32_t pix = px[i];
    uint32_t best;
    total += pixel_err(pair02x64(pix), pair13x64(pix), c, kf, wf, &best);
    idx |= (uint64_t)best << (4 * i);
  }
  return total;
}

// ---------------------------------------------------------------------------
// The nonuniform error metric (m_ErrorMetric = eErrorMetric_Nonuniform,
// BPTCCompressor.h:73-77; weights kErrorMetrics, Compressor.cpp:205-208).
// Each channel's absolute difference is multiplied by its weight before
// squaring, and the four squares are summed in float in channel order from
// zero (VectorBase::Dot, VectorBase.h:96-101).  The errors are then floats
// whose values depend on the order of the additions, so every sum below runs
// in the reference's order: channels, then the pixels of a subset in pixel
// order.  A float error is kept as its bit pattern in the 32-bit error fields
// the uniform metric fills with integers: for errors >= 0 the bit patterns
// order as the values do, so comparisons and the "> 0" tests are shared.
// ---------------------------------------------------------------------------
struct Weights {
  float w[4];
};

__device__ __forceinline__ float werr(int d0, int d1, int d2, int d3, const Weights &m) {
  const float e0 = (float)abs(d0) * m.w[0];
  const float e1 = (float)abs(d1) * m.w[1];
  const float e2 = (float)abs(d2) * m.w[2];
  const float e3 = (float)abs(d3) * m.w[3];
  return ((e0 * e0 + e1 * e1) + e2 * e2) + e3 * e3;
}

// The weights a rotation mode sees (GetErrorMetric, CompressionMode.h:196-205):
// rotation r swaps channel r-1's weight with alpha's.
__device__ __forceinline__ Weights rotate_weights(const Weights &m, int rot) {
  Weights r = m;
  if (rot >= 1 && rot <= 3) {
    r.w[rot - 1] = m.w[3];
    r.w[3] = m.w[rot - 1];
  }
  return r;
}

__device__ __forceinline__ Weights params_weights(const Bc7Params &prm) {
  Weights m;
#pragma unroll
  for (int k = 0; k < 4; k++) m.w[k] = prm.metric[k];
  return m;
}

// QuantizedError under per-channel weights m (qerr's float counterpart):
// per pixel the weighted error of each of the two neighbouring indices, the
// second kept only when strictly better, summed in float in pixel order.
template <int UNROLL>
__device__ __forceinline__ float qerr_nu(const uint32_t px[16], uint32_t smask, int ptmode,
                                         uint32_t qp1, uint32_t qp2, int nb, const Weights &m,
                                         uint64_t &idx) {
  int a[4], b[4], dir[4];
  int lsq = 0;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    a[k] = (int)chan(qp1, k);
    b[k] = (int)chan(qp2, k);
    dir[k] = b[k] - a[k];
    lsq += dir[k] * dir[k];
  }
  idx = 0;
  float total = 0.0f;
  if (lsq == 0) {
#pragma unroll
    for (int i = 0; i < 16; i++) {
      if (!((smask >> i) & 1)) continue;
      total += werr((int)chan(px[i], 0) - a[0], (int)chan(px[i], 1) - a[1],
                    (int)chan(px[i], 2) - a[2], (int)chan(px[i], 3) - a[3], m);
    }
    return total;
  }
  const int prec = nb == 4 ? 2 : (nb == 8 ? 3 : 4);
  const float flsq = (float)lsq;
  const float kf = (float)(nb - 1);
#pragma unroll UNROLL
  for (int i = 0; i < 16; i++) {
    if (!((smask >> i) & 1)) continue;
    const uint32_t pt = point_of(px[i], ptmode);
    int d = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) d += ((int)chan(pt, k) - a[k]) * dir[k];
    const float pct = (float)d / flsq;
    const float t = pct * kf;
    int j1 = (int)floorf(t);
    int j2 = (int)ceilf(t);
    j1 = j1 < 0 ? 0 : j1;
    j1 = j1 > nb - 1 ? nb - 1 : j1;
    j2 = j2 > nb - 1 ? nb - 1 : j2;
    const uint32_t pix = px[i];
    int dd[4];
    {
      const int w1 = kW[prec - 1][j1], w0 = 64 - w1;
#pragma unroll
      for (int k = 0; k < 4; k++) dd[k] = (int)chan(pix, k) - ((a[k] * w0 + b[k] * w1 + 32) >> 6);
    }
    const float e1 = werr(dd[0], dd[1], dd[2], dd[3], m);
    int best = j1;
    float me = e1;
    if (j2 > j1) {
      const int w1 = kW[prec - 1][j2], w0 = 64 - w1;
#pragma unroll
      for (int k = 0; k < 4; k++) dd[k] = (int)chan(pix, k) - ((a[k] * w0 + b[k] * w1 + 32) >> 6);
      const float e2 = werr(dd[0], dd[1], dd[2], dd[3], m);
      if (e2 < e1) {
        best = j2;
        me = e2;
      }
    }
    total += me;
    idx |= (uint64_t)best << (4 * i);
  }
  return total;
}

// Per-lane description of one subset fit.
struct Fit {
  int mode;
  int rot;        // rotation (modes 4/5), 0 otherwise
  int idx_mode;   // index mode (mode 4), 0 otherwise
  int nbits_idx;  // GetNumberOfBitsPerIndex() for this fit
  uint32_t qmask;
  int pbit_type;
  int color_prec, alpha_prec;
  int npbc;
};

__device__ __forceinline__ int pbc_bit(int pbit_type, int combo, int which) {
  // GetPBitCombo (CompressionMode.h:243-250): kPBits = {0,0},{0,1},{1,0},{1,1}
  if (pbit_type == PB_SHARED) return combo ? 1 : 0;
  if (pbit_type == PB_NOTSHARED) return which == 0 ? ((combo % 4) >> 1) : ((combo % 4) & 1);
  return 0;
}

// GetQuantizationMask (CompressionMode.h:212-232).
__device__ __forceinline__ uint32_t qmask_of(int color_prec, int alpha_prec) {
  const int32_t seed = (int32_t)0x80000000u;
  const uint32_t cbits = (uint32_t)color_prec - 1;
  uint32_t m = ((uint32_t)(seed >> (24 + cbits)) & 0xFFu) |
               ((uint32_t)(seed >> (16 + cbits)) & 0xFF00u) |
               ((uint32_t)(seed >> (8 + cbits)) & 0xFF0000u);
  if (alpha_prec > 0) m |= (uint32_t)(seed >> (alpha_prec - 1)) & 0xFF000000u;
  return m;
}

// CompressSingleColor (Compressor.cpp:252-353) through the precomputed
// per-value endpoint table.  Returns the per-pixel error; under the
// nonuniform metric (NU) its float bit pattern, weighted by the unrotated
// weights mu (Compressor.cpp:334-339) and summed in channel order.
template <bool NU = false>
__device__ __forceinline__ uint32_t single_color(const Fit &f, const uint32_t *sctab, uint32_t pixel,
                                 uint32_t &p1, uint32_t &p2, int &pbc,
                                 const Weights *mu = nullptr) {
  uint32_t best = NU ? __float_as_uint(FLT_MAX) : 0xFFFFFFFFu;
  const int bpi = f.nbits_idx - 1;
  for (int pbi = 0; pbi < f.npbc; pbi++) {
    uint32_t err = 0, q1 = 0, q2 = 0;
    float ferr = 0.0f;
#pragma unroll
    for (int ci = 0; ci < 4; ci++) {
      const uint32_t val = chan(pixel, ci);
      const int nbits = ci == 3 ? f.alpha_prec : f.color_prec;
      uint32_t lo, hi, dist;
      if (nbits == 0) {
        lo = hi = 0xFFu;
        dist = 0xFFu - val;
      } else {
        int cfg = 0;
        if (f.pbit_type != PB_NONE)
          cfg = 1 + 2 * pbc_bit(f.pbit_type, pbi, 0) + pbc_bit(f.pbit_type, pbi, 1);
        const uint32_t e = sctab[(((nbits - 4) * 5 + cfg) * 4 + bpi) * 256 + val];
        lo = e & 0xFFu;
        hi = (e >> 8) & 0xFFu;
        dist = (e >> 16) & 0xFFu;
      }
      if constexpr (NU) {
        const float e = (float)dist * mu->w[ci];
        ferr += e * e;
      } else {
        err += dist * dist;
      }
      q1 |= lo << (8 * ci);
      q2 |= hi << (8 * ci);
    }
    if constexpr (NU) err = __float_as_uint(ferr);
    if (err < best) {
      best = err;
      pbc = pbi;
      p1 = q1;
      p2 = q2;
    }
  }
  return best;
}

// MatrixSquare<float,4>::PowerMethod without the eigenvalue
// (Base/include/FasTC/MatrixSquare.h:44-105).
__device__ __forceinline__ void power_method(const float m[16], float b[4]) {
  const float norm = 1.0f / sqrtf(4.0f);
#pragma unroll
  for (int i = 0; i < 4; i++) b[i] = norm;
  bool bad = false, fixed = false;
  int iters = 0;
  while (!fixed && ++iters < 5) {
    float nb[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      nb[j] = 0.0f;
#pragma unroll
      for (int i = 0; i < 4; i++) nb[j] += m[j * 4 + i] * b[i];
    }
    const float len = len4(nb);
    if ((double)len < 1e-10) {
      if (bad) return;
      b[0] = 1.0f;
      b[1] = 1.0f;
      normalize4(b);
      bad = true;
      continue;
    }
    normalize4(nb);
    if (fabs((double)(1.0f - dot4(b, nb))) < 1e-8) fixed = true;
#pragma unroll
    for (int i = 0; i < 4; i++) b[i] = nb[i];
  }
}

__device__ __forceinline__ void unpack4f(uint32_t p, float v[4]) {
#pragma unroll
  for (int k = 0; k < 4; k++) v[k] = (float)chan(p, k);
}

// GetPrincipalAxis with no eigenvalues (RGBAEndpoints.cpp:327-428),
// including the collinearity test's reads of default (-1,-1,-1,-1) entries
// past the last unique point (:364-371).
__device__ __forceinline__ void principal_axis(const uint32_t px[16], uint32_t smask, int ptmode, int n,
                               const float avg[4], float axis[4]) {
  // the repeated points: equal to an earlier one of the subset.  Unrolled on
  // register copies: the 120 comparisons take one instruction each (rolled,
  // with two LDS reads apiece, they were a fifth of a fit's latency)
  uint32_t dup = 0;
  {
    uint32_t pt[16];
#pragma unroll
    for (int i = 0; i < 16; i++) pt[i] = point_of(px[i], ptmode);
#pragma unroll
    for (int i = 1; i < 16; i++) {
      bool seen = false;
#pragma unroll
      for (int j = 0; j < i; j++) seen = seen | (((smask >> j) & 1) && pt[j] == pt[i]);
      dup |= seen ? 1u << i : 0u;
    }
  }
  // unique points in first-occurrence order; test u2.. as they appear
  int nu = 0;
  float u0[4], dir[4];
  bool collinear = true;
  uint32_t u0p = 0;
#pragma unroll 1
  for (int i = 0; i < 16; i++) {
    if (!(((smask & ~dup) >> i) & 1)) continue;
    const uint32_t pi = point_of(px[i], ptmode);
    if (nu == 0) {
      u0p = pi;
      unpack4f(pi, u0);
    } else if (nu == 1) {
      float u1[4];
      unpack4f(pi, u1);
#pragma unroll
      for (int k = 0; k < 4; k++) dir[k] = u1[k] - u0[k];
      normalize4(dir);
    } else if (collinear) {
      float v[4];
      unpack4f(pi, v);
#pragma unroll
      for (int k = 0; k < 4; k++) v[k] -= u0[k];
      if (fabs(fabs((double)dot4(v, dir)) - (double)len4(v)) > 1e-7) collinear = false;
    }
    nu++;
  }
  (void)u0p;
  if (nu == 1) {
#pragma unroll
    for (int k = 0; k < 4; k++) axis[k] = 0.0f;
    return;
  }
  // the loop runs i = 2 .. n-1 over upts[]; entries past nu are (-1,-1,-1,-1)
  if (collinear && n > (nu > 2 ? nu : 2)) {
    float v[4];
#pragma unroll
    for (int k = 0; k < 4; k++) v[k] = -1.0f - u0[k];
    if (fabs(fabs((double)dot4(v, dir)) - (double)len4(v)) > 1e-7) collinear = false;
  }
  if (collinear) {
#pragma unroll
    for (int k = 0; k < 4; k++) axis[k] = dir[k];
    return;
  }
  // each entry sums its products in point order
  float sum[10];
#pragma unroll
  for (int e = 0; e < 10; e++) sum[e] = 0.0f;
#pragma unroll 1
  for (int p = 0; p < 16; p++) {
    if (!((smask >> p) & 1)) continue;
    const uint32_t pt = point_of(px[p], ptmode);
    float t[4];
#pragma unroll
    for (int k = 0; k < 4; k++) t[k] = (float)chan(pt, k) - avg[k];
    int e = 0;
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int j = 0; j <= i; j++) sum[e++] += t[i] * t[j];
  }
  float cov[16];
  {
    int e = 0;
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int j = 0; j <= i; j++) {
        // x / 3.0f for a float x as a double product, correctly rounded:
        // x / 3 is a float or, with 3 left in its denominator, at least
        // 2^-27 (relative) from every float rounding boundary
        cov[i * 4 + j] = (float)((double)sum[e++] * (1.0 / 3.0));
        cov[j * 4 + i] = cov[i * 4 + j];
      }
  }
  power_method(cov, axis);
}

// Counter-based annealing stream (the oracle defines the same function).
__device__ __forceinline__ uint32_t mix32(uint32_t x) {
  x ^= x >> 16;
  x *= 0x7feb352du;
  x ^= x >> 15;
  x *= 0x846ca68bu;
  x ^= x >> 16;
  return x;
}
__device__ __forceinline__ uint32_t fit_key(uint64_t seed, uint64_t block_id, uint32_t tag) {
  uint32_t k = mix32((uint32_t)seed ^ 0x2545F491u);
  k = mix32(k ^ (uint32_t)(seed >> 32));
  k = mix32(k ^ (uint32_t)block_id);
  k = mix32(k ^ (uint32_t)(block_id >> 32));
  return mix32(k ^ tag);
}

// x: key + (draws made) * 0x9E3779B9, kept as a running sum.
constexpr uint32_t kRngStep = 0x9E3779B9u;
struct Rng {
  uint32_t x;
  __device__ __forceinline__ uint32_t next() {
    const uint32_t h = mix32(x);
    x += kRngStep;
    return h;
  }
  __device__ __forceinline__ uint32_t next16() { return next() >> 16; }
  // frand (Compressor.cpp:506-519)
  __device__ __forceinline__ float frand() {
    const uint32_t r = next16();
    return __uint_as_float((127u << 23) | ((r << 8) | (r >> 7))) - 1.0f;
  }
};

// One endpoint's neighbour: every channel moved by delta = k1 - bit * k2
// (channel pairs; bit k of the draw's top half is channel k's), clamped to
// 0..255.
__device__ __forceinline__ uint32_t step_endpoint(uint32_t p, uint32_t h, s16x2 k1_02,
                                                  s16x2 k1_13, s16x2 k2_02, s16x2 k2_13) {
  const uint32_t b02 = ((h >> 16) & 1u) | ((h >> 2) & 0x10000u);
  const uint32_t b13 = ((h >> 17) & 1u) | ((h >> 3) & 0x10000u);
  const s16x2 lo = {0, 0}, hi = {255, 255};
  s16x2 n02 = as_s16x2(p & 0x00FF00FFu) + (k1_02 - as_s16x2(b02) * k2_02);
  s16x2 n13 = as_s16x2((p >> 8) & 0x00FF00FFu) + (k1_13 - as_s16x2(b13) * k2_13);
  n02 = __builtin_elementwise_min(__builtin_elementwise_max(n02, lo), hi);
  n13 = __builtin_elementwise_min(__builtin_elementwise_max(n13, lo), hi);
  return __builtin_bit_cast(uint32_t, n02) | (__builtin_bit_cast(uint32_t, n13) << 8);
}

// ---------------------------------------------------------------------------
// Per-subset fit set-up: CompressCluster up to the annealing loop.
// ---------------------------------------------------------------------------

__device__ __forceinline__ void set_fit_attr(Fit &f, const ModeAttr a, int mode, int rot,
                                             int im) {
  f.mode = mode;
  f.rot = rot;
  f.idx_mode = im;
  f.nbits_idx = im == 0 ? a.idx_bits : a.alpha_idx_bits;
  f.color_prec = a.color_prec;
  f.alpha_prec = a.alpha_prec;
  f.qmask = qmask_of(a.color_prec, a.alpha_prec);
  f.pbit_type = a.pbit_type;
  f.npbc = a.pbit_type == PB_SHARED ? 2 : (a.pbit_type == PB_NOTSHARED ? 4 : 1);
}

__device__ __forceinline__ void set_fit(Fit &f, int mode, int rot, int im) {
  set_fit_attr(f, kModes[mode], mode, rot, im);
}

// Where a subset fit stands once CompressCluster reaches
// OptimizeEndpointsForCluster (Compressor.cpp:550-580), or its final result
// when no annealing follows (single colour, quality 0, zero error).
struct SubStart {
  uint32_t err;  // QuantizedError of the start endpoints (or the final error)
  bool sc;       // CompressSingleColor's result: the subset's error is n * err
  uint32_t p1, p2;  // endpoint state (integers): annealing start, or final endpoints
  uint64_t idx;     // indices at pixel positions of this subset
  int pbc;
  bool anneal;
};

// Index of the centroid nearest to v (squared distance, first minimum).
template <int NB>
__device__ __forceinline__ int nearest_centroid(const float c[NB][4], const float v[4]) {
  int minb = -1;
  float mind = FLT_MAX;
#pragma unroll
  for (int j = 0; j < NB; j++) {
    float d[4];
#pragma unroll
    for (int k = 0; k < 4; k++) d[k] = v[k] - c[j][k];
    const float ds = dot4(d, d);
    if (ds < mind) {
      mind = ds;
      minb = j;
    }
  }
  return minb;
}

__device__ __forceinline__ void km_add(uint32_t *p, uint32_t v) {
  __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}

// NU: the nonuniform metric, mu its unrotated weights (single colour), mr
// the weights of this candidate's rotation (QuantizedError).
// km: this lane's k-means accumulators in LDS, words (j * 3 + k) * 64 of
// bucket j: the sums of channels 0 and 2 (<< 16), of 1 and 3, the count.  A sum
// is at most 16 * 255, so 16 bits hold it, and integer sums are the reference's
// float sums exactly; they are added in place without being read, where five
// float sums a point took a read and a write each.
template <int NB, bool NU = false>
__device__ __forceinline__ void kmeans_setup(const Fit &f, uint32_t q, const uint32_t *sctab,
                             const uint32_t px[16], uint32_t smask, int ptmode, int n,
                             const float avg[4], SubStart &out,
                             const Weights *mu, const Weights *mr, uint32_t *km) {
  float axis[4];
  principal_axis(px, smask, ptmode, n, avg, axis);
  float mindp = FLT_MAX, maxdp = -FLT_MAX;
#pragma unroll 1
  for (int i = 0; i < 16; i++) {
    if (!((smask >> i) & 1)) continue;
    float v[4];
    unpack4f(point_of(px[i], ptmode), v);
#pragma unroll
    for (int k = 0; k < 4; k++) v[k] -= avg[k];
    const float dp = dot4(v, axis);
    if (dp < mindp) mindp = dp;
    if (dp > maxdp) maxdp = dp;
  }
  float p1[4], p2[4];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    p1[k] = avg[k] + axis[k] * mindp;
    p2[k] = avg[k] + axis[k] * maxdp;
    // ClampEndpoints (RGBAEndpoints.cpp:436-441)
    p1[k] = p1[k] < 0.0f ? 0.0f : (p1[k] > 255.0f ? 255.0f : p1[k]);
    p2[k] = p2[k] < 0.0f ? 0.0f : (p2[k] > 255.0f ? 255.0f : p2[k]);
  }
  // Lloyd k-means from NB evenly spaced seeds (Compressor.cpp:961-1026)
  float c[NB][4];
#pragma unroll
  for (int i = 0; i < NB; i++) {
    const float s = (float)i / (float)(NB - 1);
#pragma unroll
    for (int k = 0; k < 4; k++) c[i][k] = p1[k] * (1.0f - s) + p2[k] * s;
  }
  uint32_t cnt[NB];
  bool fixed = false;
  int guard = 0;
  while (!fixed && guard++ < 4096) {
    // every point into its nearest centroid's sums (Compressor.cpp:997-1009)
#pragma unroll
    for (int j = 0; j < NB * 3; j++) km[j * 64] = 0u;
#pragma unroll 1
    for (int i = 0; i < 16; i++) {
      if (!((smask >> i) & 1)) continue;
      const uint32_t pt = point_of(px[i], ptmode);
      float v[4];
      unpack4f(pt, v);
      uint32_t *b = km + nearest_centroid<NB>(c, v) * 3 * 64;
      km_add(b, pt & 0x00FF00FFu);
      km_add(b + 64, (pt >> 8) & 0x00FF00FFu);
      km_add(b + 2 * 64, 1u);
    }
    fixed = true;
#pragma unroll
    for (int j = 0; j < NB; j++) {
      const uint32_t k02 = km[(j * 3) * 64], k13 = km[(j * 3 + 1) * 64];
      const uint32_t cn = km[(j * 3 + 2) * 64];
      float s[4];
      // sum / cn in float, correctly rounded, as a double product: the sum
      // is an integer below 2^13 and cn one of 1..16, so sum / cn is either
      // a float or, in lowest terms p / q with q odd, at least 2^-29
      // (relative) from every float rounding boundary, far beyond the
      // product's 2^-52 (kInvCount[0] is 0: an empty bucket's mean is 0)
      const double inv = kInvCount[cn];
      s[0] = (float)((double)(k02 & 0xFFFFu) * inv);
      s[1] = (float)((double)(k13 & 0xFFFFu) * inv);
      s[2] = (float)((double)(k02 >> 16) * inv);
      s[3] = (float)((double)(k13 >> 16) * inv);
      if (s[0] != c[j][0] || s[1] != c[j][1] || s[2] != c[j][2] || s[3] != c[j][3])
        fixed = false;
#pragma unroll
      for (int k = 0; k < 4; k++) c[j][k] = s[k];
      cnt[j] = cn;
    }
  }
  int nfilled = 0, last = 0;
#pragma unroll
  for (int j = 0; j < NB; j++)
    if (cnt[j] > 0) {
      nfilled++;
      last = j;
    }
  uint64_t ones = 0;
#pragma unroll
  for (int i = 0; i < 16; i++)
    if ((smask >> i) & 1) ones |= (uint64_t)1 << (4 * i);
  if (nfilled == 1) {
    float cl[4];
#pragma unroll
    for (int j = 0; j < NB; j++)
      if (j == last) {
#pragma unroll
        for (int k = 0; k < 4; k++) cl[k] = c[j][k];
      }
    const uint32_t e = single_color<NU>(f, sctab, to_pixel_f(cl, 0xFFFFFFFFu, -1), out.p1,
                                        out.p2, out.pbc, mu);
    out.err = NU ? e : (uint32_t)n * e;
    out.sc = true;
    out.idx = ones;
    out.anneal = false;
    return;
  }
  // least squares (Compressor.cpp:1053-1077)
  float asq = 0.0f, bsq = 0.0f, ab = 0.0f;
  float ax[4] = {0.0f, 0.0f, 0.0f, 0.0f}, bx[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < NB; i++) {
    const float fbi = (float)(NB - 1 - i);
    const float fb = (float)(NB - 1);
    const float fi = (float)i;
    const float fn = (float)cnt[i];
    const float a = fbi / fb;
    const float b = fi / fb;
    asq += fn * a * a;
    bsq += fn * b * b;
    ab += fn * a * b;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      ax[k] += c[i][k] * a * fn;
      bx[k] += c[i][k] * b * fn;
    }
  }
  const float fdet = 1.0f / (asq * bsq - ab * ab);
#pragma unroll
  for (int k = 0; k < 4; k++) {
    p1[k] = (ax[k] * bsq - bx[k] * ab) * fdet;
    p2[k] = (bx[k] * asq - ax[k] * ab) * fdet;
  }
  // ClampEndpointsToGrid (Compressor.cpp:212-250)
#pragma unroll
  for (int k = 0; k < 4; k++) {
    p1[k] = p1[k] < 0.0f ? 0.0f : (p1[k] > 255.0f ? 255.0f : p1[k]);
    p2[k] = p2[k] < 0.0f ? 0.0f : (p2[k] > 255.0f ? 255.0f : p2[k]);
  }
  int pbc = 0;
  uint32_t g1 = 0xFFFFFFFFu, g2 = 0xFFFFFFFFu;
  {
    const bool has_pb = f.npbc > 1;
    float mind = FLT_MAX;
    for (int i = 0; i < f.npbc; i++) {
      const uint32_t q1 = to_pixel_f(p1, f.qmask, has_pb ? pbc_bit(f.pbit_type, i, 0) : -1);
      const uint32_t q2 = to_pixel_f(p2, f.qmask, has_pb ? pbc_bit(f.pbit_type, i, 1) : -1);
      float n1[4], n2[4], d1[4], d2[4];
      unpack4f(q1, n1);
      unpack4f(q2, n2);
#pragma unroll
      for (int k = 0; k < 4; k++) {
        d1[k] = n1[k] - p1[k];
        d2[k] = n2[k] - p2[k];
      }
      const float dist = dot4(d1, d1) + dot4(d2, d2);
      if (dist < mind) {
        mind = dist;
        g1 = q1;
        g2 = q2;
        pbc = i;
      }
    }
  }
  // OptimizeEndpointsForCluster's start (Compressor.cpp:550-580): the error
  // is measured with the combo's p-bits even for modes without p-bits (it
  // always receives a combo), the state keeps the grid endpoints.
  const int nb = 1 << f.nbits_idx;
  const uint32_t q1 = to_pixel_int(g1, f.qmask, pbc_bit(f.pbit_type, pbc, 0));
  const uint32_t q2 = to_pixel_int(g2, f.qmask, pbc_bit(f.pbit_type, pbc, 1));
  if constexpr (NU) out.err = __float_as_uint(qerr_nu<1>(px, smask, ptmode, q1, q2, nb, *mr, out.idx));
  else out.err = qerr(px, smask, ptmode, q1, q2, nb, out.idx);
  out.sc = false;
  out.pbc = pbc;
  if (f.pbit_type != PB_NONE) {
    out.p1 = q1;
    out.p2 = q2;
  } else {
    out.p1 = to_pixel_int(g1, f.qmask, -1);
    out.p2 = to_pixel_int(g2, f.qmask, -1);
  }
  out.anneal = q > 0 && out.err > 0;
}

// CompressCluster, RGB variant (Compressor.cpp:921-1094) up to the annealing.
template <bool NU = false>
__device__ __forceinline__ void subset_setup(const Fit &f, uint32_t q, const uint32_t *sctab,
                             const uint32_t px[16], uint32_t smask, int ptmode, int n,
                             const float avg[4], bool all_same, SubStart &out,
                             const Weights *mu, const Weights *mr, uint32_t *km) {
  if (all_same) {
    const int first = __ffs(smask) - 1;
    uint32_t pt = 0;
#pragma unroll
    for (int i = 0; i < 16; i++)
      if (i == first) pt = point_of(px[i], ptmode);
    const uint32_t e = single_color<NU>(f, sctab, pt, out.p1, out.p2, out.pbc, mu);
    out.err = NU ? e : (uint32_t)n * e;
    out.sc = true;
    out.idx = 0;
#pragma unroll
    for (int i = 0; i < 16; i++)
      if ((smask >> i) & 1) out.idx |= (uint64_t)1 << (4 * i);
    out.anneal = false;
    return;
  }
  if (f.nbits_idx == 2)
    kmeans_setup<4, NU>(f, q, sctab, px, smask, ptmode, n, avg, out, mu, mr, km);
  else if (f.nbits_idx == 3)
    kmeans_setup<8, NU>(f, q, sctab, px, smask, ptmode, n, avg, out, mu, mr, km);
  else
    kmeans_setup<16, NU>(f, q, sctab, px, smask, ptmode, n, avg, out, mu, mr, km);
}

// The alpha channel of the rotation modes (Compressor.cpp:697-911): a 1-D
// k-means and least-squares fit (or the table lookup for a constant alpha).
// Returns the alpha error; a1q/a2q are the alpha bytes Pack will write
// (rounded, then quantised to the mode's alpha precision).  NU: the
// nonuniform metric, whose alpha term (a double sum of float per-pixel
// errors, weighted by the rotated alpha weight aw, Compressor.cpp:712) goes
// to *nu_err.
template <bool NU = false>
__device__ __forceinline__ uint32_t alpha_fit(const Fit &f, const uint32_t px[16], uint64_t &aidx, uint32_t &a1q,
                              uint32_t &a2q, uint32_t *km, float aw = 1.0f,
                              double *nu_err = nullptr) {
  const int src = f.rot == 0 ? 3 : f.rot - 1;
  uint32_t lo = 255, hi = 0;
#pragma unroll 1
  for (int i = 0; i < 16; i++) {
    const uint32_t v = chan(px[i], src);
    lo = v < lo ? v : lo;
    hi = v > hi ? v : hi;
  }
  const float amin = (float)lo, amax = (float)hi;
  const int abits = f.idx_mode == 0 ? kModes[f.mode].alpha_idx_bits : kModes[f.mode].idx_bits;
  const int nb = 1 << abits;
  float a1 = amin, a2 = amax;
  uint32_t alpha_err = 0;
  double alpha_nu = 0.0;
  aidx = 0;
  if (a1 == a2) {
    const uint32_t a1be = (uint32_t)a1, a2be = (uint32_t)a2;
    if (f.mode != 5) {
      if (kDxt6Tab[a1be][0][0]) {
        a1 = (float)((kDxt6Tab[a1be][1][1] << 2) | (kDxt6Tab[a1be][0][1] >> 4));
        a2 = (float)((kDxt6Tab[a2be][1][2] << 2) | (kDxt6Tab[a2be][0][1] >> 4));
      } else {
        a1 = (float)((kDxt6Tab[a1be][0][1] << 2) | (kDxt6Tab[a1be][0][1] >> 4));
        a2 = (float)((kDxt6Tab[a2be][0][2] << 2) | (kDxt6Tab[a2be][0][1] >> 4));
      }
      const uint32_t fill = f.idx_mode == 1 ? 1u : 2u;
#pragma unroll
      for (int i = 0; i < 16; i++) aidx |= (uint64_t)fill << (4 * i);
      const int w1 = kW[abits - 1][fill], w0 = 64 - w1;
      const uint32_t ip = (((uint32_t)a1 * w0) + ((uint32_t)a2 * w1) + 32) >> 6 & 0xFFu;
      const uint32_t d = a1be > ip ? a1be - ip : ip - a1be;
      alpha_err = 16 * d * d;
      if constexpr (NU) {
        float pe = aw * (float)d;
        pe *= pe;
        alpha_nu = (double)(16.0f * pe);
      }
    }
  } else {
    float vals[8];
#pragma unroll
    for (int i = 0; i < 8; i++) vals[i] = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; i++)
      if (i < nb) vals[i] = amin + ((float)i / (float)(nb - 1)) * (amax - amin);
    // every value into its nearest entry's LDS word, sum | count << 16 (as
    // for the colours, integer sums are the reference's float sums exactly)
    auto assign = [&]() {
#pragma unroll
      for (int j = 0; j < 8; j++) km[j * 64] = 0u;
#pragma unroll 1
      for (int i = 0; i < 16; i++) {
        const uint32_t val = chan(px[i], src);
        const float a = (float)val;
        float md = 255.0f;
        int b = 0;
#pragma unroll
        for (int j = 0; j < 8; j++) {
          if (j >= nb) continue;
          const float d = fabsf(a - vals[j]);
          if (d < md) {
            md = d;
            b = j;
          }
        }
        km_add(km + b * 64, val | 0x10000u);
      }
    };
    float npts[8];
    bool fixed = false;
    int guard = 0;
    assign();
    while (!fixed && guard++ < 4096) {
      fixed = true;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const uint32_t w = km[j * 64];
        // integer sum over a count of 0..16: the double product is the
        // correctly rounded quotient (as for the colour k-means)
        const float s = (float)((double)(w & 0xFFFFu) * kInvCount[w >> 16]);
        npts[j] = (float)(w >> 16);
        if (j < nb) fixed = fixed && (s == vals[j]);
        vals[j] = s;
      }
      if (!fixed) assign();
    }
    float asq = 0.0f, bsq = 0.0f, ab = 0.0f, ax = 0.0f, bx = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      if (i >= nb) continue;
      const float fbi = (float)(nb - 1 - i);
      const float fb = (float)(nb - 1);
      const float fi = (float)i;
      const float a = fbi / fb;
      const float b = fi / fb;
      const float n = npts[i];
      const float x = vals[i];
      asq += n * a * a;
      bsq += n * b * b;
      ab += n * a * b;
      ax += x * a * n;
      bx += x * b * n;
    }
    const float fd = 1.0f / (asq * bsq - ab * ab);
    a1 = fd * (ax * bsq - bx * ab);
    a2 = fd * (bx * asq - ax * ab);
    {
      float t = 0.0f < a1 ? a1 : 0.0f;
      a1 = t < 255.0f ? t : 255.0f;
      t = 0.0f < a2 ? a2 : 0.0f;
      a2 = t < 255.0f ? t : 255.0f;
    }
    // QuantizeChannel(uint8(a)) truncates here, while Pack rounds (:876-879)
    const uint32_t amask = (uint32_t)((int8_t)-0x7F >> (f.alpha_prec - 1)) & 0xFFu;
    const uint32_t a1b = quant_channel((uint32_t)a1 & 0xFFu, amask, -1);
    const uint32_t a2b = quant_channel((uint32_t)a2 & 0xFFu, amask, -1);
#pragma unroll 1
    for (int i = 0; i < 16; i++) {
      const uint32_t val = chan(px[i], src);
      uint32_t me = 0xFFFFFFFFu;
      float mef = FLT_MAX;
      uint32_t bb = 0;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        if (j >= nb) continue;
        const int w1 = kW[abits - 1][j], w0 = 64 - w1;
        const uint32_t ip = ((a1b * w0) + (a2b * w1) + 32) >> 6 & 0xFFu;
        const uint32_t d = val > ip ? val - ip : ip - val;
        if constexpr (NU) {
          float pe = aw * (float)d;
          pe *= pe;
          if (pe < mef) {
            mef = pe;
            bb = (uint32_t)j;
          }
        } else {
          const uint32_t e = d * d;
          if (e < me) {
            me = e;
            bb = (uint32_t)j;
          }
        }
      }
      if constexpr (NU) alpha_nu += (double)mef;
      else alpha_err += me;
      aidx |= (uint64_t)bb << (4 * i);
    }
  }
  const uint32_t am = chan(f.qmask, 3);
  a1q = quant_channel(round_half_up(a1) & 0xFFu, am, -1);
  a2q = quant_channel(round_half_up(a2) & 0xFFu, am, -1);
  if constexpr (NU) *nu_err = alpha_nu;
  return alpha_err;
}

// ---------------------------------------------------------------------------
// Work items.
// ---------------------------------------------------------------------------

// Candidates of a block: one per (mode, shape entry) of CompressClusters
// (Compressor.cpp:1771-1809), with the rotation modes split per (rotation,
// index mode), stored in the order the reference tries them (modes 0, 2, 1,
// 3, 7, 4, 5, 6; shape entries; rotations; index modes), so that the first
// strict minimum over the slots is the reference's choice.  Up to 32 slots
// per block (16 in Compress's search; CompressWithStats runs modes 4, 5 and
// 6 once per shape entry), each a 16-bit descriptor:
//   mode 3 | shape 6 << 3 | rotation 2 << 9 | index mode 1 << 11 | entry 3 << 12
// (entry = the shape selection's entry, 0..4, which keys the annealing stream).
// Candidate types (work queues, sorted so that a wave runs one code path):
//   0 mode 0, 1 mode 2, 2 mode 1, 3 mode 3, 4 mode 7, 5 mode 6, 6 mode 4, 7 mode 5.
constexpr int kNumTypes = 8;
constexpr int kSlotBits = 5;
constexpr int kMaxCands = 1 << kSlotBits;
constexpr int kMaxBoxCands = 16;  // slots of a BoxSelection or learned block
// most candidates of one type a block can have (mode 4: 8 per shape entry)
constexpr int kMaxPerType = 16;

// Candidate id: relative block << kSlotBits | slot; also the candidate's
// index in the per-slot arrays (block * kMaxCands + slot).
__host__ __device__ __forceinline__ uint32_t cand_id(uint32_t rel, uint32_t slot) {
  return (rel << kSlotBits) | slot;
}
__host__ __device__ __forceinline__ uint32_t id_block(uint32_t id) { return id >> kSlotBits; }
__host__ __device__ __forceinline__ uint32_t id_slot(uint32_t id) {
  return id & (kMaxCands - 1u);
}
__constant__ int kTypeOfMode[8] = {0, 2, 1, 3, 6, 7, 5, 4};

// Block class and candidate count, packed: cls 2 | count 5 << 2 (at most 31).
// kSelFull marks a block of the learned search that runs the full search
// (the ranker was not confident): every candidate annealed, the reference's
// choice by internal error, the quality guard.
__device__ __forceinline__ uint32_t sel_pack(int cls, int count) {
  return (uint32_t)cls | ((uint32_t)count << 2);
}
constexpr uint32_t kSelFull = 1u << 7;
__device__ __forceinline__ int sel_cls(uint32_t s) { return s & 3; }
__device__ __forceinline__ int sel_count(uint32_t s) { return (s >> 2) & 31; }
__device__ __forceinline__ bool sel_full(uint32_t s) { return (s & kSelFull) != 0; }

struct Cand {
  int mode, entry, rot, im, shape, nsub;
};

__device__ __forceinline__ uint32_t cdesc_pack(int mode, int shape, int rot, int im, int entry) {
  return (uint32_t)mode | ((uint32_t)shape << 3) | ((uint32_t)rot << 9) | ((uint32_t)im << 11) |
         ((uint32_t)entry << 12);
}

__device__ __forceinline__ void cand_from_desc(uint32_t d, Cand &k) {
  k.mode = d & 7;
  k.shape = (d >> 3) & 63;
  k.rot = (d >> 9) & 3;
  k.im = (d >> 11) & 1;
  k.entry = (d >> 12) & 7;
  k.nsub = kModes[k.mode].subsets;
}

// The candidate list of a searched block after BoxSelection, in the
// reference's order (see above).  Returns the count.
__device__ int box_candidates(bool opaque_layout, int nshapes, int s2, int s3, uint32_t modes,
                              uint32_t q, uint16_t out[kMaxBoxCands]) {
  int n = 0;
  if (opaque_layout) {
    if (nshapes >= 2) {
      if (((modes >> 0) & 1) && s3 < 16) out[n++] = (uint16_t)cdesc_pack(0, s3, 0, 0, 1);
      if ((modes >> 2) & 1) out[n++] = (uint16_t)cdesc_pack(2, s3, 0, 0, 1);
    }
    if ((modes >> 1) & 1) out[n++] = (uint16_t)cdesc_pack(1, s2, 0, 0, 0);
    if ((modes >> 3) & 1) out[n++] = (uint16_t)cdesc_pack(3, s2, 0, 0, 0);
    if ((modes >> 7) & 1) out[n++] = (uint16_t)cdesc_pack(7, s2, 0, 0, 0);
    if ((modes >> 6) & 1) {
      out[n++] = (uint16_t)cdesc_pack(6, s2, 0, 0, 0);
      // both mode-6 entries fit the same 16 pixels; without annealing the
      // second repeats the first exactly and cannot win (strict <)
      if (nshapes >= 2 && q > 0) out[n++] = (uint16_t)cdesc_pack(6, s3, 0, 0, 1);
    }
  } else {
    if ((modes >> 7) & 1) out[n++] = (uint16_t)cdesc_pack(7, s2, 0, 0, 0);
    if ((modes >> 4) & 1)
      for (int c = 0; c < 8; c++) out[n++] = (uint16_t)cdesc_pack(4, 0, c >> 1, c & 1, 0);
    if ((modes >> 5) & 1)
      for (int c = 0; c < 4; c++) out[n++] = (uint16_t)cdesc_pack(5, 0, c, 0, 0);
    if ((modes >> 6) & 1) out[n++] = (uint16_t)cdesc_pack(6, s2, 0, 0, 0);
  }
  return n;
}

// CandRec::meta bit set when annealing rewrote the record.
constexpr uint32_t kMetaAnnealed = 1u << 12;

// Result of one candidate, read by the pack kernel.
struct CandRec {
  uint32_t err;       // total error; 0xFFFFFFFF = not a candidate
  uint32_t px1[3], px2[3];
  uint32_t cidx_lo, cidx_hi;
  uint32_t aidx_lo, aidx_hi;
  uint32_t meta;      // pbc per subset (2 bits each) | rot << 8 | im << 10 | annealed << 12
};

// Annealing work item (start state from the set-up kernel).
struct AState {
  uint32_t id;        // cand_id(relative block, slot)
  uint32_t info;      // mode | rot << 3 | im << 5 | nsub << 6 | shape << 8 | active << 14 | entry 3 << 17
  uint32_t p1[3], p2[3];
  uint32_t err[3];
  uint32_t pbc;       // 2 bits per subset
  uint32_t idx_lo, idx_hi;
  uint32_t extra_err; // alpha error of rotation candidates
  uint32_t pad;
};

// Learned search: candidates whose quality-0 block decodes to more than
// 1 + 1/kAnnealMarginDiv times the block's best quality-0 error are not
// annealed (annealing lowers a fit's error by a few percent at most).
constexpr unsigned long long kAnnealMarginDiv = 50;

// Word offsets of the counters.  Each that is counted up while others are read
// has a cache line of its own: an atomic takes some 7 ns of its line, and
// loads of a line under atomics wait for them (with all of them on two lines,
// reading the three state counts at every refill took the 508x380 annealing
// from 2.0 to 3.2 ms, and mode 4's set-up at 4096 x 4096 1.6 to 3.4).
enum {
  kCntQueue = 0,         // 8 words: the type queues' sizes
  kCntFront = 32,        // annealing states of the modes without rotation
  kCntRot4 = 64,         // and of modes 4
  kCntRot5 = 96,         // and 5
  kCntFetch = 128,       // annealing states taken
  kCntList = 160,        // length of the learned annealing list
  kCntFallback = 192,    // learned search: blocks for the full search
  kCntRotFetch = 224,    // learned search: rotation states taken
  kCntTail = 256,        // candidates handed over
  kCntTailFetch = 288,   // and taken
  kCntWords = 320
};

struct Work {
  uint32_t *sel;          // per block
  uint16_t *cdesc;        // per block x 16 candidate descriptors
  CandRec *rec;           // per block x 16
  uint32_t *queue;        // per-type candidate queues, kMaxPerType entries per block each
  // see kCnt*
  uint32_t *counters;
  // the annealing states: those of the modes without rotation from the front,
  // the rotation modes' at the back (state_map)
  AState *astate;
  uint32_t qcap;          // entries per type queue
  uint32_t astate_cap;
  // learned search: the annealing states to run (slots of astate, in
  // order), kCntList of them; null in the reference search
  const uint32_t *alist;
  // learned search: astate[i].id for every state (read when the list is
  // built, without touching the 64-byte states); null in the reference search
  uint32_t *aid;
  // nonuniform metric: each candidate's total error, the double the
  // reference compares (per block x kMaxCands); null under the uniform metric
  double *nu_total;
};

// Annealing state i of the kCntFront, kCntRot4 and kCntRot5: its slot of astate.
// The rotation modes come last, mode 5 after mode 4: the longer a mode's
// chains, the earlier annealing starts on them (it runs from the end).  The
// three regions cannot meet: mode 4's lies below room for every candidate of
// mode 5, and a job's candidates all fit.
// (Read once per kernel, plainly: the counts stand when it starts.  Volatile
// loads go past the caches, and every wave's to the same lines, one after
// another: some 100 us of an annealing of 3072 waves.)
struct StateMap {
  uint32_t front, c4, c5, base4, base5;
  __device__ __forceinline__ uint32_t count() const { return front + c4 + c5; }
  __device__ __forceinline__ uint32_t slot(uint32_t i) const {
    if (i < front) return i;
    i -= front;
    return i < c4 ? base4 + i : base5 + (i - c4);
  }
};
__device__ __forceinline__ StateMap state_map(const Work &w) {
  const uint32_t *c = w.counters;
  StateMap m;
  m.front = c[kCntFront];
  m.c4 = c[kCntRot4];
  m.c5 = c[kCntRot5];
  m.base4 = w.astate_cap - c[kCntQueue + 7] - m.c4;  // below room for mode 5's whole queue
  m.base5 = w.astate_cap - m.c5;
  return m;
}

// Whether an annealing list of `total` states runs one lane per pixel
// (anneal_spread_kernel) rather than one lane per candidate (anneal_kernel);
// the two are launched together and this decides on the device, where the
// count is.  Rotation states have the longest chains, which set the one-lane
// form's time, so a list with at least one in eight of them may be twice as
// long.  Annealing in ms, one lane per pixel against one per candidate:
//   quality 50, few rotation states: 24,000 states 0.27 / 0.73, 66,000
//     (learned search) 0.86 / 1.04, 95,000 0.89 / 0.82, 188,000 1.95 / 1.02;
//   quality 50, many: 30,000 1.04 / 2.62, 141,000 2.49 / 2.85, 187,000
//     3.28 / 3.11, 229,000 (noise) 7.56 / 4.22;
//   quality 8, few: 24,000 0.13 / 0.17, 54,000 0.27 / 0.21;
//   quality 8, many: 68,000 0.62 / 0.64, 120,000 0.97 / 0.62.
// By the number of blocks alone, the rule before, a learned job of 64,000
// blocks none of which the ranker was sure about annealed its 457,000 states
// in 7.9 ms; 4.2 now.
constexpr uint32_t kSpreadStates = 90112, kSpreadStatesShort = kSpreadStates / 2;
constexpr uint32_t kShortChains = 16;  // the quality below which the chains are short
__device__ __forceinline__ bool spread_list(const StateMap &m, uint32_t total,
                                            uint32_t max_states) {
  return total <= (8u * (m.c4 + m.c5) >= total ? 2u * max_states : max_states);
}

// Learned search: the list of annealing states that pass the margin, in
// the order of state_map (for large jobs the set-up kernels append by mode, so
// annealing waves stay uniform; the list's end holds the rotation modes).  An ordered
// compaction over chunks of 4096 states: per-chunk counts, their exclusive
// scan, then each chunk writes its passing states from its offset.
constexpr uint32_t kListChunk = 4096;

// Flags of the states cb + 256 k + t (k = 0..15) of thread t: bit k set when
// the state passes the margin.  Adjacent lanes read adjacent states.
__device__ __forceinline__ uint32_t list_flags(const Work &w, const StateMap &sm,
                                               const unsigned long long *cerr,
                                               const unsigned long long *q0best, uint32_t cb,
                                               int t) {
  uint32_t flags = 0;
#pragma unroll
  for (int k = 0; k < 16; k++) {
    const uint32_t i = cb + 256u * (uint32_t)k + (uint32_t)t;
    if (i < sm.count()) {
      const uint32_t id = w.aid[sm.slot(i)];
      const uint32_t rel = id_block(id);
      const unsigned long long best = q0best[rel];
      // a full-search block anneals every candidate
      if (sel_full(w.sel[rel]) || cerr[id] <= best + best / kAnnealMarginDiv) flags |= 1u << k;
    }
  }
  return flags;
}

// Exclusive prefix over the 256 threads of a workgroup; returns the total.
__device__ __forceinline__ uint32_t wg_exclusive_scan(uint32_t v, uint32_t *excl,
                                                      uint32_t *s_wave) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint32_t incl = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t u = __shfl_up(incl, o);
    if (lane >= o) incl += u;
  }
  if (lane == 63) s_wave[wave] = incl;
  __syncthreads();
  uint32_t before = 0, all = 0;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    before += q < wave ? s_wave[q] : 0u;
    all += s_wave[q];
  }
  *excl = before + incl - v;
  return all;
}

__global__ void __launch_bounds__(256) list_count_kernel(Work w, const unsigned long long *cerr,
                                                         const unsigned long long *q0best,
                                                         uint32_t *chunk_count) {
  __shared__ uint32_t s_wave[4];
  const StateMap sm = state_map(w);
  const uint32_t cb = blockIdx.x * kListChunk;
  if (cb >= sm.count()) return;  // whole workgroup
  const uint32_t flags = list_flags(w, sm, cerr, q0best, cb, threadIdx.x);
  uint32_t excl;
  const uint32_t all = wg_exclusive_scan((uint32_t)__popc(flags), &excl, s_wave);
  if (threadIdx.x == 0) chunk_count[blockIdx.x] = all;
}

// One workgroup: exclusive scan of the chunk counts (at most 64 per thread),
// the list length into kCntList.
__global__ void __launch_bounds__(256) list_scan_kernel(Work w, uint32_t *chunk_count) {
  __shared__ uint32_t s_wave[4];
  const uint32_t nchunks = (state_map(w).count() + kListChunk - 1) / kListChunk;
  const uint32_t per = (nchunks + 255) / 256;
  const uint32_t c0 = threadIdx.x * per;
  uint32_t sum = 0;
  for (uint32_t c = c0; c < c0 + per && c < nchunks; c++) sum += chunk_count[c];
  uint32_t excl;
  const uint32_t all = wg_exclusive_scan(sum, &excl, s_wave);
  for (uint32_t c = c0; c < c0 + per && c < nchunks; c++) {
    const uint32_t v = chunk_count[c];
    chunk_count[c] = excl;
    excl += v;
  }
  if (threadIdx.x == 0) w.counters[kCntList] = all;
}

__global__ void __launch_bounds__(256) list_write_kernel(Work w, const unsigned long long *cerr,
                                                         const unsigned long long *q0best,
                                                         const uint32_t *chunk_offset,
                                                         uint32_t *alist) {
  const StateMap sm = state_map(w);
  const uint32_t cb = blockIdx.x * kListChunk;
  if (cb >= sm.count()) return;  // whole workgroup
  const uint32_t flags = list_flags(w, sm, cerr, q0best, cb, threadIdx.x);
  // round k places the passing states cb + 256 k .. cb + 256 k + 255 in
  // order: rank within the wave by ballot, then the waves before it
  __shared__ uint32_t s_round[2][4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t pos = chunk_offset[blockIdx.x];
#pragma unroll
  for (int k = 0; k < 16; k++) {
    const bool f = (flags >> k) & 1u;
    const uint64_t m = __ballot(f);
    if (lane == 0) s_round[k & 1][wave] = (uint32_t)__popcll(m);
    __syncthreads();
    uint32_t before = 0, all = 0;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      before += q < wave ? s_round[k & 1][q] : 0u;
      all += s_round[k & 1][q];
    }
    if (f)
      alist[pos + before + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] =
          sm.slot(cb + 256u * (uint32_t)k + (uint32_t)threadIdx.x);
    pos += all;
  }
}

__device__ __forceinline__ void load_block(const BlockRange &r, uint32_t rel, uint32_t px[16]) {
  const uint32_t b = r.first_block + rel;
  const uint32_t bx = b % r.blocks_wide, by = b / r.blocks_wide;
  const uint32_t *p = r.img + (size_t)(by * 4) * r.width + bx * 4;
#pragma unroll
  for (int y = 0; y < 4; y++) {
    const uint4 row = *reinterpret_cast<const uint4 *>(p + (size_t)y * r.width);
    px[y * 4 + 0] = row.x;
    px[y * 4 + 1] = row.y;
    px[y * 4 + 2] = row.z;
    px[y * 4 + 3] = row.w;
  }
}

__device__ __forceinline__ uint32_t idx_at(uint32_t lo, uint32_t hi, int i) {
  return i < 8 ? (lo >> (4 * i)) & 0xFu : (hi >> (4 * (i - 8))) & 0xFu;
}

// Key of one fit's annealing stream; shape entries 0..4 take bits 3-4 and 10.
__device__ __forceinline__ uint32_t cand_tag(int mode, int entry, int subset, int rot, int im) {
  return (uint32_t)mode | ((uint32_t)(entry & 3) << 3) | ((uint32_t)subset << 5) |
         ((uint32_t)rot << 7) | ((uint32_t)im << 9) | ((uint32_t)(entry >> 2) << 10);
}

// Appends the workgroup's valid candidates to their type queues: slots are
// taken with LDS atomics, then one global atomic per type per workgroup.
// Every thread of the workgroup must call it.
__device__ __forceinline__ void wg_enqueue(Work &w, bool valid, int type, uint32_t id,
                                           uint32_t *s_cnt, uint32_t *s_base) {
  const int t = threadIdx.x;
  if (t < kNumTypes) s_cnt[t] = 0;
  __syncthreads();
  uint32_t local = 0;
  if (valid) local = atomicAdd(&s_cnt[type], 1u);
  __syncthreads();
  if (t < kNumTypes && s_cnt[t]) s_base[t] = atomicAdd(&w.counters[kCntQueue + t], s_cnt[t]);
  __syncthreads();
  if (valid) w.queue[(size_t)type * w.qcap + s_base[type] + local] = id;
}

// The nonuniform metric's pixel pass (the metric is described above qerr_nu):
// the same two neighbouring indices, scored under the weights (pair lanes:
// .x channels 0 / 1, .y 2 / 3), the second kept only when strictly better.
__device__ __forceinline__ float pixel_err_nu(uint32_t p02, uint32_t p13, const SubConst &c,
                                              float kf, WeightFn wf, const Weights &m,
                                              uint32_t *best) {
  uint32_t j1, j2;
  pixel_bounds(p02, p13, c, kf, j1, j2);
  const s16x2 z02 = as_s16x2(c.a02) - as_s16x2(p02), z13 = as_s16x2(c.a13) - as_s16x2(p13);
  const uint32_t w1 = weight_word(wf, j1), w2 = weight_word(wf, j2);
  const s16x2 x02 = interp_diff(z02, c.d02, w1), x13 = interp_diff(z13, c.d13, w1);
  const s16x2 y02 = interp_diff(z02, c.d02, w2), y13 = interp_diff(z13, c.d13, w2);
  const float e1 = werr(x02.x, x13.x, x02.y, x13.y, m);
  const float e2 = werr(y02.x, y13.x, y02.y, y13.y, m);
  *best = e2 < e1 ? j2 : j1;
  return e2 < e1 ? e2 : e1;
}

__device__ __forceinline__ SubConst pick_sub(bool c, const SubConst &x, const SubConst &y) {
  SubConst r;
  r.a02 = c ? x.a02 : y.a02;
  r.a13 = c ? x.a13 : y.a13;
  r.ad = c ? x.ad : y.ad;
  r.d02 = c ? x.d02 : y.d02;
  r.d13 = c ? x.d13 : y.d13;
  r.q02 = c ? x.q02 : y.q02;
  r.q13 = c ? x.q13 : y.q13;
  r.rl = c ? x.rl : y.rl;
  return r;
}

// Subset of pixel i under shape masks m1, m2 (0 when the bit of m1 is clear).
__device__ __forceinline__ uint32_t subset_of(uint32_t m1, uint32_t m2, int i) {
  return ((m1 >> i) & 1u) ? 1u + ((m2 >> i) & 1u) : 0u;
}

// Bounding-box corners of every subset of a shape (GetBoundingBox after
// SetPartition, RGBAEndpoints.h:205-226), as packed RGBA8.
template <int NS>
__device__ __forceinline__ void subset_corners(const uint32_t px[16], uint32_t m1, uint32_t m2,
                                               uint32_t lo[NS], uint32_t hi[NS]) {
  uint32_t mn02[NS], mn13[NS], mx02[NS], mx13[NS];
#pragma unroll
  for (int t = 0; t < NS; t++) {
    mn02[t] = mn13[t] = 0x00FF00FFu;
    mx02[t] = mx13[t] = 0u;
  }
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const uint32_t s = subset_of(m1, m2, i);
    const u16x2 p02 = as_u16x2(px[i] & 0x00FF00FFu), p13 = as_u16x2((px[i] >> 8) & 0x00FF00FFu);
#pragma unroll
    for (int t = 0; t < NS; t++) {
      const bool in = s == (uint32_t)t;
      const u16x2 top = {0xFF, 0xFF}, bottom = {0, 0};
      mn02[t] = __builtin_bit_cast(uint32_t,
                                   __builtin_elementwise_min(as_u16x2(mn02[t]), in ? p02 : top));
      mn13[t] = __builtin_bit_cast(uint32_t,
                                   __builtin_elementwise_min(as_u16x2(mn13[t]), in ? p13 : top));
      mx02[t] = __builtin_bit_cast(uint32_t,
                                   __builtin_elementwise_max(as_u16x2(mx02[t]), in ? p02 : bottom));
      mx13[t] = __builtin_bit_cast(uint32_t,
                                   __builtin_elementwise_max(as_u16x2(mx13[t]), in ? p13 : bottom));
    }
  }
#pragma unroll
  for (int t = 0; t < NS; t++) {
    lo[t] = mn02[t] | (mn13[t] << 8);
    hi[t] = mx02[t] | (mx13[t] << 8);
  }
}

// BoxSelection's estimate of one partition shape (EstimateTwoClusterError /
// EstimateThreeClusterError, Compressor.cpp:1626-1655): the sum over subsets
// of 0.0001 + QuantizedError of the subset's points between its bounding-box
// corners (no quantisation, NB index entries), 0 for a one-colour subset.  Each
// pixel is scored once, against its own subset's corners; per-subset errors
// are exact integers, added in double in subset order as the reference does.
template <int NS, int NB>
__device__ __forceinline__ double shape_estimate(const uint32_t px[16], int shape) {
  const uint32_t m1 = NS == 2 ? (uint32_t)kShape2[shape] : (uint32_t)kShape3[shape][0];
  const uint32_t m2 = NS == 3 ? (uint32_t)kShape3[shape][1] : 0u;
  uint32_t lo[NS], hi[NS];
  subset_corners<NS>(px, m1, m2, lo, hi);
  SubConst c[NS];
  bool flat[NS];
#pragma unroll
  for (int t = 0; t < NS; t++) {
    c[t] = sub_const(lo[t], hi[t]);
    flat[t] = lo[t] == hi[t];
  }
  const WeightFn wf = weight_fn(NB);
  uint32_t e[NS];
#pragma unroll
  for (int t = 0; t < NS; t++) e[t] = 0;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const uint32_t s = ((m1 >> i) & 1u) ? 1u + ((m2 >> i) & 1u) : 0u;
    const SubConst k = NS == 2 ? pick_sub(s != 0, c[1], c[0])
                               : pick_sub(s == 0, c[0], pick_sub(s == 1, c[1], c[NS - 1]));
    uint32_t best;
    const uint32_t me =
        pixel_err(pair02x64(px[i]), pair13x64(px[i]), k, (float)(NB - 1), wf, &best);
#pragma unroll
    for (int t = 0; t < NS; t++) e[t] += s == (uint32_t)t ? me : 0u;
  }
  double err = 0.0;
#pragma unroll
  for (int t = 0; t < NS; t++) {
    if (!flat[t]) err += 0.0001 + (double)e[t];
    else err += 0.0;
  }
  return err;
}

// shape_estimate under the nonuniform metric's unrotated weights
// (Compressor.cpp:1634, 1650): each subset's error is a float sum in pixel
// order, added to 0.0001 in double.
template <int NS, int NB>
__device__ __forceinline__ double shape_estimate_nu(const uint32_t px[16], int shape,
                                                    const Weights &m) {
  const uint32_t m1 = NS == 2 ? (uint32_t)kShape2[shape] : (uint32_t)kShape3[shape][0];
  const uint32_t m2 = NS == 3 ? (uint32_t)kShape3[shape][1] : 0u;
  uint32_t lo[NS], hi[NS];
  subset_corners<NS>(px, m1, m2, lo, hi);
  SubConst c[NS];
  bool flat[NS];
#pragma unroll
  for (int t = 0; t < NS; t++) {
    c[t] = sub_const(lo[t], hi[t]);
    flat[t] = lo[t] == hi[t];
  }
  const WeightFn wf = weight_fn(NB);
  float e[NS];
#pragma unroll
  for (int t = 0; t < NS; t++) e[t] = 0.0f;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const uint32_t s = ((m1 >> i) & 1u) ? 1u + ((m2 >> i) & 1u) : 0u;
    const SubConst k = NS == 2 ? pick_sub(s != 0, c[1], c[0])
                               : pick_sub(s == 0, c[0], pick_sub(s == 1, c[1], c[NS - 1]));
    uint32_t best;
    const float me =
        pixel_err_nu(pair02x64(px[i]), pair13x64(px[i]), k, (float)(NB - 1), wf, m, &best);
#pragma unroll
    for (int t = 0; t < NS; t++) e[t] += s == (uint32_t)t ? me : 0.0f;
  }
  double err = 0.0;
#pragma unroll
  for (int t = 0; t < NS; t++) {
    if (!flat[t]) err += 0.0001 + (double)e[t];
  }
  return err;
}

// ---------------------------------------------------------------------------
// Kernel 1: classification and BoxSelection (Compressor.cpp:1670-1750,
// 1819-1860), lane i scoring shape i; the candidates go to per-type queues.
// ---------------------------------------------------------------------------
// Classification (solid / transparent / searched) and BoxSelection of one
// block by a whole wave (lane i scores two- and three-subset shape i); the
// block's candidates in CompressClusters' order go to cd.  Returns the
// packed class and count.
template <bool NU>
__device__ uint32_t box_select_block(uint32_t px[16], int lane, const Bc7Params &prm,
                                     uint16_t cd[kMaxBoxCands]) {
  bool solid = true, transparent = true, opaque = true;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    solid = solid && px[i] == px[0];
    transparent = transparent && (px[i] >> 24) == 0;
    opaque = opaque && (px[i] >> 24) >= 250;
  }
  uint32_t sel;
  int count = 0;
  if (solid) {
    sel = sel_pack(0, 0);
  } else if (transparent) {
    sel = sel_pack(1, 0);
  } else {
    double err2, err3;
    // The first estimate ends before the second starts, and the second's
    // texel pairs are its own: left to the compiler the two run into each
    // other and share 32 registers of pairs, which takes 214 (nonuniform
    // metric 219) VGPRs and two waves a SIMD where 109 (108) give four.
    // 4096x4096: 4.89 -> 4.06 ms, nonuniform 6.75 -> 5.79.
    auto settle = [&]() {
      asm volatile("" : "+v"(err2));
#pragma unroll
      for (int i = 0; i < 16; i++) asm volatile("" : "+v"(px[i]));
    };
    if constexpr (NU) {
      const Weights m = params_weights(prm);
      err2 = shape_estimate_nu<2, 8>(px, lane, m);
      settle();
      err3 = opaque ? shape_estimate_nu<3, 4>(px, lane, m) : 0.0;
    } else {
      err2 = shape_estimate<2, 8>(px, lane);
      settle();
      err3 = opaque ? shape_estimate<3, 4>(px, lane) : 0.0;
    }
    double v2 = err2, v3 = err3;
    int i2 = lane, i3 = lane;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
      const double o2 = __shfl_xor(v2, off);
      const int oi2 = __shfl_xor(i2, off);
      if (o2 < v2 || (o2 == v2 && oi2 < i2)) {
        v2 = o2;
        i2 = oi2;
      }
      const double o3 = __shfl_xor(v3, off);
      const int oi3 = __shfl_xor(i3, off);
      if (o3 < v3 || (o3 == v3 && oi3 < i3)) {
        v3 = o3;
        i3 = oi3;
      }
    }
    uint32_t modes;
    bool opaque_layout = true;
    int nshapes = 1, s3 = 0;
    if (v2 < 1e-9) {
      modes = (1u << 1) | (1u << 3) | (1u << 7);
    } else if (!opaque) {
      modes = (1u << 4) | (1u << 5) | (1u << 6) | (1u << 7);
      opaque_layout = false;
    } else {
      modes = 0xFFu & ~((1u << 4) | (1u << 5));
      nshapes = 2;
      s3 = i3;
      if (v3 < 1e-9) modes = (1u << 0) | (1u << 2);
    }
    count = box_candidates(opaque_layout, nshapes, i2, s3, modes & prm.block_modes,
                           prm.quality, cd);
    sel = sel_pack(2, count);
  }
  return sel;
}

// ---------------------------------------------------------------------------
// CompressWithStats' block path (Compressor.cpp:1954-2183): its own shape
// scan and the statistics it logs.
// ---------------------------------------------------------------------------
// QuantizedError of every subset of a shape between its bounding-box corners
// quantised with endpoint masks mask_a and mask_b (ToPixel without p-bit,
// RGBAEndpoints.cpp:167-177), NB index entries: ea/eb per subset (exact
// integers), flat when the subset is one colour.  Each pixel is scored once
// per mask, against its own subset's endpoints; TWO = false scores mask_a only.
template <int NS, int NB, bool TWO = true>
__device__ __forceinline__ void masked_subset_errors(const uint32_t px[16], uint32_t m1,
                                                     uint32_t m2, uint32_t mask_a,
                                                     uint32_t mask_b, bool flat[NS],
                                                     uint32_t ea[NS], uint32_t eb[NS]) {
  uint32_t lo[NS], hi[NS];
  subset_corners<NS>(px, m1, m2, lo, hi);
  SubConst ca[NS], cb[NS];
#pragma unroll
  for (int t = 0; t < NS; t++) {
    flat[t] = lo[t] == hi[t];
    ca[t] = sub_const(to_pixel_int(lo[t], mask_a, -1), to_pixel_int(hi[t], mask_a, -1));
    cb[t] = sub_const(to_pixel_int(lo[t], mask_b, -1), to_pixel_int(hi[t], mask_b, -1));
    ea[t] = eb[t] = 0;
  }
  const WeightFn wf = weight_fn(NB);
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const uint32_t sub = subset_of(m1, m2, i);
    SubConst ka = ca[0], kb = cb[0];
#pragma unroll
    for (int t = 1; t < NS; t++) {
      ka = pick_sub(sub == (uint32_t)t, ca[t], ka);
      kb = pick_sub(sub == (uint32_t)t, cb[t], kb);
    }
    const uint32_t p02 = pair02x64(px[i]), p13 = pair13x64(px[i]);
    uint32_t best;
    const uint32_t xa = pixel_err(p02, p13, ka, (float)(NB - 1), wf, &best);
    const uint32_t xb = TWO ? pixel_err(p02, p13, kb, (float)(NB - 1), wf, &best) : 0u;
#pragma unroll
    for (int t = 0; t < NS; t++) {
      ea[t] += sub == (uint32_t)t ? xa : 0u;
      eb[t] += sub == (uint32_t)t ? xb : 0u;
    }
  }
}

// std::min(a, b): b only when strictly smaller.
__device__ __forceinline__ double min_ref(double a, double b) { return b < a ? b : a; }

// One shape of the statistics scan (EstimateTwoClusterErrorStats and
// EstimateThreeClusterErrorStats, Compressor.cpp:1862-1935, summed over the
// subsets as at :2074-2092 and :2124-2141): the selection error and the two
// per-mode estimates (modes 1 and 3 for two subsets, 0 and 2 for three), in
// the reference's double operations and order.
template <int NS>
__device__ __forceinline__ double stats_shape(const uint32_t px[16], int shape, double &est_a,
                                              double &est_b) {
  constexpr int NB = NS == 2 ? 8 : 4;
  const uint32_t m1 = NS == 2 ? (uint32_t)kShape2[shape] : (uint32_t)kShape3[shape][0];
  const uint32_t m2 = NS == 3 ? (uint32_t)kShape3[shape][1] : 0u;
  const uint32_t mask_a = NS == 2 ? 0xFFFCFCFCu : 0xFFF0F0F0u;
  const uint32_t mask_b = NS == 2 ? 0xFFFEFEFEu : 0xFFF8F8F8u;
  bool flat[NS];
  uint32_t ea[NS], eb[NS];
  masked_subset_errors<NS, NB>(px, m1, m2, mask_a, mask_b, flat, ea, eb);
  double err = 0.0;
#pragma unroll
  for (int t = 0; t < NS; t++) {
    double x = 0.0, sa = 0.0, sb = 0.0;
    if (!flat[t]) {
      // two subsets: the estimates are the errors; three: 0.0001 + the errors
      sa = NS == 2 ? (double)ea[t] : 0.0001 + (double)ea[t];
      sb = NS == 2 ? (double)eb[t] : 0.0001 + (double)eb[t];
      x = 0.0001;
      x += min_ref(sa, sb);
    }
    err += x;
    est_a = t == 0 ? sa : est_a + sa;
    est_b = t == 0 ? sb : est_b + sb;
  }
  return err;
}

__device__ __forceinline__ double wave_min(double v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = fmin(v, __shfl_xor(v, off));
  return v;
}

// The scan over 64 shapes, lane i holding shape i's error: the scan stops
// after the first shape below 1e-9 (brk, 64 if none); a shape is logged when
// strictly below every earlier scanned one (bestError starts at DBL_MAX).
// The logged errors go to log[], in shape order, the rest of its 64 entries
// are zeroed; returns the mask of logged shapes (the last of them is the
// chosen shape).
__device__ __forceinline__ uint64_t stats_scan(double err, int lane, int &brk, double *log) {
  const uint64_t under = __ballot(err < 1e-9);
  brk = under ? __ffsll((unsigned long long)under) - 1 : 64;
  const bool scanned = lane <= brk;
  double pm = scanned ? err : DBL_MAX;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const double u = __shfl_up(pm, o);
    if (lane >= o) pm = fmin(pm, u);
  }
  double before = __shfl_up(pm, 1);
  if (lane == 0) before = DBL_MAX;
  const bool logged = scanned && err < before;
  const uint64_t mask = __ballot(logged);
  if (logged) log[__popcll(mask & ((1ull << lane) - 1ull))] = err;
  if (lane >= __popcll(mask)) log[lane] = 0.0;
  return mask;
}

// The candidates of a statistics block in CompressClusters' order
// (Compressor.cpp:1771-1809) for the shape entries (2 subsets, s2) and, on
// opaque blocks, (3 subsets, s3): a single-subset mode runs once per entry;
// without annealing its second entry repeats the first exactly and cannot
// win (strict <), so it is left out.
__device__ int stats_candidates(int nshapes, int s2, int s3, uint32_t modes, uint32_t q,
                                uint16_t out[kMaxCands]) {
  constexpr int kOrder[8] = {0, 2, 1, 3, 7, 4, 5, 6};
  int n = 0;
#pragma unroll
  for (int mi = 0; mi < 8; mi++) {
    const int mode = kOrder[mi];
    if (!((modes >> mode) & 1)) continue;
    for (int e = 0; e < nshapes; e++) {
      const int parts = e == 0 ? 2 : 3, idx = e == 0 ? s2 : s3;
      const int nsub = kModes[mode].subsets;
      if (nsub != 1 && nsub != parts) continue;
      if (mode == 0 && idx >= 16) continue;
      if (nsub == 1 && e > 0 && q == 0) continue;
      if (mode == 4) {
        for (int c = 0; c < 8; c++) out[n++] = (uint16_t)cdesc_pack(4, 0, c >> 1, c & 1, e);
      } else if (mode == 5) {
        for (int c = 0; c < 4; c++) out[n++] = (uint16_t)cdesc_pack(5, 0, c, 0, e);
      } else {
        out[n++] = (uint16_t)cdesc_pack(mode, idx, 0, 0, e);
      }
    }
  }
  return n;
}

// Classification, the statistics scan and the candidates of one block by a
// whole wave (lane i scores shape i); writes the block's statistics except
// the mode (known once the block is packed).  Returns the packed class and
// count.
__device__ uint32_t stats_select_block(const uint32_t px[16], int lane, const Bc7Params &prm,
                                       uint16_t cd[kMaxCands], fh_bc7_block_stats *bs) {
  bool solid = true, transparent = true, opaque = true;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    solid = solid && px[i] == px[0];
    transparent = transparent && (px[i] >> 24) == 0;
    opaque = opaque && (px[i] >> 24) == 255;
  }
  // every field of the record is written once (the caller's buffer may hold
  // anything): estimates -1 unless set, unused shape entries 0
  if (lane < 8) bs->mode_error[lane] = -1.0;
  if (!opaque || solid || transparent) bs->three_shape[lane] = 0.0;
  if (solid || transparent) {
    bs->two_shape[lane] = 0.0;
    if (lane < 8) bs->mode_estimate[lane] = -1.0;
    if (lane == 0) {
      bs->path = solid ? 0 : 1;
      bs->num_two_shape = bs->num_three_shape = 0;
    }
    return sel_pack(solid ? 0 : 1, 0);
  }
  // mode 6: the whole block as one line, four index values, 7-bit
  // endpoints (Compressor.cpp:2046-2061); never one colour here
  double est6;
  {
    bool flat[1];
    uint32_t ea[1], eb[1];
    masked_subset_errors<1, 4, false>(px, 0u, 0u, 0xFEFEFEFEu, 0xFEFEFEFEu, flat, ea, eb);
    est6 = flat[0] ? 0.0 : 0.0001 + (double)ea[0];
  }
  double e1, e3;
  const double err2 = stats_shape<2>(px, lane, e1, e3);
  int brk2;
  const uint64_t log2 = stats_scan(err2, lane, brk2, bs->two_shape);
  const int s2 = 63 - __clzll((long long)log2);
  uint32_t modes = 0xFFu;
  int path = 3;
  if (brk2 < 64) {
    path = 2;
    modes = (1u << 1) | (1u << 3) | (1u << 7);
  }
  // UpdateErrorEstimate keeps the minimum over the scanned shapes
  const double est1 = wave_min(lane <= brk2 ? e1 : DBL_MAX);
  const double est3 = wave_min(lane <= brk2 ? e3 : DBL_MAX);
  int s3 = 0, nshapes = 1;
  uint64_t log3 = 0;
  double est0 = -1.0, est2 = -1.0;
  if (opaque) {
    // runs even when the two-subset scan stopped early
    double e0, e2;
    const double err3 = stats_shape<3>(px, lane, e0, e2);
    int brk3;
    log3 = stats_scan(err3, lane, brk3, bs->three_shape);
    s3 = 63 - __clzll((long long)log3);
    nshapes = 2;
    if (brk3 < 64) {
      path = 2;
      modes = (1u << 0) | (1u << 2);
    }
    est0 = wave_min(lane <= brk3 ? e0 : DBL_MAX);
    est2 = wave_min(lane <= brk3 ? e2 : DBL_MAX);
  }
  if (lane < 8) {
    // modes 4, 5 and 7 get no estimate on this path
    const double est = lane == 0 ? est0 : lane == 1 ? est1 : lane == 2 ? est2
                     : lane == 3 ? est3 : lane == 6 ? est6 : -1.0;
    bs->mode_estimate[lane] = est;
  }
  if (lane == 0) {
    bs->path = path;
    bs->num_two_shape = (uint32_t)__popcll(log2);
    bs->num_three_shape = (uint32_t)__popcll(log3);
  }
  const int count = stats_candidates(nshapes, s2, s3, modes & prm.block_modes, prm.quality, cd);
  return sel_pack(2, count);
}

// The candidates of a caller's ShapeSelection (CompressionSettings::
// m_ShapeSelectionFn, Compressor.cpp:1840-1858) in CompressClusters' order
// (:1752-1809): the first min(5, num_shapes) entries, or one entry and no
// multi-subset mode when there are none.  As in the statistics search, a
// single-subset mode's entries after the first are left out without
// annealing.  At most 31 slots (the host checks every selection first).
__device__ int given_candidates(const fh_shape_selection &g, uint32_t block_modes, uint32_t q,
                                uint16_t out[kMaxCands]) {
  constexpr int kOrder[8] = {0, 2, 1, 3, 7, 4, 5, 6};
  uint32_t modes = g.selected_modes & block_modes;
  int nsh = g.num_shapes < 5 ? (int)g.num_shapes : 5;
  if (nsh == 0) {
    nsh = 1;
    modes &= ~((1u << 0) | (1u << 1) | (1u << 2) | (1u << 3) | (1u << 7));
  }
  int n = 0;
  auto emit = [&](uint32_t d) {
    if (n < kMaxCands - 1) out[n++] = (uint16_t)d;
  };
#pragma unroll
  for (int mi = 0; mi < 8; mi++) {
    const int mode = kOrder[mi];
    if (!((modes >> mode) & 1)) continue;
    for (int e = 0; e < nsh; e++) {
      const uint32_t parts = g.shapes[e].num_partitions, idx = g.shapes[e].index & 63u;
      const int nsub = kModes[mode].subsets;
      if (nsub != 1 && (uint32_t)nsub != parts) continue;
      if (mode == 0 && g.shapes[e].index >= 16) continue;
      if (nsub == 1 && e > 0 && q == 0) continue;
      if (mode == 4) {
        for (int c = 0; c < 8; c++) emit(cdesc_pack(4, 0, c >> 1, c & 1, e));
      } else if (mode == 5) {
        for (int c = 0; c < 4; c++) emit(cdesc_pack(5, 0, c, 0, e));
      } else {
        emit(cdesc_pack(mode, (int)idx, 0, 0, e));
      }
    }
  }
  return n;
}

// Classification and a caller's selection of one block (solid and
// transparent blocks never reach the selection function).
__device__ uint32_t given_select_block(const uint32_t px[16], const Bc7Params &prm,
                                       const fh_shape_selection &g, uint16_t cd[kMaxCands]) {
  bool solid = true, transparent = true;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    solid = solid && px[i] == px[0];
    transparent = transparent && (px[i] >> 24) == 0;
  }
  if (solid || transparent) return sel_pack(solid ? 0 : 1, 0);
  return sel_pack(2, given_candidates(g, prm.block_modes, prm.quality, cd));
}

// Kernel 1: one workgroup of four waves selects 16 blocks, each wave four
// in turn; the workgroup's candidates go to the type queues with one global
// atomic per type.  list, if given, holds the blocks to select (list_count
// of them, a device word); otherwise all blocks of the range.
// SEL: which selection (BoxSelection, the statistics scan, the caller's).
enum { kSelBox = 0, kSelStats = 1, kSelGiven = 2 };

template <int SEL, bool NU = false>
__global__ void __launch_bounds__(256) select_kernel(BlockRange r, Bc7Params prm, Work w,
                                                     const uint32_t *list,
                                                     const uint32_t *list_count) {
  constexpr int kSlots = SEL == kSelBox ? kMaxBoxCands : kMaxCands;
  __shared__ uint32_t s_px[16][16];
  __shared__ uint32_t s_sel[16];
  __shared__ uint16_t s_cd[16][kSlots];
  __shared__ uint32_t s_cnt[kNumTypes], s_base[kNumTypes];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t base = blockIdx.x * 16;  // position in the list or the range
  const uint32_t total = list ? *list_count : r.num_blocks;
  if (base >= total) return;  // whole workgroup
  auto rel_of = [&](uint32_t i) { return list ? list[i] : i; };
  {
    const int blk = tid >> 4, p = tid & 15;
    const uint32_t i = base + blk;
    if (i < total) {
      const uint32_t rel = rel_of(i);
      const uint32_t b = r.first_block + rel;
      const uint32_t bx = b % r.blocks_wide, by = b / r.blocks_wide;
      s_px[blk][p] = r.img[(size_t)(by * 4 + (p >> 2)) * r.width + bx * 4 + (p & 3)];
    }
  }
  __syncthreads();
  for (int k = 0; k < 4; k++) {
    const int blk = wave * 4 + k;
    if (base + blk >= total) break;  // uniform in the wave
    const uint32_t rel = rel_of(base + blk);
    uint32_t px[16];
#pragma unroll
    for (int i = 0; i < 16; i++) px[i] = s_px[blk][i];
    uint16_t cd[kSlots];
    uint32_t sel = SEL == kSelStats ? stats_select_block(px, lane, prm, cd, prm.stats + rel)
                 : SEL == kSelGiven ? given_select_block(px, prm, prm.selections[rel], cd)
                                    : box_select_block<NU>(px, lane, prm, cd);
    // the learned search's low-confidence blocks (the fallback list) run the
    // full search
    if (list && sel_cls(sel) == 2) sel |= kSelFull;
    const int count = sel_count(sel);
    if (lane == 0) {
      s_sel[blk] = sel;
      w.sel[rel] = sel;
    }
    // slot c of this block's descriptors goes out from lane c
    if (lane < count) w.cdesc[(size_t)rel * kMaxCands + lane] = cd[lane];
    if (lane < kSlots) s_cd[blk][lane] = lane < count ? cd[lane] : (uint16_t)0;
  }
  __syncthreads();
  // enqueue: thread = (block, candidate slot), 16 slots per round
#pragma unroll
  for (int half = 0; half < kSlots / 16; half++) {
    const int blk = tid >> 4, c = (tid & 15) + 16 * half;
    bool valid = false;
    int type = 0;
    uint32_t rel = 0;
    if (base + blk < total && c < sel_count(s_sel[blk])) {
      // mode 6's second shape entry has the same quality-0 fit as the first
      // (its slot follows it): the set-up of the first writes both
      const uint32_t d = s_cd[blk][c];
      valid = !((d & 7) == 6 && ((d >> 12) & 7) == 1);
      rel = rel_of(base + blk);
      type = kTypeOfMode[d & 7];
    }
    wg_enqueue(w, valid, type, cand_id(rel, (uint32_t)c), s_cnt, s_base);
  }
}

// The mode of each written block (the lowest set bit of its first byte; 8
// for the reserved encoding) into its statistics.
__global__ void __launch_bounds__(256) stats_mode_kernel(BlockRange r, fh_bc7_block_stats *stats) {
  const uint32_t rel = blockIdx.x * 256 + threadIdx.x;
  if (rel >= r.num_blocks) return;
  const uint32_t b0 = r.out[(size_t)(r.first_block + rel) * 16];
  stats[rel].mode = b0 ? __ffs(b0) - 1 : 8;
}

// ---------------------------------------------------------------------------
// Kernel 1b (learned candidate pruning).  The ranker gives each block 512
// logits, logit = mode * 64 + slot; these name the real candidates among
// them and the candidate each one stands for.
// ---------------------------------------------------------------------------
__device__ __forceinline__ bool logit_real(int j) {
  const int mode = j >> 6, slot = j & 63;
  switch (mode) {
    case 0: return slot < 16;
    case 4: return slot < 8;
    case 5: return slot < 4;
    case 6: return slot == 0;
    default: return true;
  }
}

__device__ __forceinline__ uint32_t cdesc_of_logit(int j) {
  const int mode = j >> 6, slot = j & 63;
  const int shape = kModes[mode].subsets > 1 ? slot : 0;
  const int rot = mode == 4 ? (slot >> 1) : (mode == 5 ? slot : 0);
  const int im = mode == 4 ? (slot & 1) : 0;
  return cdesc_pack(mode, shape, rot, im, 0);
}


// ---------------------------------------------------------------------------
// The learned search's ranking and selection in one kernel: a workgroup of
// four waves takes 64 blocks through the ranker (ranker_tile.h: logits
// bit-identical to the forward pass) and makes each block's decision from
// the fp32 logits staged in LDS, so they never reach HBM.  The output layer
// runs in four phases of 128 logits; the softmax is accumulated online over
// the phases (its total differs from a single sum by rounding only) and the
// top-k list is exact (largest logit first, the lower logit on ties).  Solid and transparent blocks are
// marked as the reference writes them, a confident block (top probability
// at least the threshold) keeps its top-k candidates, and the rest go on the
// fallback list for the full search.
// ---------------------------------------------------------------------------
// Strict order of the top-k list: the larger logit first, the lower logit
// index on ties.
// (Bitwise operators keep the comparisons free of branches.)
__device__ __forceinline__ bool top_before(float va, int ja, float vb, int jb) {
  return (va > vb) | ((va == vb) & (ja < jb));
}

// The same order as one unsigned 64-bit key: the logit's bits made
// monotone (-0 counted as +0, as the float comparisons do) above the
// complemented index, so a larger key comes first.
__device__ __forceinline__ uint64_t top_key(float v, int j) {
  const uint32_t u = __float_as_uint(v + 0.0f);
  const uint32_t o = u ^ ((uint32_t)((int32_t)u >> 31) | 0x80000000u);
  return ((uint64_t)o << 32) | (uint64_t)(0xFFFFFFFFu - (uint32_t)j);
}
__device__ __forceinline__ float key_value(uint64_t k) {
  const uint32_t o = (uint32_t)(k >> 32);
  return __uint_as_float(o ^ ((uint32_t)((int32_t)~o >> 31) | 0x80000000u));
}
__device__ __forceinline__ int key_index(uint64_t k) {
  return (int)(0xFFFFFFFFu - (uint32_t)k);
}

// Logits per mode that name a real candidate (logit_real).
__device__ __forceinline__ int real_logits(int mode) {
  return mode == 0 ? 16 : (mode == 4 ? 8 : (mode == 5 ? 4 : (mode == 6 ? 1 : 64)));
}

constexpr int kStageStride = 144;  // fp32 logits per staged row: 128 + 16, so that the
                                   // row-quad reads and the wave's writes avoid bank conflicts
static_assert(mlp::kRankRows * kStageStride * 4 <= mlp::kLdsH2, "staging over X and H1");

// Two workgroups per CU (their LDS fits twice): the bound holds the kernel to
// the registers that allows, so one workgroup's MFMA work overlaps the
// other's selection.
__global__ void __launch_bounds__(256, 2) rank_select_kernel(BlockRange r, Bc7Params prm, Work w,
                                                          const uint16_t *w1, const uint16_t *w2,
                                                          const uint16_t *w3,
                                                          const float *params,
                                                          uint32_t *fallback,
                                                          uint32_t *fallback_count) {
  __shared__ __align__(16) uint8_t lds[mlp::kLdsBytes];
  __shared__ uint32_t s_cnt[kNumTypes], s_base[kNumTypes];
  __shared__ uint32_t s_fb, s_fbbase;
  __shared__ uint16_t s_cd[mlp::kRankRows][8];
  __shared__ uint32_t s_count[mlp::kRankRows];
  __shared__ uint32_t s_fbslot[mlp::kRankRows];
  uint16_t *xs = reinterpret_cast<uint16_t *>(lds + mlp::kLdsX);
  uint16_t *h1 = reinterpret_cast<uint16_t *>(lds + mlp::kLdsH1);
  uint16_t *h2 = reinterpret_cast<uint16_t *>(lds + mlp::kLdsH2);
  float *stage = reinterpret_cast<float *>(lds);  // over X and H1 once layer 2 is done
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t n = r.num_blocks;
  const uint32_t tile0 = blockIdx.x * mlp::kRankRows;
  if (tid == 0) s_fb = 0;
  mlp::rank_features(r, n, tile0, tid, xs);
  __syncthreads();
  mlp::rank_hidden<64, mlp::kXs, 2>(xs, w1, params + mlp::kRankOffB1, wave * 64, lane, h1);
  __syncthreads();
  mlp::rank_hidden<256, mlp::kHs, 2>(h1, w2, params + mlp::kRankOffB2, wave * 64, lane, h2);
  __syncthreads();

  // Block srow's decision is made by its four threads (seg 0..3), which hold
  // the same running softmax (m, sum) and top-k list (lv, lj) throughout.
  const int srow = tid >> 2, seg = tid & 3;
  const int kk = prm.topk < 1 ? 1 : (prm.topk > 8 ? 8 : (int)prm.topk);
  const float *b3 = params + mlp::kRankOffB3;
  float m = -INFINITY, sum = 0.0f;
  // the list as keys; an empty entry is (-inf, 2^30)
  const uint64_t kFill = top_key(-INFINITY, 1 << 30);
  uint64_t lk[8];
#pragma unroll
  for (int i = 0; i < 8; i++) lk[i] = kFill;
  // the output layer in four phases of 128 logits (modes 2p and 2p + 1),
  // 32 per wave; each phase is staged in LDS and folded into the row state
#pragma unroll 1
  for (int p = 0; p < 4; p++) {
    mlp::floatx16 acc[2][1] = {};
    const int c0 = 128 * p + 32 * wave;
    mlp::rank_mma<256, mlp::kHs, 1>(h2, w3, c0, lane, acc);
    const float bias = b3[c0 + (lane & 31)];
    if (p > 0) __syncthreads();  // the previous phase's stage is read
#pragma unroll
    for (int rb = 0; rb < 2; rb++)
#pragma unroll
      for (int v = 0; v < 16; v++)
        stage[mlp::acc_row(rb, v, lane) * kStageStride + 32 * wave + (lane & 31)] =
            acc[rb][0][v] + bias;
    __syncthreads();
    // this thread's logits: 128 p + 16 i + 4 seg + e (i < 8, e < 4)
    float z[32];
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const float4 q =
          *reinterpret_cast<const float4 *>(stage + srow * kStageStride + 16 * i + 4 * seg);
      z[4 * i] = q.x;
      z[4 * i + 1] = q.y;
      z[4 * i + 2] = q.z;
      z[4 * i + 3] = q.w;
    }
    const int na = ((prm.block_modes >> (2 * p)) & 1) ? real_logits(2 * p) : 0;
    const int nb = ((prm.block_modes >> (2 * p + 1)) & 1) ? real_logits(2 * p + 1) : 0;
    // a logit that names no real candidate of an allowed mode drops out as
    // -inf: never the maximum, exp() = 0 in the sum, never in the top-k
#pragma unroll
    for (int k = 0; k < 32; k++) {
      const int slot = 16 * ((k >> 2) & 3) + 4 * seg + (k & 3);
      z[k] = slot < (k < 16 ? na : nb) ? z[k] : -INFINITY;
    }
    float pm = -INFINITY;
#pragma unroll
    for (int k = 0; k < 32; k++) pm = fmaxf(pm, z[k]);
    pm = fmaxf(pm, __shfl_xor(pm, 1));
    pm = fmaxf(pm, __shfl_xor(pm, 2));
    const float mn = fmaxf(m, pm);
    const float shift = mn > -INFINITY ? mn : 0.0f;
    // the hardware exponential (v_exp_f32 of x log2 e, relative error about
    // 2^-21): the top probability 1 / sum is a threshold test, and its
    // rounding (like that of the summation order) only matters for blocks
    // within about 1e-6 of the threshold
    float ps = 0.0f;
#pragma unroll
    for (int k = 0; k < 32; k++) ps += __expf(z[k] - shift);
    ps += __shfl_xor(ps, 1);
    ps += __shfl_xor(ps, 2);
    if (mn > -INFINITY) {  // the same in the row's four threads
      sum = (m > -INFINITY ? sum * __expf(m - mn) : 0.0f) + ps;
      m = mn;
    }
    // The list changes only if a logit of this phase beats its kk-th entry
    // (an equal one comes later in list order: its index is larger): when
    // no row of the wave has one, as in most waves in the mode-2/3 phase, the
    // merge below would rebuild the same list.
    uint64_t kthk = kFill;
#pragma unroll
    for (int i = 0; i < 8; i++) kthk = i == kk - 1 ? lk[i] : kthk;
    if (!__ballot(pm > key_value(kthk))) continue;
    // this phase's logits as keys (index 128 p + 16 i + 4 seg + e); a masked
    // one gets key 0, below every real key and the empty entry, so it is
    // never taken
    const int jbase = 128 * p + 4 * seg;
    uint64_t zk[32];
#pragma unroll
    for (int k = 0; k < 32; k++)
      zk[k] = z[k] > -INFINITY ? top_key(z[k], jbase + 16 * (k >> 2) + (k & 3)) : 0ull;
    // top-kk of the running list and this phase's logits: the t-th entry is
    // the largest key below entry t - 1's
    uint64_t nk[8];
#pragma unroll
    for (int i = 0; i < 8; i++) nk[i] = kFill;
    uint64_t pk = ~0ull;
#pragma unroll 1
    for (int t = 0; t < kk; t++) {
      uint64_t bk = kFill;
#pragma unroll
      for (int k = 0; k < 32; k++) {
        const bool take = (zk[k] < pk) & (zk[k] > bk);
        bk = take ? zk[k] : bk;
      }
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const bool take = (seg == 0) & (lk[i] < pk) & (lk[i] > bk);
        bk = take ? lk[i] : bk;
      }
#pragma unroll
      for (int off = 1; off < 4; off <<= 1) {
        const uint64_t ok = __shfl_xor(bk, off);
        bk = ok > bk ? ok : bk;
      }
#pragma unroll
      for (int i = 0; i < 8; i++) nk[i] = i == t ? bk : nk[i];
      pk = bk;
    }
#pragma unroll
    for (int i = 0; i < 8; i++) lk[i] = nk[i];
  }
  float lv[8];
  int lj[8];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    lv[i] = key_value(lk[i]);
    lj[i] = key_index(lk[i]);
  }

  // solid and transparent blocks, from the row's four texel rows
  const uint32_t rel = tile0 + (uint32_t)srow;
  uint4 px = make_uint4(0, 0, 0, 0);
  if (rel < n) {
    const uint32_t b = r.first_block + rel;
    const uint32_t bx = b % r.blocks_wide, by = b / r.blocks_wide;
    px = *reinterpret_cast<const uint4 *>(r.img + (size_t)(by * 4 + seg) * r.width + bx * 4);
  }
  const uint32_t p0 = __shfl(px.x, lane & ~3);
  uint32_t flags = ((px.x != p0 || px.y != p0 || px.z != p0 || px.w != p0) ? 1u : 0u) |
                   (((px.x | px.y | px.z | px.w) >> 24) ? 2u : 0u);
  flags |= __shfl_xor(flags, 1);
  flags |= __shfl_xor(flags, 2);
  uint32_t count = 0, fbslot = 0;
  if (seg == 0 && rel < n) {
    if (!(flags & 1u) || !(flags & 2u)) {
      w.sel[rel] = sel_pack((flags & 1u) ? 1 : 0, 0);  // solid, else transparent
    } else if (!(m > -INFINITY) || 1.0f / sum < prm.threshold) {
      // top probability = exp(0) / sum below the threshold: the full search
      fbslot = atomicAdd(&s_fb, 1u) + 1u;  // 1-based: 0 marks no fallback
    } else {
#pragma unroll
      for (int i = 0; i < 8; i++) {
        if (i < kk && lv[i] > -INFINITY) {
          const uint16_t d = (uint16_t)cdesc_of_logit(lj[i]);
          s_cd[srow][i] = d;
          w.cdesc[(size_t)rel * kMaxCands + i] = d;
          count++;
        }
      }
      w.sel[rel] = sel_pack(2, (int)count);
    }
  }
  if (seg == 0) {
    s_count[srow] = count;
    s_fbslot[srow] = fbslot;
  }
  __syncthreads();
  // fallback list: one global atomic per workgroup
  if (tid == 0 && s_fb) s_fbbase = atomicAdd(fallback_count, s_fb);
  __syncthreads();
  if (tid < mlp::kRankRows && s_fbslot[tid])
    fallback[s_fbbase + s_fbslot[tid] - 1u] = tile0 + (uint32_t)tid;
  // enqueue the confident blocks' candidates: 64 rows x 8 slots
  for (int u = 0; u < 2; u++) {
    const int item = 256 * u + tid;
    const int row = item >> 3, slot = item & 7;
    const bool valid = (uint32_t)slot < s_count[row];
    const int type = valid ? kTypeOfMode[s_cd[row][slot] & 7] : 0;
    wg_enqueue(w, valid, type, cand_id(tile0 + (uint32_t)row, (uint32_t)slot), s_cnt, s_base);
  }
}

// ---------------------------------------------------------------------------
// Kernel 2: candidate set-up, persistent over the type queues in order.
// ---------------------------------------------------------------------------
// One subset of a mode without rotation: its average, then its fit.  Returns
// its pixel count.
template <bool NU>
__device__ __forceinline__ int fit_subset(const Fit &f, uint32_t quality, const uint32_t *sctab,
                                          const uint32_t px[16], uint32_t smask, SubStart &ss,
                                          const Weights *mu, uint32_t *km) {
  const int n = __popc(smask);
  uint32_t sum02 = 0, sum13 = 0;
  bool same = true;
  uint32_t firstp = 0;
  bool have_first = false;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    if (!((smask >> i) & 1)) continue;
    if (!have_first) {
      firstp = px[i];
      have_first = true;
    }
    same = same && px[i] == firstp;
    sum02 += px[i] & 0x00FF00FFu;
    sum13 += (px[i] >> 8) & 0x00FF00FFu;
  }
  // integer sums over n in 1..16: the double product is the correctly
  // rounded quotient (as for the k-means means)
  float avg[4];
  avg[0] = (float)((double)(sum02 & 0xFFFFu) * kInvCount[n]);
  avg[1] = (float)((double)(sum13 & 0xFFFFu) * kInvCount[n]);
  avg[2] = (float)((double)(sum02 >> 16) * kInvCount[n]);
  avg[3] = (float)((double)(sum13 >> 16) * kInvCount[n]);
  subset_setup<NU>(f, quality, sctab, px, smask, 0, n, avg, same, ss, mu, mu, km);
  return n;
}

// Quality-0 fit of one candidate: every subset's endpoints, indices and
// error (CompressionMode::Compress, Compressor.cpp:1300-1371, without the
// annealing), the record the pack kernel reads, and the annealing start
// state.  Returns the mask of subsets that annealing continues (quality > 0).
// MODE >= 0 specialises the fit for that mode at compile time (k.mode must
// equal it); -1 reads the mode from k.
//
// NU: the nonuniform metric with unrotated weights *mu.  The subset errors
// are float bit patterns (a single-colour subset's is the per-pixel error,
// flagged in st.pbc bit 8 + subset, its error being n times it), the alpha
// term a double in st.extra_err / st.pad, and the candidate's total, the
// double sum the reference compares (Compressor.cpp:1300-1371), in *tot_nu.
template <int MODE, bool NU = false>
__device__ __forceinline__ uint32_t fit_candidate(const Cand &k, const uint32_t px[16],
                                                  uint32_t quality, const uint32_t *sctab,
                                                  CandRec &rec, AState &st, uint32_t &total,
                                                  const Weights *mu, double *tot_nu,
                                                  uint32_t *km) {
  Fit f;
  const ModeAttr attr = MODE >= 0 ? kModeTab[MODE < 0 ? 0 : MODE] : kModes[k.mode];
  const int nsub = attr.subsets;
  // a specialised mode without rotation or index-mode bits fixes both at
  // zero, so only its own index width's k-means is compiled
  const int rot = (MODE >= 0 && !attr.has_rot) ? 0 : k.rot;
  const int im = (MODE >= 0 && MODE != 4) ? 0 : k.im;
  set_fit_attr(f, attr, MODE >= 0 ? MODE : k.mode, rot, im);
  rec.err = 0;
  rec.px1[0] = rec.px1[1] = rec.px1[2] = 0;
  rec.px2[0] = rec.px2[1] = rec.px2[2] = 0;
  rec.aidx_lo = rec.aidx_hi = 0;
  st.extra_err = 0;
  st.pad = 0;
  uint32_t active = 0, pbcs = 0, scf = 0;
  total = 0;
  double tnu = 0.0;
  uint64_t cidx = 0;
  if (attr.has_rot) {
    uint64_t aidx;
    uint32_t a1q, a2q;
    Weights mr;
    double aerr_nu = 0.0;
    if constexpr (NU) mr = rotate_weights(*mu, rot);
    const uint32_t aerr = alpha_fit<NU>(f, px, aidx, a1q, a2q, km, NU ? mr.w[3] : 1.0f,
                                        &aerr_nu);
    // the RGB fit sees the stale statistics of the unrotated cluster
    float avg[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < 16; i++)
#pragma unroll
      for (int kk = 0; kk < 4; kk++) avg[kk] += (float)chan(px[i], kk);
#pragma unroll
    for (int kk = 0; kk < 4; kk++) avg[kk] = avg[kk] / 16.0f;
    SubStart s0;
    subset_setup<NU>(f, quality, sctab, px, 0xFFFFu, rot + 1, 16, avg, false, s0, mu, &mr, km);
    rec.aidx_lo = (uint32_t)aidx;
    rec.aidx_hi = (uint32_t)(aidx >> 32);
    // Pack writes the RGB of the fit and the fitted alpha, no p-bit
    rec.px1[0] = (to_pixel_int(s0.p1, f.qmask, -1) & 0x00FFFFFFu) | (a1q << 24);
    rec.px2[0] = (to_pixel_int(s0.p2, f.qmask, -1) & 0x00FFFFFFu) | (a2q << 24);
    st.p1[0] = s0.p1;
    st.p2[0] = s0.p2;
    st.err[0] = s0.err;
    st.extra_err = aerr;
    if constexpr (NU) {
      // rgbError + alphaError (Compressor.cpp:918)
      const double rgb = s0.sc ? 16.0 * (double)__uint_as_float(s0.err)
                               : (double)__uint_as_float(s0.err);
      tnu = rgb + aerr_nu;
      const uint64_t ab = (uint64_t)__double_as_longlong(aerr_nu);
      st.extra_err = (uint32_t)ab;
      st.pad = (uint32_t)(ab >> 32);
      scf = s0.sc ? 1u : 0u;
    }
    cidx = s0.idx;
    total = s0.err + aerr;
    active = s0.anneal ? 1u : 0u;
  } else {
#pragma unroll 1
    for (int s = 0; s < nsub; s++) {
      // keeps the texels' LDS reads inside the loop: hoisted, their channels
      // take 80 registers
      asm volatile("" ::: "memory");
      SubStart ss;
      const int n = fit_subset<NU>(f, quality, sctab, px, subset_mask(k.shape, nsub, s), ss, mu, km);
      if constexpr (NU) {
        tnu += ss.sc ? (double)n * (double)__uint_as_float(ss.err)
                     : (double)__uint_as_float(ss.err);
        scf |= (ss.sc ? 1u : 0u) << s;
      }
      const int pb0 = f.pbit_type == PB_NONE ? -1 : pbc_bit(f.pbit_type, ss.pbc, 0);
      const int pb1 = f.pbit_type == PB_NONE ? -1 : pbc_bit(f.pbit_type, ss.pbc, 1);
      const uint32_t e1 = to_pixel_int(ss.p1, f.qmask, pb0);
      const uint32_t e2 = to_pixel_int(ss.p2, f.qmask, pb1);
      if (s == 0) {
        rec.px1[0] = e1; rec.px2[0] = e2;
        st.p1[0] = ss.p1; st.p2[0] = ss.p2; st.err[0] = ss.err;
      } else if (s == 1) {
        rec.px1[1] = e1; rec.px2[1] = e2;
        st.p1[1] = ss.p1; st.p2[1] = ss.p2; st.err[1] = ss.err;
      } else {
        rec.px1[2] = e1; rec.px2[2] = e2;
        st.p1[2] = ss.p1; st.p2[2] = ss.p2; st.err[2] = ss.err;
      }
      pbcs |= (uint32_t)ss.pbc << (2 * s);
      cidx |= ss.idx;
      total += ss.err;
      if (ss.anneal) active |= 1u << s;
    }
  }
  rec.cidx_lo = (uint32_t)cidx;
  rec.cidx_hi = (uint32_t)(cidx >> 32);
  rec.meta = pbcs | ((uint32_t)rot << 8) | ((uint32_t)im << 10);
  rec.err = total;  // the quality-0 result; annealing overwrites active ones
  st.pbc = pbcs;
  if constexpr (NU) {
    st.pbc |= scf << 8;
    *tot_nu = tnu;
  }
  st.idx_lo = (uint32_t)cidx;
  st.idx_hi = (uint32_t)(cidx >> 32);
  return active;
}

// One launch per mode (its type queue), specialised at compile time so that
// each mode gets its own register allocation.
constexpr int kPxStride = 17;  // odd stride: lanes reading texel i hit distinct banks

// Index entries of the widest k-means a mode's set-up runs (the colour
// indices; mode 4 with index mode 1 has 3-bit colour indices).
constexpr int kSetupBuckets(int mode) {
  return mode == 6 ? 16 : ((mode == 0 || mode == 1 || mode == 4) ? 8 : 4);
}

// Runs the batches of the mode's queue from `first` on, `stride` apart: one
// lane each, or with several subsets one adjacent lane per subset (64
// candidates, or 32 or 21), whose fits run side by side.  (One lane for all
// subsets took their fits' time one after another: 155 us for a batch of
// mode 0.)  The batches cost alike, so the waves stride over them: fetching
// them from a counter cost small jobs an atomic per wave and mode, 2048 waves'
// 16 thousand of them on one cache line.  s_px: the lanes' texels; s_km: the k-means sums and counts, per
// bucket a row of 64 lanes each.
template <int MODE, bool NU>
__device__ __forceinline__ void setup_run(const BlockRange &r, const Bc7Params &prm,
                                          const Work &w, const uint32_t *sctab, uint32_t *s_px,
                                          uint32_t *s_km, uint32_t first, uint32_t stride) {
  constexpr int kTypeOf[8] = {0, 2, 1, 3, 6, 7, 5, 4};
  constexpr int t = kTypeOf[MODE], kSub = kModeTab[MODE].subsets, kBatch = 64 / kSub;
  const int lane = threadIdx.x, sub = lane % kSub, lead = lane - sub;
  const uint32_t count = w.counters[kCntQueue + t];
  // mode 4's states end below room for mode 5's whole queue
  const uint32_t top4 = w.astate_cap - 1u - w.counters[kCntQueue + kTypeOf[5]];
  for (uint32_t batch = first; batch < (count + kBatch - 1) / kBatch; batch += stride) {
    const uint32_t item = batch * kBatch + (uint32_t)(lane / kSub);
    const bool mine = lane < kBatch * kSub && item < count;
    const uint32_t id = mine ? w.queue[(size_t)t * w.qcap + item] : 0u;
    const uint32_t rel = id_block(id);
    const int c = (int)id_slot(id);
    Cand k;
    cand_from_desc(mine ? w.cdesc[(size_t)rel * kMaxCands + c] : (uint16_t)MODE, k);
    // the lane's texels live in LDS: the fit reads them many times, and
    // keeping them (and values derived from them) out of registers lets
    // the loops below stay rolled
    uint32_t *px = s_px + lane * kPxStride;
    if (mine) {
      uint32_t v[16];
      load_block(r, rel, v);
#pragma unroll
      for (int i = 0; i < 16; i++) px[i] = v[i];
    }
    Weights mu;
    if constexpr (NU) mu = params_weights(prm);
    CandRec *out = &w.rec[(size_t)rel * kMaxCands + c];
    if constexpr (kSub > 1) {
      Fit f;
      set_fit_attr(f, kModeTab[MODE], MODE, 0, 0);
      SubStart ss = {};
      int n = 0;
      if (mine)
        n = fit_subset<NU>(f, prm.quality, sctab, px, subset_mask(k.shape, kSub, sub), ss, &mu,
                           s_km + lane);
      const bool has_pb = f.pbit_type != PB_NONE;
      const uint32_t e1 =
          to_pixel_int(ss.p1, f.qmask, has_pb ? pbc_bit(f.pbit_type, ss.pbc, 0) : -1);
      const uint32_t e2 =
          to_pixel_int(ss.p2, f.qmask, has_pb ? pbc_bit(f.pbit_type, ss.pbc, 1) : -1);
      // the candidate's record from its subsets' lanes (every lane of the
      // wave takes part)
      const uint32_t bits = (uint32_t)ss.pbc | ((ss.anneal ? 1u : 0u) << 2) |
                            ((ss.sc ? 1u : 0u) << 3);
      const int nerr = ss.sc ? n : 1;
      const double terr = NU ? (double)nerr * (double)__uint_as_float(ss.err) : 0.0;
      uint32_t total = 0, pbcs = 0, active = 0, scf = 0, lo = 0, hi = 0;
      double tnu = 0.0;
#pragma unroll
      for (int s = 0; s < kSub; s++) {
        const int from = (lead + s) & 63;
        const uint32_t b = (uint32_t)__shfl((int)bits, from);
        total += (uint32_t)__shfl((int)ss.err, from);
        lo |= (uint32_t)__shfl((int)(uint32_t)ss.idx, from);
        hi |= (uint32_t)__shfl((int)(uint32_t)(ss.idx >> 32), from);
        pbcs |= (b & 3u) << (2 * s);
        active |= ((b >> 2) & 1u) << s;
        scf |= ((b >> 3) & 1u) << s;
        if constexpr (NU) tnu += __shfl(terr, from);
      }
      uint32_t slot = 0;
      if (mine && sub == 0 && active) slot = atomicAdd(&w.counters[kCntFront], 1u);
      slot = (uint32_t)__shfl((int)slot, lead);
      if (mine) {
        out->px1[sub] = e1;
        out->px2[sub] = e2;
        if (sub == 0) {
          if (kSub == 2) out->px1[2] = out->px2[2] = 0;
          out->err = total;  // the quality-0 result; annealing overwrites active ones
          out->cidx_lo = lo;
          out->cidx_hi = hi;
          out->aidx_lo = out->aidx_hi = 0;
          out->meta = pbcs;
          if constexpr (NU) w.nu_total[(size_t)rel * kMaxCands + c] = tnu;
        }
        if (active) {
          AState &st = w.astate[slot];
          st.p1[sub] = ss.p1;
          st.p2[sub] = ss.p2;
          st.err[sub] = ss.err;
          if (sub == 0) {
            st.id = id;
            st.info = (uint32_t)MODE | ((uint32_t)kSub << 6) | ((uint32_t)k.shape << 8) |
                      (active << 14) | ((uint32_t)k.entry << 17);
            st.pbc = pbcs | (NU ? scf << 8 : 0u);
            st.idx_lo = lo;
            st.idx_hi = hi;
            st.extra_err = 0;
            st.pad = 0;
            if (w.aid) w.aid[slot] = id;
          }
        }
      }
    } else if (mine) {
      CandRec rec;
      AState st = {};
      uint32_t total = 0;
      double tnu = 0.0;
      const uint32_t active = fit_candidate<MODE, NU>(k, px, prm.quality, sctab, rec, st, total,
                                                      &mu, &tnu, s_km + lane);
      st.id = id;
      *out = rec;
      if constexpr (NU) w.nu_total[(size_t)rel * kMaxCands + c] = tnu;
      // mode 6, shape entry 0 followed by entry 1 (opaque blocks with two
      // shapes): the second slot gets the same fit and its own annealing state
      bool twin = false;
      if (MODE == 6 && c + 1 < kMaxCands && c + 1 < sel_count(w.sel[rel])) {
        const uint32_t d1 = w.cdesc[(size_t)rel * kMaxCands + c + 1];
        twin = (d1 & 7) == 6 && ((d1 >> 12) & 7) == 1;
      }
      if (twin) {
        out[1] = rec;
        if constexpr (NU) w.nu_total[(size_t)rel * kMaxCands + c + 1] = tnu;
      }
      if (active) {
        st.info = (uint32_t)k.mode | ((uint32_t)k.rot << 3) | ((uint32_t)k.im << 5) |
                  ((uint32_t)k.nsub << 6) | ((uint32_t)k.shape << 8) | (active << 14) |
                  ((uint32_t)k.entry << 17);
        uint32_t slot;
        if (MODE == 5) slot = w.astate_cap - 1u - atomicAdd(&w.counters[kCntRot5], 1u);
        else if (MODE == 4)
          slot = top4 - atomicAdd(&w.counters[kCntRot4], 1u);
        else slot = atomicAdd(&w.counters[kCntFront], twin ? 2u : 1u);
        w.astate[slot] = st;
        if (w.aid) w.aid[slot] = id;
        if (twin) {
          st.id = id + 1;
          st.info |= 1u << 17;
          w.astate[slot + 1] = st;
          if (w.aid) w.aid[slot + 1] = id + 1;
        }
      }
    }
  }
}

// Waves of a mode's set-up that a CU holds: two per SIMD for mode 6, whose 16
// centroids take 64 registers, four for the modes with 4 buckets and two
// subsets or more, else three.
constexpr uint32_t setup_waves(int mode) {
  return mode == 6 ? 8u : (mode == 2 || mode == 3 || mode == 7 ? 16u : 12u);
}

template <int MODE, bool NU = false>
__global__ void __launch_bounds__(64)
    __attribute__((amdgpu_waves_per_eu(setup_waves(MODE) / 4)))
    setup_kernel(BlockRange r, Bc7Params prm, Work w, const uint32_t *sctab) {
  __shared__ uint32_t s_px[64 * kPxStride];
  __shared__ uint32_t s_km[kSetupBuckets(MODE) * 3 * 64];
  setup_run<MODE, NU>(r, prm, w, sctab, s_px, s_km, blockIdx.x, gridDim.x);
}

// Every mode in one launch, for jobs that leave the chip idle: a batch of fits
// takes 50 to 170 us whatever the job's size (one lane's serial fit), so
// eight launches in a row add up where one lets the modes run side by side.
// The annealing states come out in no order but the rotation modes' place.
template <bool NU>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2)))
setup_all_kernel(BlockRange r, Bc7Params prm, Work w,
                                                       const uint32_t *sctab) {
  __shared__ uint32_t s_px[64 * kPxStride];
  __shared__ uint32_t s_km[kSetupBuckets(6) * 3 * 64];
  // this wave's batches of the modes' batches one after another, the slowest
  // modes' first: each mode's starting where the last one's end left off
  uint32_t first = blockIdx.x;
  auto run = [&](auto mode) {
    constexpr int M = decltype(mode)::value;
    constexpr int kTypeOf[8] = {0, 2, 1, 3, 6, 7, 5, 4};
    constexpr uint32_t kBatch = 64 / kModeTab[M].subsets;
    setup_run<M, NU>(r, prm, w, sctab, s_px, s_km, first, gridDim.x);
    const uint32_t n = (w.counters[kCntQueue + kTypeOf[M]] + kBatch - 1) / kBatch % gridDim.x;
    first = first >= n ? first - n : first + gridDim.x - n;
  };
  run(std::integral_constant<int, 4>{});
  run(std::integral_constant<int, 5>{});
  run(std::integral_constant<int, 1>{});
  run(std::integral_constant<int, 0>{});
  run(std::integral_constant<int, 6>{});
  run(std::integral_constant<int, 2>{});
  run(std::integral_constant<int, 3>{});
  run(std::integral_constant<int, 7>{});
}

// ---------------------------------------------------------------------------
// Kernel 3: simulated annealing (OptimizeEndpointsForCluster,
// Compressor.cpp:583-624), persistent.  A lane owns one candidate and
// advances every still-annealing subset of it by one step per iteration; the
// 16 pixels are scored in one pass, each against its own subset's
// endpoints.  Finished lanes wait until kRefillLanes of the wave are idle and
// then take the next candidates together, from a wave-local window of the
// global list.
// ---------------------------------------------------------------------------
constexpr int kRowWords = 37;  // a lane's LDS row: 32 texel words, 4 of index bits, odd

// What a step needs of the candidate's mode, in one word:
//   colour step 5 bits | alpha step 5 << 5 | p-bit flip 2 << 10 |
//   first p-bit's shift 1 << 12 | no p-bits 1 << 13 |
//   colour and alpha rows of the quantisation table 3 << 14, 3 << 17 |
//   index bits 3 << 20
// The endpoints' p-bits are those of the combination c (GetPBitCombo,
// CompressionMode.h:243-250): (c >> shift) & 1 and c & 1; the next
// combination tried is c ^ flip.
__device__ __forceinline__ uint32_t step_cfg_pack(const Fit &f) {
  const bool has_pb = f.pbit_type != PB_NONE;
  const uint32_t cs = 1u << (8 - f.color_prec);
  // the opaque modes' alpha (channel 3) stays
  const uint32_t as = f.mode < 4 ? 0u : 1u << (8 - f.alpha_prec);
  const uint32_t flip = f.pbit_type == PB_SHARED ? 1u : (has_pb ? 3u : 0u);
  const uint32_t qa = f.alpha_prec ? (uint32_t)f.alpha_prec - 3u : 0u;
  return cs | (as << 5) | (flip << 10) | ((f.pbit_type == PB_NOTSHARED ? 1u : 0u) << 12) |
         ((has_pb ? 0u : 1u) << 13) | (((uint32_t)f.color_prec - 3u) << 14) | (qa << 17) |
         ((uint32_t)f.nbits_idx << 20);
}

struct StepCfg {
  uint32_t s02, s13, k2_02, k2_13, flip, sh, nopb, qc, qa;
  float kf;
  WeightFn wf;
};

__device__ __forceinline__ StepCfg step_cfg(uint32_t c) {
  StepCfg k;
  const uint32_t cs = c & 31u, as = (c >> 5) & 31u;
  k.flip = (c >> 10) & 3u;
  k.sh = (c >> 12) & 1u;
  k.nopb = (c >> 13) & 1u;
  k.s02 = cs | (cs << 16);
  k.s13 = cs | (as << 16);
  k.k2_02 = k.s02 << k.nopb;
  k.k2_13 = k.s13 << k.nopb;
  k.qc = ((c >> 14) & 7u) << 9;
  k.qa = ((c >> 17) & 7u) << 9;
  const int nb = 1 << ((c >> 20) & 7u);
  k.kf = (float)(nb - 1);
  k.wf = weight_fn(nb);
  return k;
}

// The quantisation table's rows (kQuant) for the annealing's precisions (0,
// 4..8 bits) and p-bits, in LDS: row (bits ? bits - 3 : 0) * 2 + p-bit.
constexpr int kStepQuantBytes = 6 * 2 * 256;
__device__ __forceinline__ void step_quant_load(uint8_t *lds) {
  uint32_t *dst = reinterpret_cast<uint32_t *>(lds);
  for (int t = threadIdx.x; t < kStepQuantBytes / 4; t += blockDim.x) {
    const int row = t >> 6, bits = row < 2 ? 0 : (row >> 1) + 3, pb = row & 1;
    dst[t] = reinterpret_cast<const uint32_t *>(kQuant)[(bits * 3 + pb + 1) * 64 + (t & 63)];
  }
}
// An endpoint quantised with its p-bit (ToPixel).
__device__ __forceinline__ uint32_t step_quant(const uint8_t *lds, const StepCfg &k, uint32_t p,
                                               uint32_t pbit) {
  const uint8_t *c = lds + (k.qc + (pbit << 8)), *a = lds + (k.qa + (pbit << 8));
  return (uint32_t)c[chan(p, 0)] | ((uint32_t)c[chan(p, 1)] << 8) |
         ((uint32_t)c[chan(p, 2)] << 16) | ((uint32_t)a[chan(p, 3)] << 24);
}

// The reference's acceptance expression.  A call, not inlined: inlined, the
// exponential's constants are hoisted out of the annealing loop and cost it
// some 20 registers for a branch that is hardly ever taken.
__device__ __attribute__((noinline)) bool accept_exact(float rr, float cf, float ef, int q,
                                                       int energy) {
  const float temp = (float)energy / (float)(q - 1);
  return (double)rr < exp(((double)0.1f * ((double)cf - (double)ef)) / (double)temp);
}

// AcceptNewEndpointError (Compressor.cpp:524-536) for err >= cur: accept when
// frand() < exp(0.1 (cur - err) / temp), temp = energy / (q - 1).  The
// probability is at most 1, so a draw rr in [1, 3) never accepts.
//
// A single-precision estimate of the probability decides unless rr lies
// within 1e-4 (relative) of it, which covers the estimate's error (the
// hardware reciprocal and exponential are within a few 2^-23 of theirs, and
// where the exponent is large enough to magnify its own rounding past the
// margin the probability is below every nonzero draw, 2^-16 at least); then
// the double expression of the reference decides.  The uniform metric's
// errors are integers below 2^24, so their float difference is exact; the
// nonuniform metric's are floats, whose difference has a relative error of at
// most 2^-23 where it is not exact, well inside the margin.  At energy 0 and
// equal errors both forms are NaN, which never accepts.
__device__ __forceinline__ bool accept_worse(float rr, float cf, float ef, int q, int energy) {
  const float pf =
      __expf(0.1f * (cf - ef) * ((float)(q - 1) * __builtin_amdgcn_rcpf((float)energy)));
  const bool low = rr < pf * 0.9999f, high = rr > pf * 1.0001f;
  bool accept = (rr != 0.0f) & low & (rr < 1.0f);
  if ((rr < 1.0f) & ((rr == 0.0f) | !(low | high))) {
    accept = accept_exact(rr, cf, ef, q, energy);
  }
  return accept;
}

// One subset's annealing state.
struct SubState {
  uint32_t p1, p2, bp1, bp2, cur, best, cpbc, bpbc, x;  // x: its random stream (Rng)
  int energy;
};

// PickBestNeighboringEndpoints (Compressor.cpp:426-498) on integer endpoints.
// A channel's bit of the draw chooses its direction: without p-bits +step or
// -step; with them the p-bits flip, and an endpoint whose p-bit was 0 moves
// by -step or 0, one whose p-bit was 1 by 0 or +step.  Up to 16 draws while
// the neighbour is the best state itself (`live` lanes only); every lane of
// the wave takes part.
__device__ __forceinline__ void pick_neighbor(const StepCfg &k, bool live, SubState &t,
                                              uint32_t &np1, uint32_t &np2, uint32_t &npbc) {
  npbc = t.cpbc ^ k.flip;
  const uint32_t up2 = ((t.cpbc >> k.sh) & 1u) | k.nopb, up1 = (t.cpbc & 1u) | k.nopb;
  auto draw = [&]() {
    // endpoint 2's draw comes first
    Rng rng;
    rng.x = t.x;
    np2 = step_endpoint(t.p2, rng.next(), as_s16x2(up2 ? k.s02 : 0u),
                        as_s16x2(up2 ? k.s13 : 0u), as_s16x2(k.k2_02), as_s16x2(k.k2_13));
    np1 = step_endpoint(t.p1, rng.next(), as_s16x2(up1 ? k.s02 : 0u),
                        as_s16x2(up1 ? k.s13 : 0u), as_s16x2(k.k2_02), as_s16x2(k.k2_13));
    t.x = rng.x;
  };
  draw();
  bool again = live & (np1 == t.bp1) & (np2 == t.bp2) & (npbc == t.bpbc);
  for (int tries = 1; __ballot(again) && tries < 16; tries++) {
    if (again) {
      draw();
      again = (np1 == t.bp1) & (np2 == t.bp2);
    }
  }
}

// The rest of a step, once the neighbour's error is known: acceptance and
// the best state (Compressor.cpp:590-624).  Returns whether the best state
// was replaced, and in `accept` whether the neighbour was taken; live becomes
// false when the subset has finished.
template <bool NU = false>
__device__ __forceinline__ bool finish_step(SubState &t, bool &live, uint32_t err, uint32_t np1,
                                            uint32_t np2, uint32_t npbc, int q, bool &accept) {
  // the acceptance draw, made only where the error is not below cur
  Rng rng;
  rng.x = t.x;
  const float rr = rng.frand();
  const bool lower = err < t.cur;
  accept = live & (lower | accept_worse(rr, NU ? __uint_as_float(t.cur) : (float)t.cur,
                                        NU ? __uint_as_float(err) : (float)err, q, t.energy));
  t.x = lower ? t.x : rng.x;
  t.cur = accept ? err : t.cur;
  t.p1 = accept ? np1 : t.p1;
  t.p2 = accept ? np2 : t.p2;
  t.cpbc = accept ? npbc : t.cpbc;
  const bool better = live & (err < t.best);
  t.best = better ? err : t.best;
  t.bp1 = better ? np1 : t.bp1;
  t.bp2 = better ? np2 : t.bp2;
  t.bpbc = better ? npbc : t.bpbc;
  t.energy = better ? 1 : t.energy + 1;
  live = live & (t.best > 0) & (t.energy < q);
  return better;
}

struct Lane {
  bool has;
  uint32_t id, info;   // AState's
  uint32_t cfg;        // step_cfg_pack
  int nsub;
  uint32_t m12;        // masks of the pixels of subsets 1 and 2 (<< 16)
  int ptmode;
  uint32_t sel02, sel13;  // rotation_selectors(ptmode)
  uint32_t *px;        // this lane's row of LDS: the 16 texels (64 times their pairs
                       // 02 and 13), then the index bits of subsets 1 and 2
  uint32_t active;     // subsets still annealing
  SubState t0, t1, t2; // per subset
  uint64_t idx;        // indices of all subsets (best so far)
  uint32_t extra;
  // nonuniform metric: the candidate's weights (its rotation applied), the
  // single-colour subsets (their error is n times the stored one) and the
  // alpha term
  Weights m;
  uint32_t scf;
  double extra_nu;
};

// The low 8 bits of m as a mask of nibbles.
__device__ __forceinline__ uint32_t nibble_mask(uint32_t m) {
  uint32_t x = m & 0xFFu;
  x = (x | (x << 12)) & 0x000F000Fu;
  x = (x | (x << 6)) & 0x03030303u;
  x = (x | (x << 3)) & 0x11111111u;
  return (x << 4) - x;
}

template <bool NU = false>
__device__ __forceinline__ void lane_load(Lane &L, const BlockRange &r, const Bc7Params &prm, const AState &st) {
  L.has = true;
  L.id = st.id;
  L.info = st.info;
  const int mode = st.info & 7, rot = (st.info >> 3) & 3, im = (st.info >> 5) & 1;
  const int shape = (st.info >> 8) & 63, entry = (st.info >> 17) & 7;
  L.nsub = (st.info >> 6) & 3;
  L.active = (st.info >> 14) & 7;
  Fit f;
  set_fit(f, mode, rot, im);
  L.cfg = step_cfg_pack(f);
  L.ptmode = kModes[mode].has_rot ? rot + 1 : 0;
  rotation_selectors(L.ptmode, L.sel02, L.sel13);
  L.m12 = 0;
#pragma unroll
  for (int s = 1; s < 3; s++) {
    const uint32_t m = s < L.nsub ? subset_mask(shape, L.nsub, s) : 0u;
    L.m12 |= m << (16 * (s - 1));
    L.px[32 + 2 * (s - 1)] = nibble_mask(m);
    L.px[33 + 2 * (s - 1)] = nibble_mask(m >> 8);
  }
  {
    uint32_t v[16];
    load_block(r, id_block(st.id), v);
#pragma unroll
    for (int i = 0; i < 16; i++) {
      L.px[2 * i] = pair02x64(v[i]);
      L.px[2 * i + 1] = pair13x64(v[i]);
    }
  }
  const uint64_t bid = prm.block_id_base + r.first_block + id_block(st.id);
  auto start = [&](SubState &t, int s) {
    t.p1 = t.bp1 = st.p1[s];
    t.p2 = t.bp2 = st.p2[s];
    t.cur = t.best = st.err[s];
    t.cpbc = t.bpbc = (st.pbc >> (2 * s)) & 3u;
    t.energy = 0;
    t.x = fit_key(prm.seed, bid, cand_tag(mode, entry, s, rot, im));
  };
  start(L.t0, 0);
  start(L.t1, 1);
  start(L.t2, 2);
  L.idx = (uint64_t)st.idx_lo | ((uint64_t)st.idx_hi << 32);
  L.extra = st.extra_err;
  if constexpr (NU) {
    L.m = rotate_weights(params_weights(prm), rot);
    L.scf = (st.pbc >> 8) & 7u;
    L.extra_nu = __longlong_as_double((long long)((uint64_t)st.extra_err |
                                                  ((uint64_t)st.pad << 32)));
  }
}

// The constants of pixel i: those of its subset (NSUB = 1 takes sc0).
// ROT: whether a lane of the wave holds a rotation mode; without one every
// axis is the endpoint difference itself, which saves the two selects.
template <int NSUB, bool ROT>
__device__ __forceinline__ SubConst pixel_const(bool in1, bool in2, const SubConst &sc0,
                                                const SubConst &sc1, const SubConst &sc2) {
  SubConst c = sc0;
  if (NSUB > 1) c = pick_sub(in1, sc1, c);
  if (NSUB > 2) c = pick_sub(in2, sc2, c);
  if (NSUB > 1 && !ROT) {
    c.q02 = c.d02;
    c.q13 = c.d13;
  }
  return c;
}

// The 16-pixel pass for up to NSUB subsets: errors per subset and the
// indices.  Every pixel is scored; errors of subsets that have stopped
// annealing are not used.
template <int NSUB, bool ROT>
__device__ __forceinline__ void score_pixels(const Lane &L, const SubConst &sc0,
                                             const SubConst &sc1, const SubConst &sc2, float kf,
                                             WeightFn wf, uint32_t &n0, uint32_t &n1,
                                             uint32_t &n2, uint64_t &nidx) {
  uint32_t all = 0, lo = 0, hi = 0;
  n1 = n2 = 0;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const bool in1 = NSUB > 1 && (L.m12 & (1u << i)) != 0;
    const bool in2 = NSUB > 2 && (L.m12 & (1u << (16 + i))) != 0;
    const SubConst c = pixel_const<NSUB, ROT>(in1, in2, sc0, sc1, sc2);
    uint32_t best;
    const uint32_t me = pixel_err(L.px[2 * i], L.px[2 * i + 1], c, kf, wf, &best);
    all += me;
    if (NSUB > 1) n1 += in1 ? me : 0u;
    if (NSUB > 2) n2 += in2 ? me : 0u;
    if (i < 8) lo |= best << (4 * i);
    else hi |= best << (4 * (i - 8));
  }
  n0 = all - n1 - n2;
  nidx = (uint64_t)lo | ((uint64_t)hi << 32);
}

// The pixel pass under the nonuniform metric: float errors, each subset's
// summed in pixel order (adding 0 to the other subsets' sums leaves them
// unchanged).
template <int NSUB, bool ROT>
__device__ __forceinline__ void score_pixels_nu(const Lane &L, const SubConst &sc0,
                                                const SubConst &sc1, const SubConst &sc2,
                                                float kf, WeightFn wf, float &n0, float &n1,
                                                float &n2, uint64_t &nidx) {
  uint32_t lo = 0, hi = 0;
  n0 = n1 = n2 = 0.0f;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const bool in1 = NSUB > 1 && (L.m12 & (1u << i)) != 0;
    const bool in2 = NSUB > 2 && (L.m12 & (1u << (16 + i))) != 0;
    const SubConst c = pixel_const<NSUB, ROT>(in1, in2, sc0, sc1, sc2);
    uint32_t best;
    const float me = pixel_err_nu(L.px[2 * i], L.px[2 * i + 1], c, kf, wf, L.m, &best);
    n0 += in1 || in2 ? 0.0f : me;
    if (NSUB > 1) n1 += in1 ? me : 0.0f;
    if (NSUB > 2) n2 += in2 ? me : 0.0f;
    if (i < 8) lo |= best << (4 * i);
    else hi |= best << (4 * (i - 8));
  }
  nidx = (uint64_t)lo | ((uint64_t)hi << 32);
}

// One annealing step of every active subset, for waves whose running
// candidates have at most NSUB subsets.  Every lane of the wave takes part.
template <int NSUB, bool ROT, bool NU>
__device__ __forceinline__ void lane_step_n(Lane &L, const uint8_t *quant, int q) {
  const StepCfg k = step_cfg(L.cfg);
  struct Next {
    uint32_t p1 = 0, p2 = 0, pbc = 0, err = 0;
  } n0, n1, n2;
  auto propose = [&](SubState &t, int s, Next &n) {
    pick_neighbor(k, (L.active >> s) & 1u, t, n.p1, n.p2, n.pbc);
    return sub_const(step_quant(quant, k, n.p1, (n.pbc >> k.sh) & 1u),
                     step_quant(quant, k, n.p2, n.pbc & 1u));
  };
  SubConst sc0 = propose(L.t0, 0, n0), sc1 = sc0, sc2 = sc0;
  if (ROT) rotate_axis(sc0, L.ptmode, L.sel02, L.sel13);
  if (NSUB > 1) sc1 = propose(L.t1, 1, n1);
  if (NSUB > 2) sc2 = propose(L.t2, 2, n2);
  uint64_t nidx;
  if constexpr (NU) {
    float e0, e1, e2;
    score_pixels_nu<NSUB, ROT>(L, sc0, sc1, sc2, k.kf, k.wf, e0, e1, e2, nidx);
    n0.err = __float_as_uint(e0);
    n1.err = __float_as_uint(e1);
    n2.err = __float_as_uint(e2);
  } else {
    score_pixels<NSUB, ROT>(L, sc0, sc1, sc2, k.kf, k.wf, n0.err, n1.err, n2.err, nidx);
  }
  // index bits of the subsets whose best state is replaced
  const uint64_t m1 = NSUB > 1 ? (uint64_t)L.px[32] | ((uint64_t)L.px[33] << 32) : 0;
  const uint64_t m2 = NSUB > 2 ? (uint64_t)L.px[34] | ((uint64_t)L.px[35] << 32) : 0;
  uint64_t taken = 0;
  auto finish = [&](SubState &t, int s, const Next &n, uint64_t mine) {
    bool live = (L.active >> s) & 1u;
    const uint32_t was = live ? 1u << s : 0u;
    bool accept;
    const bool better = finish_step<NU>(t, live, n.err, n.p1, n.p2, n.pbc, q, accept);
    taken |= better ? mine : 0ull;
    if (!live) L.active &= ~was;
  };
  finish(L.t0, 0, n0, ~(m1 | m2));
  if (NSUB > 1) finish(L.t1, 1, n1, m1);
  if (NSUB > 2) finish(L.t2, 2, n2, m2);
  L.idx = (L.idx & ~taken) | (nidx & taken);
}

// The widest subset count among the wave's running lanes picks the compiled
// step (a wave-uniform branch): the list is ordered by mode, so most waves
// hold candidates of one subset count.  (Under the nonuniform metric, whose
// steps are mostly the rotation modes', annealing with the three-subset step
// alone takes 11.5 ms for 1024x1024 and 18.9 for 2048x2048; by count 8.8 and
// 14.5.)
template <bool NU>
__device__ __forceinline__ void lane_step(Lane &L, const uint8_t *quant, int q) {
  const bool run = L.active != 0;
  if (!__ballot(run && L.nsub > 1)) lane_step_n<1, true, NU>(L, quant, q);
  else if (__ballot(run && L.ptmode != 0)) lane_step_n<3, true, NU>(L, quant, q);
  else if (__ballot(run && L.nsub == 3)) lane_step_n<3, false, NU>(L, quant, q);
  else lane_step_n<2, false, NU>(L, quant, q);
}

template <bool NU = false>
__device__ __forceinline__ void lane_finish(Lane &L, Work &w) {
  CandRec *rc = &w.rec[L.id];
  Fit f;
  set_fit(f, L.info & 7, (L.info >> 3) & 3, (L.info >> 5) & 1);
  uint32_t total = L.extra;
  // nonuniform metric: the reference's double total, subsets in order, then
  // the alpha term of a rotation mode (Compressor.cpp:918, 1300-1371)
  double tnu = 0.0;
  uint32_t pbcs = rc->meta & 0x3Fu;
  auto put = [&](const SubState &t, int s) {
    if (s >= L.nsub) return;
    total += t.best;
    if constexpr (NU) {
      double e = (double)__uint_as_float(t.best);
      if ((L.scf >> s) & 1) {
        const int n1 = __popc(L.m12 & 0xFFFFu), n2 = __popc(L.m12 >> 16);
        e = (double)(s == 0 ? 16 - n1 - n2 : (s == 1 ? n1 : n2)) * e;
      }
      tnu += e;
    }
    const int pb = (int)t.bpbc;
    const int pb0 = f.pbit_type == PB_NONE ? -1 : pbc_bit(f.pbit_type, pb, 0);
    const int pb1 = f.pbit_type == PB_NONE ? -1 : pbc_bit(f.pbit_type, pb, 1);
    uint32_t e1 = to_pixel_int(t.bp1, f.qmask, pb0);
    uint32_t e2 = to_pixel_int(t.bp2, f.qmask, pb1);
    if (L.ptmode) {
      e1 = (e1 & 0x00FFFFFFu) | (rc->px1[0] & 0xFF000000u);
      e2 = (e2 & 0x00FFFFFFu) | (rc->px2[0] & 0xFF000000u);
    }
    rc->px1[s] = e1;
    rc->px2[s] = e2;
    pbcs = (pbcs & ~(3u << (2 * s))) | ((uint32_t)pb << (2 * s));
  };
  put(L.t0, 0);
  put(L.t1, 1);
  put(L.t2, 2);
  rc->cidx_lo = (uint32_t)L.idx;
  rc->cidx_hi = (uint32_t)(L.idx >> 32);
  rc->meta = (rc->meta & ~0x3Fu) | pbcs | kMetaAnnealed;
  rc->err = total;
  if constexpr (NU) w.nu_total[L.id] = tnu + L.extra_nu;
}

// A candidate in the middle of its annealing, handed from the one-lane form
// to the one-lane-per-pixel form.
struct TailState {
  uint32_t id, info;  // info: AState's, with the subsets still annealing
  uint32_t extra, pbc;  // pbc: 2 bits per subset, current then (<< 6) best
  uint32_t p1[3], p2[3], bp1[3], bp2[3], cur[3], best[3], energy[3], x[3];
  uint32_t idx_lo, idx_hi;
  uint32_t pad[2];
};
static_assert(sizeof(TailState) == 128, "TailState");

__device__ __forceinline__ void lane_hand_over(const Lane &L, TailState &o) {
  o.id = L.id;
  o.info = (L.info & ~(7u << 14)) | (L.active << 14);
  o.extra = L.extra;
  uint32_t pbc = 0;
  auto put = [&](const SubState &t, int s) {
    o.p1[s] = t.p1;
    o.p2[s] = t.p2;
    o.bp1[s] = t.bp1;
    o.bp2[s] = t.bp2;
    o.cur[s] = t.cur;
    o.best[s] = t.best;
    o.energy[s] = (uint32_t)t.energy;
    o.x[s] = t.x;
    pbc |= (t.cpbc << (2 * s)) | (t.bpbc << (6 + 2 * s));
  };
  put(L.t0, 0);
  put(L.t1, 1);
  put(L.t2, 2);
  o.pbc = pbc;
  o.idx_lo = (uint32_t)L.idx;
  o.idx_hi = (uint32_t)(L.idx >> 32);
}

// Idle lanes of a wave at which it loads new candidates: loading and
// finishing cost a whole wave's issue however few lanes do it, idle lanes
// waste their share of every step.  Measured at 4096 x 4096: 4 lanes 28.1 ms
// (reference search) and 3.29 ms (learned), 8 28.5 and 3.31, 12 28.9 and 3.36,
// 16 29.4 and 3.39; looking after every step and loading at one idle lane:
// 33.8 and 4.0.
constexpr int kRefillLanes = 4;
// The wave mask of each group's first lane (lanes 0, g, 2g, ...).
constexpr uint64_t group_leaders(int g, int lane = 0) {
  return lane >= 64 ? 0ull : (1ull << lane) | group_leaders(g, lane + g);
}
static_assert(group_leaders(16) == 0x0001000100010001ull, "group leaders");

// Groups still running at which a wave of the four-lane form hands over.
constexpr int kHandGroups = 4;

// ---------------------------------------------------------------------------
// The same annealing with G lanes per candidate.  G = 16: a row of 16 lanes
// holds one candidate, a lane its own pixel and the state of its own subset
// only (every lane of a subset computes the same step), so a step is one
// pixel's work plus three row sums instead of sixteen pixels' work for up to
// three subsets: about a quarter of the instructions, and of the latency, of
// a step of the one-lane form.  A wave advances four candidates where the
// one-lane form advances 64, so per candidate a step costs about four times
// more issue: this form is for lists that leave the chip idle, where the
// longest chain sets the time.  G = 4: candidates of one subset only, four
// pixels a lane, between the two in both respects.
//
// Looking ahead (G = 16): a wave left with one or two candidates, or given no
// more (lists shorter than the waves), runs each with two or four rows.  A
// step that is rejected leaves the state as it was but for three draws of the
// random stream and the energy, so row k proposes and scores the k-th next
// step as if the ones before it were rejected, and the first row where
// something else happens (an acceptance, a repeated draw, the end) gives the
// next state.  Modes 4 and 5 accept one step in five and one in four, the
// others fewer than one in sixteen: four rows advance 2.8 and nearly 4 steps
// at once.  The subsets are chains of their own and may advance differently.
// ---------------------------------------------------------------------------
// Sum over the G lanes of a group (every lane of the wave active).
template <int G>
__device__ __forceinline__ uint32_t group_sum(uint32_t v) {
  if (G == 16) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xf, 0xf, true);  // row_ror:8
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x124, 0xf, 0xf, true);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x122, 0xf, 0xf, true);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x121, 0xf, 0xf, true);
  } else {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4e, 0xf, 0xf, true);  // quad 2,3,0,1
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xb1, 0xf, 0xf, true);  // quad 1,0,3,2
  }
  return v;
}

// Runs the candidates [begin, end) of a list, taken from its end through
// *fetch by `waves` waves, until none is left.  SRC: kFromList (the annealing states),
// kFromTail (the candidates handed over in `tail`) or kFromListHand (the
// annealing states; once they are used up a wave with few groups running
// hands them over through `tail` and returns).
// Called by whole waves.  COUNT: the work counters of anneal_kernel.
enum { kFromList = 0, kFromTail = 1, kFromListHand = 2 };

template <int G, int SRC, bool COUNT>
__device__ __forceinline__ void spread_run(const BlockRange &r, const Bc7Params &prm,
                                           const Work &w, TailState *tail, const uint8_t *quant,
                                           uint32_t begin, uint32_t end, uint32_t waves,
                                           uint32_t *fetch,
                                           unsigned long long &n_ref, unsigned long long &n_gpu) {
  static_assert(G == 16 || G == 4, "lanes per candidate");
  constexpr int P = 16 / G;  // pixels per lane
  constexpr bool kTail = SRC == kFromTail;
  constexpr uint64_t kLeaders = group_leaders(G);
  const StateMap sm = state_map(w);
  constexpr uint64_t kGroup = (1ull << G) - 1ull;
  const int lane = threadIdx.x & 63, m = lane & (G - 1);
  const int q = (int)prm.quality;
  const uint32_t total = end - begin;
  // the candidate (the same in the group) and its constants
  bool has = false;
  uint32_t id = 0, info = 0, extra = 0, sel02 = 0, sel13 = 0;
  int ptmode = 0, nsub = 1;
  StepCfg k = step_cfg(0);
  // this lane's pixels m * P .., their subset and that subset's state
  uint32_t p02[P] = {}, p13[P] = {}, sub = 0, bidx = 0;
  bool active = false;
  SubState t = {};
  bool exhausted = total == 0;
  // rows per candidate: 1, 2 or 4 (see above); lead: this lane's group of rows
  int rpc = G == 16 && total <= 2 * waves ? (total <= waves ? 4 : 2) : 1;
  int lead = lane & ~(G * rpc - 1);
  for (;;) {
    // idle groups take the next candidates, from the end of the list (the
    // rotation modes, whose chains are the longest, first)
    uint64_t leaders = kLeaders;
    if (G == 16 && rpc > 1) leaders = rpc == 2 ? group_leaders(32) : 1ull;
    uint64_t hasm = __ballot(has) & leaders;
    const uint64_t need = ~hasm & leaders;
    if (need && !exhausted) {
      const uint32_t want = (uint32_t)__popcll(need);
      uint32_t base = 0;
      if (lane == 0) base = atomicAdd(fetch, want);
      base = __shfl(base, 0);
      if (base >= total || total - base <= want) exhausted = true;
      const uint32_t item = base + (uint32_t)__popcll(need & ((1ull << lead) - 1ull));
      if (!has && item < total) {
        const uint32_t at = end - 1u - item;
        const TailState *ts = kTail ? tail + at : nullptr;
        const AState *st = kTail ? nullptr : w.astate + (w.alist ? w.alist[at] : sm.slot(at));
        has = true;
        id = kTail ? ts->id : st->id;
        info = kTail ? ts->info : st->info;
        extra = kTail ? ts->extra : st->extra_err;
        const int mode = info & 7, rot = (info >> 3) & 3, im = (info >> 5) & 1;
        const int shape = (info >> 8) & 63;
        Fit f;
        set_fit(f, mode, rot, im);
        k = step_cfg(step_cfg_pack(f));
        ptmode = kModes[mode].has_rot ? rot + 1 : 0;
        rotation_selectors(ptmode, sel02, sel13);
        if (G == 16) {
          nsub = (info >> 6) & 3;
          sub = 0;
          if (nsub == 2) sub = (kShape2[shape] >> m) & 1u;
          if (nsub == 3) sub = subset_of(kShape3[shape][0], kShape3[shape][1], m);
        }
        const uint32_t rel = id_block(id), b = r.first_block + rel;
        const uint32_t bx = b % r.blocks_wide, by = b / r.blocks_wide;
        const uint32_t *src =
            r.img + (size_t)(by * 4 + (m * P >> 2)) * r.width + bx * 4 + ((m * P) & 3);
#pragma unroll
        for (int i = 0; i < P; i++) {
          const uint32_t pix = src[i];
          p02[i] = pair02x64(pix);
          p13[i] = pair13x64(pix);
        }
        active = (info >> (14 + sub)) & 1u;
        const uint32_t pbc = kTail ? ts->pbc : st->pbc;
        t.p1 = kTail ? ts->p1[sub] : st->p1[sub];
        t.p2 = kTail ? ts->p2[sub] : st->p2[sub];
        t.bp1 = kTail ? ts->bp1[sub] : t.p1;
        t.bp2 = kTail ? ts->bp2[sub] : t.p2;
        t.cur = kTail ? ts->cur[sub] : st->err[sub];
        t.best = kTail ? ts->best[sub] : t.cur;
        t.cpbc = (pbc >> (2 * sub)) & 3u;
        t.bpbc = kTail ? (pbc >> (6 + 2 * sub)) & 3u : t.cpbc;
        t.energy = kTail ? (int)ts->energy[sub] : 0;
        t.x = kTail ? ts->x[sub]
                    : fit_key(prm.seed, prm.block_id_base + b,
                              cand_tag(mode, (int)((info >> 17) & 7), (int)sub, rot, im));
        const uint64_t idx = kTail ? (uint64_t)ts->idx_lo | ((uint64_t)ts->idx_hi << 32)
                                   : (uint64_t)st->idx_lo | ((uint64_t)st->idx_hi << 32);
        bidx = (uint32_t)(idx >> (4 * P * m)) & ((1u << (4 * P)) - 1u);
      }
      hasm = __ballot(has) & leaders;
    }
    if (!hasm) break;
    if (SRC == kFromListHand && exhausted && __popcll(hasm) <= kHandGroups) {
      uint32_t base = 0;
      if (lane == 0) base = atomicAdd(&w.counters[kCntTail], (uint32_t)__popcll(hasm));
      base = __shfl(base, 0);
      if (has) {
        TailState &o = tail[base + (uint32_t)__popcll(hasm & ((1ull << lead) - 1ull))];
        if (m == 0) {
          o.id = id;
          o.info = info;  // one subset, still active
          o.extra = extra;
          o.pbc = t.cpbc | (t.bpbc << 6);
          o.p1[0] = t.p1;
          o.p2[0] = t.p2;
          o.bp1[0] = t.bp1;
          o.bp2[0] = t.bp2;
          o.cur[0] = t.cur;
          o.best[0] = t.best;
          o.energy[0] = (uint32_t)t.energy;
          o.x[0] = t.x;
        }
        reinterpret_cast<uint16_t *>(&o.idx_lo)[m] = (uint16_t)bidx;
      }
      break;
    }
    if (G == 16 && rpc < 4 && exhausted) {
      // few candidates left: give each more rows
      const int n = __popcll(hasm);
      const int wide = n == 1 ? 4 : (n == 2 ? 2 : 1);
      if (wide > rpc) {
        rpc = wide;
        lead = lane & ~(G * rpc - 1);
        // the first or the last running group's lane of the same pixel
        const int first = __ffsll((unsigned long long)hasm) - 1;
        const int last = 63 - __clzll((long long)hasm);
        const int from = (lead == 0 ? first : last) + m;
        auto take = [&](auto &v) { v = __shfl(v, from); };
        take(id);
        take(info);
        take(extra);
        take(sel02);
        take(sel13);
        take(ptmode);
        take(nsub);
        take(k.s02);
        take(k.s13);
        take(k.k2_02);
        take(k.k2_13);
        take(k.flip);
        take(k.sh);
        take(k.nopb);
        take(k.qc);
        take(k.qa);
        take(k.kf);
        take(k.wf.m);
        take(k.wf.b);
        take(p02[0]);
        take(p13[0]);
        take(sub);
        take(bidx);
        take(t.p1);
        take(t.p2);
        take(t.bp1);
        take(t.bp2);
        take(t.cur);
        take(t.best);
        take(t.cpbc);
        take(t.bpbc);
        take(t.x);
        take(t.energy);
        active = __shfl(active ? 1 : 0, from) != 0;
        has = true;
      }
    }
    // stale in rows without a candidate: harmless
    const bool multi = G == 16 && __ballot(nsub > 1) != 0;
    // proposes a neighbour of v, scores it and finishes v's step; nidx: its
    // indices.  Returns finish_step's result.
    auto step = [&](SubState &v, bool &live, uint32_t &nidx, bool &accept, bool &again) {
      uint32_t np1, np2, npbc;
      const uint32_t x0 = v.x;
      pick_neighbor(k, live, v, np1, np2, npbc);
      again = v.x != x0 + 2u * kRngStep;
      SubConst sc = sub_const(step_quant(quant, k, np1, (npbc >> k.sh) & 1u),
                              step_quant(quant, k, np2, npbc & 1u));
      rotate_axis(sc, ptmode, sel02, sel13);
      uint32_t me = 0;
      nidx = 0;
#pragma unroll
      for (int i = 0; i < P; i++) {
        uint32_t j;
        me += pixel_err(p02[i], p13[i], sc, k.kf, k.wf, &j);
        nidx |= j << (4 * i);
      }
      // its subset's error
      uint32_t err = group_sum<G>(me);
      if (multi) {
        const uint32_t t1 = group_sum<G>(sub == 1 ? me : 0u);
        const uint32_t t2 = group_sum<G>(sub == 2 ? me : 0u);
        err = sub == 0 ? err - t1 - t2 : (sub == 1 ? t1 : t2);
      }
      return finish_step(v, live, err, np1, np2, npbc, q, accept);
    };
    if (G == 4 || rpc == 1) {
      for (int u = 0; u < 4; u++) {
        if constexpr (COUNT) {
          const uint64_t act = __ballot(active);
          n_ref += active ? (unsigned)P : 0u;
          n_gpu += (m == 0 && ((act >> lead) & kGroup)) ? 16u : 0u;
        }
        uint32_t nidx;
        bool accept, again;
        if (step(t, active, nidx, accept, again)) bidx = nidx;
      }
    } else {
      const int row = (lane >> 4) & (rpc - 1);
      const uint64_t rows = rpc == 4 ? kLeaders : 0x00010001ull;
      for (int u = 0; u < 4; u++) {
        // this row's step: `row` rejections ahead of t
        SubState v = t;
        v.x += (uint32_t)row * 3u * kRngStep;
        v.energy += row;
        bool live = active, accept, again;
        uint32_t nidx;
        const bool better = step(v, live, nidx, accept, again);
        const uint64_t event = __ballot(active & (accept | again | !live));
        // the first row of this lane's group with an event in its chain
        const uint64_t mine = (event >> (lead + m)) & rows;
        const int last = mine ? (__ffsll((unsigned long long)mine) - 1) >> 4 : rpc - 1;
        if constexpr (COUNT) {
          const uint64_t act = __ballot(active);
          n_ref += active && row == 0 ? (unsigned)last + 1u : 0u;
          n_gpu += (m == 0 && ((act >> lead) & kGroup)) ? 16u : 0u;
        }
        if (!event) {
          t.x += (uint32_t)rpc * 3u * kRngStep;
          t.energy += rpc;
          continue;
        }
        const int from = lead + 16 * last + m;
        uint32_t bits = v.cpbc | (v.bpbc << 2) | ((better ? nidx : bidx) << 4) |
                        ((live ? 1u : 0u) << 8);
        bits = __shfl(bits, from);
        t.p1 = __shfl(v.p1, from);
        t.p2 = __shfl(v.p2, from);
        t.bp1 = __shfl(v.bp1, from);
        t.bp2 = __shfl(v.bp2, from);
        t.cur = __shfl(v.cur, from);
        t.best = __shfl(v.best, from);
        t.x = __shfl(v.x, from);
        t.energy = __shfl(v.energy, from);
        t.cpbc = bits & 3u;
        t.bpbc = (bits >> 2) & 3u;
        bidx = (bits >> 4) & 15u;
        active = (bits >> 8) & 1u;
      }
    }
    // finished groups write their records (lane_finish)
    const uint64_t act = __ballot(active);
    const bool done = has && ((act >> lead) & kGroup) == 0;
    if (!__ballot(done)) continue;
    uint32_t sum = extra + t.best, pbcs = t.bpbc, out = bidx;
    bool leader = m == 0;
    if (G == 16) {
      // every lane of the wave takes part in the shuffles
      out = bidx | ((uint32_t)__shfl_xor((int)bidx, 1) << 4);
      const uint64_t sub1 = __ballot(sub == 1) >> lead, sub2 = __ballot(sub == 2) >> lead;
      const int first1 = __ffsll((unsigned long long)(sub1 & kGroup)) - 1;
      const int first2 = __ffsll((unsigned long long)(sub2 & kGroup)) - 1;
      leader = m == 0 || m == first1 || m == first2;
      sum = extra;
      pbcs = 0;
#pragma unroll
      for (int s = 0; s < 3; s++) {
        const int from = s == 0 ? 0 : (s == 1 ? first1 : first2);
        const uint32_t e = (uint32_t)__shfl((int)t.best, lead + (from & 15));
        const uint32_t pb = (uint32_t)__shfl((int)t.bpbc, lead + (from & 15));
        if (from >= 0) {
          sum += e;
          pbcs |= pb << (2 * s);
        }
      }
    }
    if (done && (G == 4 || lane - lead < G)) {
      CandRec *rc = &w.rec[id];
      if (leader) {
        Fit f;
        set_fit(f, info & 7, (info >> 3) & 3, (info >> 5) & 1);
        const bool has_pb = f.pbit_type != PB_NONE;
        uint32_t e1 = to_pixel_int(t.bp1, f.qmask, has_pb ? (int)((t.bpbc >> k.sh) & 1u) : -1);
        uint32_t e2 = to_pixel_int(t.bp2, f.qmask, has_pb ? (int)(t.bpbc & 1u) : -1);
        if (ptmode) {
          e1 = (e1 & 0x00FFFFFFu) | (rc->px1[0] & 0xFF000000u);
          e2 = (e2 & 0x00FFFFFFu) | (rc->px2[0] & 0xFF000000u);
        }
        rc->px1[sub] = e1;
        rc->px2[sub] = e2;
      }
      if (G == 4) reinterpret_cast<uint16_t *>(&rc->cidx_lo)[m] = (uint16_t)out;
      else if (!(m & 1)) reinterpret_cast<uint8_t *>(&rc->cidx_lo)[m >> 1] = (uint8_t)out;
      if (m == 0) {
        rc->meta = (rc->meta & ~((1u << (2 * nsub)) - 1u)) | pbcs | kMetaAnnealed;
        rc->err = sum;
      }
    }
    if (done) has = active = false;
  }
}

__device__ __forceinline__ void add_counts(const Bc7Params &prm, unsigned long long a,
                                           unsigned long long b) {
  for (int off = 32; off >= 1; off >>= 1) {
    a += __shfl_xor(a, off);
    b += __shfl_xor(b, off);
  }
  if ((threadIdx.x & 63) == 0) {
    atomicAdd(&prm.work_counts[0], a);
    atomicAdd(&prm.work_counts[1], b);
  }
}

// TAIL: the candidates the one-lane form handed over (kCntTail of them);
// otherwise the whole annealing list, if spread_list has it so.
template <bool TAIL, bool COUNT>
__global__ void __launch_bounds__(256) anneal_spread_kernel(BlockRange r, Bc7Params prm, Work w,
                                                            TailState *tail,
                                                            uint32_t max_states) {
  const StateMap sm = state_map(w);
  const uint32_t total = TAIL      ? w.counters[kCntTail]
                         : w.alist ? w.counters[kCntList]
                                   : sm.count();
  if (total == 0 || (!TAIL && !spread_list(sm, total, max_states))) return;  // whole grid
  __shared__ __align__(4) uint8_t s_quant[kStepQuantBytes];
  step_quant_load(s_quant);
  __syncthreads();
  unsigned long long n_ref = 0, n_gpu = 0;
  spread_run<16, TAIL ? kFromTail : kFromList, COUNT>(r, prm, w, tail, s_quant, 0, total,
                                                      4 * gridDim.x, &w.counters[TAIL ? kCntTailFetch : kCntFetch],
                                                      n_ref, n_gpu);
  if constexpr (COUNT) add_counts(prm, n_ref, n_gpu);
}

// max_states: of spread_list (0: the list is this kernel's).
// unroll: annealing steps between looks at the idle lanes.
// tail_lanes: once the list is used up, a wave with at most this many
// running candidates hands them to anneal_spread_kernel (through `tail`),
// whose steps are several times shorter; otherwise the longest anneals, which
// set the launch's length, would run on in nearly empty waves.
// NU: the nonuniform metric (float errors, whose sums have an order: the
// lanes finish their own candidates).
// WAVES = 3 gives the uniform form 168 VGPRs, of which 18 spill (80 bytes a lane,
// stored once per `unroll` steps): two thirds of its 1.7 GB written at 4096x4096
// are scratch, against a 27 ms issue bound.
// COUNT: also count the work into prm.work_counts: [0] the QuantizedError
// point evaluations the reference's annealing makes (each step of a subset
// scores that subset's points, Compressor.cpp:583-624), [1] the pixel scores
// this kernel makes (16 per step of a candidate, whichever subsets are
// still annealing).
template <int WAVES, bool NU = false, bool COUNT = false>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WAVES)))
anneal_kernel(BlockRange r, Bc7Params prm, Work w, uint32_t unroll, uint32_t tail_lanes,
              uint32_t rot_groups, TailState *tail, uint32_t max_states) {
  const int lane = threadIdx.x & 63;
  unsigned long long n_ref = 0, n_gpu = 0;  // COUNT
  const uint64_t lt = (1ull << lane) - 1ull;
  const StateMap sm = state_map(w);
  uint32_t total = w.alist ? w.counters[kCntList] : sm.count();
  if (spread_list(sm, total, max_states)) return;  // whole grid: anneal_spread_kernel's
  // odd row stride: conflict-free
  __shared__ uint32_t s_px[256 * kRowWords];
  __shared__ __align__(4) uint8_t s_quant[kStepQuantBytes];
  step_quant_load(s_quant);
  __syncthreads();
  // Learned search: the list is in state order, so its rotation states (slots
  // past the front's) are its suffix.  Their chains are the
  // longest by far (to 1410 steps, against a mean of 66 in mode 1), so the
  // first rot_groups workgroups start on them at once, four lanes each, while
  // the others run the rest.  That holds while they are few: where one state
  // in eight or more is a rotation's (blocks the ranker is not sure about
  // anneal the reference search's candidates, a third of them rotations), the
  // few workgroups would set the time, and one lane each is the cheapest form:
  // 2048x2048 with every block unsure 31.8 ms in this phase, 8.9 without;
  // sure (one in twenty) 1.29 with and 2.38 without.
  if (!NU && rot_groups && w.alist) {
    const uint32_t first_rot = sm.front;
    uint32_t lo = 0, hi = total;  // first list entry >= first_rot
    while (lo < hi) {
      const uint32_t mid = (lo + hi) >> 1;
      if (w.alist[mid] < first_rot) lo = mid + 1;
      else hi = mid;
    }
    if (8u * (total - lo) < total) {
      if (blockIdx.x < rot_groups)
        spread_run<4, kFromListHand, COUNT>(r, prm, w, tail, s_quant, lo, total, 4 * rot_groups,
                                            &w.counters[kCntRotFetch], n_ref, n_gpu);
      total = lo;
    }
  }
  Lane L = {};  // lanes without a candidate step along on zeros
  L.nsub = 1;
  L.px = s_px + threadIdx.x * kRowWords;
  uint32_t wbase = 0, wend = 0;  // wave-local window of the list
  bool exhausted = false;
  for (;;) {
    const uint64_t running = __ballot(L.active != 0);
    const int nrun = __popcll(running);
    if (!exhausted ? 64 - nrun >= kRefillLanes : nrun == 0) {
      if (L.has && L.active == 0) {
        lane_finish<NU>(L, w);
        L.has = false;
      }
      // refill idle lanes from the window, fetching a new window when needed
      for (;;) {
        const uint64_t need = __ballot(!L.has);
        if (!need || exhausted) break;
        if (wbase >= wend) {
          uint32_t b0 = 0;
          if (lane == 0) b0 = atomicAdd(&w.counters[kCntFetch], 64u);
          b0 = __shfl(b0, 0);
          if (b0 >= total) {
            exhausted = true;
            break;
          }
          wbase = b0;
          wend = min(b0 + 64u, total);
        }
        const uint32_t avail = wend - wbase;
        const uint32_t rank = (uint32_t)__popcll(need & lt);
        if (!L.has && rank < avail) {
          // the list runs from its end: the set-up kernels append modes 0, 2,
          // 3, 7, 6, 1, 4, 5.  The rotation modes' candidates anneal the
          // longest, so the list starts with them; then come the numerous
          // mode-1 candidates, and the short mode-7 chains are among the last
          // loaded, which keeps the tail of the launch short
          const uint32_t item = total - 1u - (wbase + rank);
          lane_load<NU>(L, r, prm, w.astate[w.alist ? w.alist[item] : sm.slot(item)]);
        }
        wbase += min(avail, (uint32_t)__popcll(need));
      }
      if (!__ballot(L.has)) break;
    }
    if (!NU && exhausted && __popcll(__ballot(L.active != 0)) <= (int)tail_lanes) {
      if (L.has && L.active == 0) {
        lane_finish(L, w);
        L.has = false;
      }
      const uint64_t left = __ballot(L.has);
      uint32_t base = 0;
      if (lane == 0) base = atomicAdd(&w.counters[kCntTail], (uint32_t)__popcll(left));
      base = __shfl(base, 0);
      if (L.has) lane_hand_over(L, tail[base + (uint32_t)__popcll(left & lt)]);
      break;
    }
    for (uint32_t u = 0; u < unroll; u++) {
      if constexpr (COUNT) {
        const int n1 = __popc(L.m12 & 0xFFFFu), n2 = __popc(L.m12 >> 16);
        if (L.active) {
          n_ref += ((L.active & 1u) ? 16 - n1 - n2 : 0) + ((L.active & 2u) ? n1 : 0) +
                   ((L.active & 4u) ? n2 : 0);
          n_gpu += 16u;
        }
      }
      // keeps the texels' LDS reads inside the step: hoisted out of this loop
      // they would take 32 registers and spill
      asm volatile("" ::: "memory");
      lane_step<NU>(L, s_quant, (int)prm.quality);
    }
  }
  if constexpr (COUNT) add_counts(prm, n_ref, n_gpu);
}

// ---------------------------------------------------------------------------
// Kernel 4: choose the mode and write the block, one lane per block.
// ---------------------------------------------------------------------------

struct BitWriter {
  uint64_t lo = 0, hi = 0;
  int pos = 0;
  __device__ __forceinline__ void put(uint32_t v, int n) {
    if (n <= 0) return;
    const uint64_t vv = (uint64_t)(n >= 32 ? v : (v & ((1u << n) - 1u)));
    if (pos >= 64) {
      hi |= vv << (pos - 64);
    } else {
      lo |= vv << pos;
      if (pos + n > 64) hi |= vv >> (64 - pos);
    }
    pos += n;
  }
};

// CompressOptimalColorBC7 (Compressor.cpp:1424-1458).
__device__ void pack_solid(uint32_t pixel, uint32_t wm, BitWriter &w) {
  w.put(1u << 5, 6);
  w.put(0, 2);
#pragma unroll
  for (int ch = 0; ch < 3; ch++) {
    const uint32_t v = chan(pixel, ch);
    w.put(kMode5Tab[v][0], 7);
    w.put(kMode5Tab[v][1], 7);
  }
  w.put(pixel >> 24, 8);
  w.put(pixel >> 24, 8);
  w.put(0xaaaaaaabu, 31);
  w.put(kWM[wm], 31);
}

__device__ __forceinline__ uint32_t invert_idx(uint32_t &lo, uint32_t &hi, uint32_t mask16,
                                               uint32_t nv) {
  uint32_t nl = 0, nh = 0;
  for (int i = 0; i < 16; i++) {
    uint32_t v = idx_at(lo, hi, i);
    if ((mask16 >> i) & 1) v = nv - v;
    if (i < 8) nl |= v << (4 * i);
    else nh |= v << (4 * (i - 8));
  }
  lo = nl;
  hi = nh;
  return 0;
}

// CompressionMode::Pack (Compressor.cpp:1096-1298).  The p-bits are written
// unswapped after an anchor fix-up swap, as the reference does
// (:1149-1170 vs :1234-1241).
__device__ __forceinline__ void pack_mode(int mode, int shape, const CandRec &rec, BitWriter &w) {
  const ModeAttr a = kModes[mode];
  const int ns = a.subsets;
  const int rot = (rec.meta >> 8) & 3;
  const int im = (rec.meta >> 10) & 1;
  w.put(1u << mode, mode + 1);
  w.put((uint32_t)shape, a.part_bits);
  if (a.has_rot) w.put((uint32_t)rot, 2);
  if (a.has_idx_mode) w.put((uint32_t)im, 1);
  uint32_t px1[3] = {rec.px1[0], rec.px1[1], rec.px1[2]};
  uint32_t px2[3] = {rec.px2[0], rec.px2[1], rec.px2[2]};
  uint32_t cl = rec.cidx_lo, ch = rec.cidx_hi;
  uint32_t al = rec.aidx_lo, ah = rec.aidx_hi;
  const int nib = (im == 0) ? a.idx_bits : a.alpha_idx_bits;
  const int nab = (im == 0) ? a.alpha_idx_bits : a.idx_bits;
  // subset loops run to 3 with a guard, so px1/px2 are indexed by constants
#pragma unroll
  for (int s = 0; s < 3; s++) {
    if (s >= ns) continue;
    const uint32_t smask = subset_mask(shape, ns, s);
    const int anchor = anchor_of(s, shape, ns);
    if (idx_at(cl, ch, anchor) >> (nib - 1)) {
      const uint32_t t = px1[s];
      px1[s] = px2[s];
      px2[s] = t;
      invert_idx(cl, ch, smask, (1u << nib) - 1);
      if (a.has_rot) invert_idx(al, ah, 0xFFFFu, (1u << nab) - 1);
    }
    if (a.has_rot && (idx_at(al, ah, anchor) >> (nab - 1)) > 0) {
      const uint32_t a1 = px1[s] >> 24, a2 = px2[s] >> 24;
      px1[s] = (px1[s] & 0x00FFFFFFu) | (a2 << 24);
      px2[s] = (px2[s] & 0x00FFFFFFu) | (a1 << 24);
      invert_idx(al, ah, 0xFFFFu, (1u << nab) - 1);
    }
  }
  const int cp = a.color_prec, ap = a.alpha_prec;
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int s = 0; s < 3; s++) {
      if (s >= ns) continue;
      w.put(chan(px1[s], c) >> (8 - cp), cp);
      w.put(chan(px2[s], c) >> (8 - cp), cp);
    }
  if (ap) {
#pragma unroll
    for (int s = 0; s < 3; s++) {
      if (s >= ns) continue;
      w.put(chan(px1[s], 3) >> (8 - ap), ap);
      w.put(chan(px2[s], 3) >> (8 - ap), ap);
    }
  }
  if (a.pbit_type != PB_NONE) {
#pragma unroll
    for (int s = 0; s < 3; s++) {
      if (s >= ns) continue;
      const int pbc = (rec.meta >> (2 * s)) & 3;
      w.put((uint32_t)pbc_bit(a.pbit_type, pbc, 0), 1);
      if (a.pbit_type != PB_SHARED) w.put((uint32_t)pbc_bit(a.pbit_type, pbc, 1), 1);
    }
  }
  if (a.has_idx_mode && im == 1) {
    for (int i = 0; i < 16; i++) w.put(idx_at(al, ah, i), i == 0 ? 1 : 2);
    for (int i = 0; i < 16; i++) w.put(idx_at(cl, ch, i), i == 0 ? 2 : 3);
  } else {
    for (int i = 0; i < 16; i++) {
      int s = 0;
      for (int t = 1; t < ns; t++)
        if ((subset_mask(shape, ns, t) >> i) & 1) s = t;
      const int anchor = anchor_of(s, shape, ns);
      w.put(idx_at(cl, ch, i), i == anchor ? nib - 1 : nib);
    }
    if (a.has_rot)
      for (int i = 0; i < 16; i++) w.put(idx_at(al, ah, i), i == 0 ? nab - 1 : nab);
  }
}

// dst == nullptr writes the block into the job's output; otherwise into
// dst[rel] (the quality-0 copy the guard compares against).
__global__ void __launch_bounds__(256) pack_kernel(BlockRange r, Bc7Scratch scr, Work w,
                                                   uint4 *dst) {
  const uint32_t rel = blockIdx.x * blockDim.x + threadIdx.x;
  if (rel >= r.num_blocks) return;
  const uint32_t b = r.first_block + rel;
  const uint32_t sel = w.sel[rel];
  BitWriter bw;
  if (sel_cls(sel) == 0) {
    const uint32_t bx = b % r.blocks_wide, by = b / r.blocks_wide;
    const uint32_t pixel = r.img[(size_t)(by * 4) * r.width + bx * 4];
    const uint32_t wm = (scr.chunk_prefix[rel / 256] + scr.local_prefix[rel]) % 9;
    pack_solid(pixel, wm, bw);
  } else if (sel_cls(sel) == 1) {
    bw.put(1u << 6, 7);  // WriteTransparentBlock (Compressor.cpp:1416-1421)
  } else {
    // the slots hold the candidates in CompressClusters' order: keep the
    // first strict minimum
    const CandRec *rc = &w.rec[(size_t)rel * kMaxCands];
    const int count = sel_count(sel);
    int bc = -1;
    if (w.nu_total) {
      // the nonuniform metric's double totals (the reference's best_err
      // starts at DBL_MAX, Compressor.cpp:1756)
      const double *tn = w.nu_total + (size_t)rel * kMaxCands;
      double best = DBL_MAX;
      for (int i = 0; i < count; i++) {
        if (tn[i] < best) {
          best = tn[i];
          bc = i;
        }
      }
    } else {
      uint32_t best = 0xFFFFFFFFu;
      for (int i = 0; i < count; i++) {
        const uint32_t e = rc[i].err;
        if (e < best) {
          best = e;
          bc = i;
        }
      }
    }
    if (bc >= 0) {
      Cand k;
      cand_from_desc(w.cdesc[(size_t)rel * kMaxCands + bc], k);
      pack_mode(k.mode, k.shape, rc[bc], bw);
    }
  }
  uint4 v;
  v.x = (uint32_t)bw.lo;
  v.y = (uint32_t)(bw.lo >> 32);
  v.z = (uint32_t)bw.hi;
  v.w = (uint32_t)(bw.hi >> 32);
  if (dst) dst[rel] = v;
  else reinterpret_cast<uint4 *>(r.out)[b] = v;
}

// Quality guard (no counterpart in the reference): where the annealed block
// decodes (reference decoder) to a larger premultiplied RGB error than the
// quality-0 block, the quality-0 block is written instead.  The error is
// sum((a*c - a'*c')^2) over pixels and RGB, Image::ComputePSNR's per-pixel
// term (Base/src/Image.cpp:205-255) scaled by 255^2 to stay an exact integer.
// |d| <= 255^2, so a square is below 2^32; the three together need more.
__device__ __forceinline__ uint64_t premul_pixel(uint32_t src, uint32_t dec) {
  const uint32_t a = src >> 24, b = dec >> 24;
  uint64_t e = 0;
#pragma unroll
  for (int c = 0; c < 3; c++) {
    const int d = (int)__umul24(a, chan(src, c)) - (int)__umul24(b, chan(dec, c));
    const uint32_t m = (uint32_t)(d < 0 ? -d : d);
    e += m * m;
  }
  return e;
}
__device__ __forceinline__ uint64_t premul_err(const uint32_t src[16], const uint32_t dec[16]) {
  uint64_t e = 0;
#pragma unroll
  for (int i = 0; i < 16; i++) e += premul_pixel(src[i], dec[i]);
  return e;
}

__global__ void __launch_bounds__(256) guard_kernel(BlockRange r, const uint4 *q0) {
  const uint32_t rel = blockIdx.x * blockDim.x + threadIdx.x;
  if (rel >= r.num_blocks) return;
  const uint32_t b = r.first_block + rel;
  uint4 *out = reinterpret_cast<uint4 *>(r.out);
  const uint4 a = out[b], z = q0[rel];
  if (a.x == z.x && a.y == z.y && a.z == z.z && a.w == z.w) return;
  uint32_t px[16];
  load_block(r, rel, px);
  uint64_t ea = 0, ez = 0;
  bc7dec::decode_pixels<false>(
      a, [&](int i, uint32_t pixel) { ea += premul_pixel(px[i], pixel); });
  bc7dec::decode_pixels<false>(
      z, [&](int i, uint32_t pixel) { ez += premul_pixel(px[i], pixel); });
  if (ez < ea) out[b] = z;
}

// The learned search chooses among a block's candidates by decoded error:
// each candidate's block is packed and decoded with the reference decoder,
// and the smallest premul_err wins (ties to the lower slot).  Pass 0 (before
// annealing) keeps the quality-0 winner and its error; the final pass writes
// its winner unless the quality-0 one decodes strictly better, so no block is
// worse than at quality 0.  The errors come from cand_error_kernel, one
// candidate per thread; pick_kernel then chooses per block.

// Candidate decoded errors into cerr[id].  Pass 0 walks the type queues (a
// wave packs one mode) and also fills the slot of a mode-6 second shape
// entry, whose set-up copied the first's record; the final pass walks the
// annealing list and re-scores only the records annealing rewrote.
// Grid-stride: the item counts are device counters.  Four waves per SIMD
// (101 VGPRs, no spills) hide the dependent loads of each item.
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
cand_error_kernel(BlockRange r, Work w, unsigned long long *cerr, int final_pass) {
  uint32_t total = 0, sizes[kNumTypes];
  if (final_pass) {
    total = w.counters[kCntList];
  } else {
#pragma unroll
    for (int q = 0; q < kNumTypes; q++) total += sizes[q] = w.counters[kCntQueue + q];
  }
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < total; t += stride) {
    uint32_t id;
    if (final_pass) {
      id = w.aid[w.alist[t]];
    } else {
      uint32_t base = 0, item = 0;
      int type = kNumTypes - 1;
#pragma unroll
      for (int q = 0; q < kNumTypes; q++) {
        const uint32_t c = sizes[q];
        if (t >= base && t < base + c) {
          type = q;
          item = t - base;
        }
        base += c;
      }
      id = w.queue[(size_t)type * w.qcap + item];
    }
    const CandRec rc = w.rec[id];
    if (final_pass && !(rc.meta & kMetaAnnealed)) continue;
    const uint32_t rel = id_block(id);
    Cand k;
    cand_from_desc(w.cdesc[id], k);
    BitWriter bw;
    pack_mode(k.mode, k.shape, rc, bw);
    const uint4 blk = make_uint4((uint32_t)bw.lo, (uint32_t)(bw.lo >> 32), (uint32_t)bw.hi,
                                 (uint32_t)(bw.hi >> 32));
    uint32_t px[16];
    load_block(r, rel, px);
    unsigned long long e = 0;
    bc7dec::decode_pixels<false>(
        blk, [&](int i, uint32_t pixel) { e += premul_pixel(px[i], pixel); });
    cerr[id] = e;
    if (!final_pass && k.mode == 6) {
      const uint32_t c = id_slot(id);
      if (c + 1 < (uint32_t)sel_count(w.sel[rel])) {
        const uint32_t d1 = w.cdesc[id + 1];
        if ((d1 & 7) == 6 && ((d1 >> 12) & 7) == 1) cerr[id + 1] = e;
      }
    }
  }
}

// Per block: the smallest candidate error (first slot on ties), packed.
// Pass 0 stores the quality-0 winner and its error; the final pass writes
// the block (solid and transparent blocks as pack_kernel does), keeping the
// quality-0 winner when it decodes strictly better (q0err, if given).
//
// A full-search block (kSelFull) chooses as the full search does: the first
// strict minimum of the internal errors (CompressClusters, Compressor.cpp:
// 1752-1817), and with the guard on the final pass keeps the quality-0 block
// when it decodes strictly better (guard_kernel's rule).
__global__ void __launch_bounds__(256) pick_kernel(BlockRange r, Bc7Scratch scr, Work w,
                                                   uint4 *q0blk, unsigned long long *q0err,
                                                   const unsigned long long *cerr,
                                                   int final_pass, int q0_guard) {
  const uint32_t rel = blockIdx.x * blockDim.x + threadIdx.x;
  if (rel >= r.num_blocks) return;
  const uint32_t b = r.first_block + rel;
  const uint32_t sel = w.sel[rel];
  uint4 best = make_uint4(0, 0, 0, 0);
  if (sel_cls(sel) != 2) {
    if (!final_pass) return;
    BitWriter bw;
    if (sel_cls(sel) == 0) {
      const uint32_t bx = b % r.blocks_wide, by = b / r.blocks_wide;
      const uint32_t pixel = r.img[(size_t)(by * 4) * r.width + bx * 4];
      const uint32_t wm = (scr.chunk_prefix[rel / 256] + scr.local_prefix[rel]) % 9;
      pack_solid(pixel, wm, bw);
    } else {
      bw.put(1u << 6, 7);  // WriteTransparentBlock (Compressor.cpp:1416-1421)
    }
    best = make_uint4((uint32_t)bw.lo, (uint32_t)(bw.lo >> 32), (uint32_t)bw.hi,
                      (uint32_t)(bw.hi >> 32));
  } else {
    unsigned long long best_err = ~0ull;
    int best_i = -1;
    const int count = sel_count(sel);
    if (sel_full(sel)) {
      uint32_t best_int = 0xFFFFFFFFu;
      for (int i = 0; i < count; i++) {
        const uint32_t e = w.rec[(size_t)rel * kMaxCands + i].err;
        if (e < best_int) {
          best_int = e;
          best_i = i;
        }
      }
      if (best_i >= 0) best_err = cerr[(size_t)rel * kMaxCands + best_i];
    } else {
      for (int i = 0; i < count; i++) {
        const unsigned long long e = cerr[(size_t)rel * kMaxCands + i];
        if (e < best_err) {
          best_err = e;
          best_i = i;
        }
      }
    }
    if (best_i >= 0) {
      Cand k;
      cand_from_desc(w.cdesc[(size_t)rel * kMaxCands + best_i], k);
      BitWriter bw;
      pack_mode(k.mode, k.shape, w.rec[(size_t)rel * kMaxCands + best_i], bw);
      best = make_uint4((uint32_t)bw.lo, (uint32_t)(bw.lo >> 32), (uint32_t)bw.hi,
                        (uint32_t)(bw.hi >> 32));
    }
    if (!final_pass) {
      q0blk[rel] = best;
      q0err[rel] = best_err;
      return;
    }
    if (q0err && (q0_guard || !sel_full(sel)) && q0err[rel] < best_err) best = q0blk[rel];
  }
  reinterpret_cast<uint4 *>(r.out)[b] = best;
}

// ---------------------------------------------------------------------------
// Exhaustive quality-0 search, the training labels of the candidate ranker:
// every mode with every partition shape, rotation and index mode (the 285
// valid outputs of the ranking network) for every block.  Each candidate is
// fitted, packed and decoded with the reference decoder, and the one with
// the smallest decoded error (premul_err) wins: the encoder's internal error
// is not the decoded error for the rotation modes (stale statistics, the
// reference decoder's mode-4 index-mode-1 reading) and the single-colour
// estimate.  Ties go to the mode tried first by CompressClusters
// (0,2,1,3,7,4,5,6), then to the lower slot.  One launch per mode, so that a
// wave runs one code path; lanes take consecutive slots of one block.
// ---------------------------------------------------------------------------
__constant__ int kModePos[8] = {0, 2, 1, 3, 5, 6, 7, 4};

__device__ __forceinline__ void slot_cand(int mode, int slot, Cand &k) {
  k.mode = mode;
  k.entry = 0;
  k.nsub = kModes[mode].subsets;
  k.shape = k.nsub > 1 ? slot : 0;
  k.rot = mode == 4 ? (slot >> 1) : (mode == 5 ? slot : 0);
  k.im = mode == 4 ? (slot & 1) : 0;
}

__global__ void __launch_bounds__(256) label_fill_kernel(unsigned long long *best, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) best[i] = ~0ull;
}

// ERRORS: every candidate's decoded error to errs (n x 512 floats, logit
// order) instead of the per-block minimum.
template <bool ERRORS>
__global__ void __launch_bounds__(64) label_kernel(BlockRange r, int mode, uint32_t nslots,
                                                   const uint32_t *sctab,
                                                   unsigned long long *best, float *errs) {
  __shared__ uint32_t s_px[64 * kPxStride];
  __shared__ uint32_t s_km[16 * 3 * 64];  // k-means sums and counts (up to 16 buckets)
  const uint64_t items = (uint64_t)r.num_blocks * nslots;
  for (uint64_t item = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; item < items;
       item += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t rel = (uint32_t)(item / nslots);
    const int slot = (int)(item % nslots);
    Cand k;
    slot_cand(mode, slot, k);
    uint32_t *px = s_px + threadIdx.x * kPxStride;  // this lane's row only
    {
      uint32_t v[16];
      load_block(r, rel, v);
#pragma unroll
      for (int i = 0; i < 16; i++) px[i] = v[i];
    }
    CandRec rec;
    AState st;
    uint32_t total = 0;
    fit_candidate<-1>(k, px, 0, sctab, rec, st, total, nullptr, nullptr,
                      s_km + threadIdx.x);
    BitWriter bw;
    pack_mode(k.mode, k.shape, rec, bw);
    const uint4 blk = make_uint4((uint32_t)bw.lo, (uint32_t)(bw.lo >> 32), (uint32_t)bw.hi,
                                 (uint32_t)(bw.hi >> 32));
    uint32_t dec[16];
    bc7dec::decode_block(blk, dec);
    const unsigned long long err = premul_err(px, dec);  // < 2^38
    if constexpr (ERRORS) {
      errs[(size_t)rel * 512 + mode * 64 + slot] = (float)err;
    } else {
      const unsigned long long key =
          (err << 16) | (unsigned long long)(kModePos[mode] * 64 + slot);
      atomicMin(&best[rel], key);
    }
  }
}

__global__ void __launch_bounds__(256) label_finish_kernel(const unsigned long long *best,
                                                           uint32_t n, int32_t *labels,
                                                           unsigned long long *errors) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const unsigned long long key = best[i];
  const int rank = (int)(key & 0xFFFFu);
  labels[i] = kOrder[rank >> 6] * 64 + (rank & 63);
  if (errors) errors[i] = key >> 16;
}

// Batches: global blocks [g0, g0 + n) of the BC7 group to a block array
// (16 pixels each), and the encoded blocks back to their surfaces.
__global__ void __launch_bounds__(256) gather_kernel(const SurfDesc *surfs,
                                                     const uint32_t *block_surf, uint32_t g0,
                                                     uint32_t n, uint32_t *blocks) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;  // block * 4 + row
  const uint32_t k = t >> 2, row = t & 3;
  if (k >= n) return;
  const SurfDesc sd = surfs[block_surf[g0 + k]];
  const uint32_t b = g0 + k - sd.first;
  const uint32_t bx = b % sd.blocks_wide, by = b / sd.blocks_wide;
  const uint4 v = *reinterpret_cast<const uint4 *>(sd.img + (size_t)(by * 4 + row) * sd.width +
                                                   bx * 4);
  reinterpret_cast<uint4 *>(blocks)[(size_t)k * 4 + row] = v;
}

__global__ void __launch_bounds__(256) scatter_kernel(const SurfDesc *surfs,
                                                      const uint32_t *block_surf, uint32_t g0,
                                                      uint32_t n, const uint8_t *enc) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const SurfDesc sd = surfs[block_surf[g0 + k]];
  reinterpret_cast<uint4 *>(sd.out)[g0 + k - sd.first] =
      reinterpret_cast<const uint4 *>(enc)[k];
}

__global__ void __launch_bounds__(256) fill_kernel(uint32_t *p, uint32_t n, uint32_t v) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

__global__ void reset_kernel(uint32_t *counters, int n) {
  const int i = threadIdx.x;
  if (i < n) counters[i] = 0;
}

// Solid-block flags and in-chunk exclusive prefix (chunks of 256 blocks).
__global__ void __launch_bounds__(256) solid_scan_kernel(BlockRange r, Bc7Scratch scr) {
  __shared__ uint32_t s_wave[4];
  const uint32_t t = threadIdx.x;
  const uint32_t rel = blockIdx.x * 256 + t;
  const uint32_t b = r.first_block + rel;
  bool solid = false;
  if (rel < r.num_blocks) {
    const uint32_t bx = b % r.blocks_wide, by = b / r.blocks_wide;
    const uint32_t *p = r.img + (size_t)(by * 4) * r.width + bx * 4;
    const uint32_t p0 = p[0];
    solid = true;
#pragma unroll
    for (int y = 0; y < 4; y++) {
      const uint4 row = *reinterpret_cast<const uint4 *>(p + (size_t)y * r.width);
      solid = solid && row.x == p0 && row.y == p0 && row.z == p0 && row.w == p0;
    }
  }
  const uint64_t ballot = __ballot(solid);
  const uint32_t lanei = t & 63, wave = t >> 6;
  const uint32_t before = __popcll(ballot & ((1ull << lanei) - 1ull));
  if (lanei == 0) s_wave[wave] = __popcll(ballot);
  __syncthreads();
  uint32_t wbase = 0;
  for (uint32_t w = 0; w < wave; w++) wbase += s_wave[w];
  if (rel < r.num_blocks) scr.local_prefix[rel] = (uint8_t)(wbase + before);
  if (t == 0) scr.chunk_prefix[blockIdx.x] = s_wave[0] + s_wave[1] + s_wave[2] + s_wave[3];
}

// Exclusive scan of chunk counts (one workgroup), seeded with the watermark
// counter c: the k-th solid block of the job gets table entry (c + 1 + k) % 9
// (gWMVal = (gWMVal + 1) % 9 per solid block, Compressor.cpp:1457).  The
// counter is left at the last entry used, or unchanged if no block was solid.
__global__ void __launch_bounds__(1024) chunk_scan_kernel(Bc7Scratch scr) {
  __shared__ uint32_t s_part[1024];
  __shared__ uint32_t s_total;
  const uint32_t t = threadIdx.x;
  const uint32_t c0 = *scr.counter;
  const uint32_t g1 = (c0 + 1u) % 9u;
  if (t == 0) s_total = 0;
  __syncthreads();
  for (uint32_t base = 0; base < scr.num_chunks; base += 1024) {
    const uint32_t i = base + t;
    const uint32_t v = i < scr.num_chunks ? scr.chunk_prefix[i] : 0;
    s_part[t] = v;
    __syncthreads();
    for (uint32_t off = 1; off < 1024; off <<= 1) {
      const uint32_t add = t >= off ? s_part[t - off] : 0;
      __syncthreads();
      s_part[t] += add;
      __syncthreads();
    }
    const uint32_t excl = s_total + s_part[t] - v;
    if (i < scr.num_chunks) scr.chunk_prefix[i] = (g1 + excl % 9u) % 9u;
    __syncthreads();
    if (t == 1023) s_total += s_part[1023];
    __syncthreads();
  }
  if (t == 0 && s_total > 0) *scr.counter = (g1 + (s_total - 1u) % 9u) % 9u;
}

}  // namespace bc7

// Host launchers -------------------------------------------------------------

namespace {
int g_tables_uploaded[64];
int g_num_cus[64];
}

hipError_t bc7_upload_tables(int device) {
  if (device < 0 || device >= 64) return hipErrorInvalidDevice;
  if (g_tables_uploaded[device]) return hipSuccess;
  uint8_t m5[256][2];
  uint8_t d6[256][2][3];
  build_bc7_mode5_table(m5);
  build_bc7_dxt6_table(d6);
  hipError_t e = hipMemcpyToSymbol(HIP_SYMBOL(bc7::kMode5Tab), m5, sizeof(m5));
  if (e != hipSuccess) return e;
  static uint8_t quant[9 * 3 * 256];
  for (int bits = 0; bits <= 8; bits++) {
    const uint32_t mask = bits == 0 ? 0u : ((0xFFu << (8 - bits)) & 0xFFu);
    for (int pb = -1; pb <= 1; pb++)
      for (uint32_t v = 0; v < 256; v++)
        quant[(bits * 3 + pb + 1) * 256 + v] = (uint8_t)bc7::quant_channel(v, mask, pb);
  }
  e = hipMemcpyToSymbol(HIP_SYMBOL(bc7::kQuant), quant, sizeof(quant));
  if (e != hipSuccess) return e;
  e = hipMemcpyToSymbol(HIP_SYMBOL(bc7::kDxt6Tab), d6, sizeof(d6));
  if (e != hipSuccess) return e;
  int cus = 0;
  e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device);
  if (e != hipSuccess) return e;
  g_num_cus[device] = cus > 0 ? cus : 1;
  // the annealing step computes index weights by multiply-shift; it must
  // reproduce the interpolation table entry for entry
  static const uint8_t kWeights[3][16] = {
      {0, 21, 43, 64},
      {0, 9, 18, 27, 37, 46, 55, 64},
      {0, 4, 9, 13, 17, 21, 26, 30, 34, 38, 43, 47, 51, 55, 60, 64}};
  for (int t = 0; t < 3; t++) {
    const int nb = 4 << t;
    for (int j = 0; j < nb; j++)
      if (bc7::weight_of(bc7::weight_fn(nb), (uint32_t)j) != kWeights[t][j])
        return hipErrorInvalidValue;
  }
  g_tables_uploaded[device] = 1;
  return hipSuccess;
}

// Blocks up to which a call's annealing may run one lane per pixel
// (spread_list decides by its states: about 7 a block in the reference
// search, 1 in the learned one where the ranker is sure).  Above, the list is
// hardly ever short enough, and the set-up, which changes at the same sizes,
// has put it in the order the one-lane form wants.
constexpr uint32_t kSpreadBlocks = 1u << 14, kSpreadBlocksLearned = 1u << 16;
// Running candidates at which a wave of the one-lane form hands over
// (learned 4096x4096: 4..12 3.3 ms, 16 3.5, 24 3.6, never 3.8; reference
// search 2048x2048: 9.5 to 9.7 at 4..24).
constexpr uint32_t kTailLanes = 12;
// One workgroup in kRotShare starts on the learned list's rotation states
// (learned 4096x4096: 4 3.9 ms, 8 3.27, 9 3.20, 10 3.14, 12 3.17, 16 4.1), of
// up to four a CU: three fit, and a larger grid must not give these states a
// larger part of the chip.
constexpr uint32_t kRotShare = 10;
// Workgroups per CU of the one-lane-per-pixel form: five fit, but more waves
// on a SIMD slow the longest chains (508x380: 4 1.75 ms, 3 1.71, 2 1.78; learned
// 1024x1024: 4 0.87, 3 0.83, 2 0.85).
constexpr uint32_t kSpreadWgPerCu = 3;

// Blocks up to which every mode's set-up runs in one launch (64x64: 0.13 ms
// against 0.89 for eight launches one after another; 508x380 0.17, learned
// 1024x1024 0.24).  Larger jobs fill the chip mode by mode, and a merged
// launch would mix the modes in the annealing list, whose one-lane form wants
// them in order.
constexpr uint32_t kSetupAllBlocks = kSpreadBlocks, kSetupAllBlocksLearned = kSpreadBlocksLearned;

// waves: persistent waves of the one-lane form.  tail: memory for tail_cap
// candidates handed over.
void launch_anneal(uint32_t waves, int cus, const BlockRange &r, const Bc7Params &p,
                   const bc7::Work &w, bc7::TailState *tail, size_t tail_cap,
                   hipStream_t stream) {
  // workgroups of 16 rows, no more than the candidates could use
  uint64_t spread = ((uint64_t)r.num_blocks * bc7::kMaxCands + 15) / 16;
  if (spread > (uint64_t)cus * kSpreadWgPerCu) spread = (uint64_t)cus * kSpreadWgPerCu;
  const dim3 sgrid((uint32_t)spread), grid((waves + 3) / 4), wg(256);
  const uint32_t unroll = w.alist ? 4u : (p.anneal_unroll ? p.anneal_unroll : 1u);
  if (w.nu_total) {  // nonuniform metric (the full search or given selections)
    hipLaunchKernelGGL((bc7::anneal_kernel<1, true>), grid, wg, 0, stream, r, p, w, unroll, 0u,
                       0u, (bc7::TailState *)nullptr, 0u);
    return;
  }
  uint32_t max_states = 0;  // of spread_list
  if (r.num_blocks <= (w.alist ? kSpreadBlocksLearned : kSpreadBlocks)) {
    max_states = p.quality < bc7::kShortChains ? bc7::kSpreadStatesShort : bc7::kSpreadStates;
    if (p.work_counts)
      hipLaunchKernelGGL((bc7::anneal_spread_kernel<false, true>), sgrid, wg, 0, stream, r, p, w,
                         (bc7::TailState *)nullptr, max_states);
    else
      hipLaunchKernelGGL((bc7::anneal_spread_kernel<false, false>), sgrid, wg, 0, stream, r, p, w,
                         (bc7::TailState *)nullptr, max_states);
    const uint32_t most = p.stats || p.selections ? bc7::kMaxCands : bc7::kMaxBoxCands;
    if (r.num_blocks <= max_states / most) return;  // however many candidates
  }
  const size_t per_wave = tail_cap / ((size_t)grid.x * 4);
  // each wave hands over at most kHandGroups rotation states and `lanes` others
  const uint32_t room = per_wave > bc7::kHandGroups ? (uint32_t)per_wave - bc7::kHandGroups : 0u;
  const uint32_t lanes = room < kTailLanes ? room : kTailLanes;
  const uint32_t share_of = grid.x < (uint32_t)cus * 4u ? grid.x : (uint32_t)cus * 4u;
  const uint32_t rots = w.alist && room ? (share_of + kRotShare - 1) / kRotShare : 0u;
  if (p.work_counts) {  // the counting instances (both searches)
    hipLaunchKernelGGL((bc7::anneal_kernel<3, false, true>), grid, wg, 0, stream, r, p, w, unroll,
                       lanes, rots, tail, max_states);
    hipLaunchKernelGGL((bc7::anneal_spread_kernel<true, true>), sgrid, wg, 0, stream, r, p, w,
                       tail, 0u);
  } else {
    hipLaunchKernelGGL((bc7::anneal_kernel<3>), grid, wg, 0, stream, r, p, w, unroll, lanes,
                       rots, tail, max_states);
    hipLaunchKernelGGL((bc7::anneal_spread_kernel<true, false>), sgrid, wg, 0, stream, r, p, w,
                       tail, 0u);
  }
}

hipError_t fill_u32(uint32_t *p, uint32_t n, uint32_t v, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(bc7::fill_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, p, n, v);
  return hipGetLastError();
}

hipError_t bc7_prepare() {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  e = bc7_upload_tables(dev);
  if (e != hipSuccess) return e;
  // the device state (single-colour table, watermark counter) is created on
  // first use
  if (!device_wm_counter(dev)) return hipErrorNotInitialized;
  return bc7_single_color_table(dev) ? hipSuccess : hipErrorNotInitialized;
}

hipError_t bc7_gather(const SurfDesc *surfs, const uint32_t *block_surf, uint32_t g0, uint32_t n,
                      uint32_t *blocks, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(bc7::gather_kernel, dim3((n * 4 + 255) / 256), dim3(256), 0, stream, surfs,
                     block_surf, g0, n, blocks);
  return hipGetLastError();
}

hipError_t bc7_scatter(const SurfDesc *surfs, const uint32_t *block_surf, uint32_t g0, uint32_t n,
                       const uint8_t *enc, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(bc7::scatter_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, surfs,
                     block_surf, g0, n, enc);
  return hipGetLastError();
}

size_t bc7_work_bytes(uint32_t num_blocks, bool learned, bool nonuniform) {
  const size_t n = num_blocks;
  // counters, sel, cdesc, rec, queues, astate, q0, alignment slack
  size_t bytes = bc7::kCntWords * 4 + n * 4 + n * bc7::kMaxCands * 2 +
                 n * bc7::kMaxCands * sizeof(bc7::CandRec) +
                 n * bc7::kNumTypes * bc7::kMaxPerType * 4 +
                 n * bc7::kMaxCands * sizeof(bc7::AState) + n * 16 + 8 * 256;
  if (learned) {
    // q0 errors, candidate errors, annealing list, fallback list
    bytes += n * 8 + n * bc7::kMaxCands * (8 + 4 + 4) + n * 4 +
             (n * bc7::kMaxCands / bc7::kListChunk + 1) * 4 + 11 * 256;
  }
  if (nonuniform) bytes += n * bc7::kMaxCands * 8 + 256;  // candidate totals
  return bytes;
}

hipError_t bc7_encode(const BlockRange &r, const Bc7Params &p, const Bc7Scratch &s, void *work,
                      hipStream_t stream) {
  if (r.num_blocks == 0) return hipSuccess;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  e = bc7_upload_tables(dev);
  if (e != hipSuccess) return e;
  const uint32_t *sct = bc7_single_color_table(dev);
  if (!sct) return hipErrorOutOfMemory;
  const uint32_t n = r.num_blocks;
  // carve the work area
  uint8_t *base = reinterpret_cast<uint8_t *>(work);
  auto carve = [&](size_t bytes) {
    uint8_t *q = base;
    base += (bytes + 255) & ~(size_t)255;
    return q;
  };
  bc7::Work w;
  const size_t nc = (size_t)n * bc7::kMaxCands;
  w.counters = reinterpret_cast<uint32_t *>(carve(bc7::kCntWords * 4));
  w.sel = reinterpret_cast<uint32_t *>(carve((size_t)n * 4));
  w.cdesc = reinterpret_cast<uint16_t *>(carve(nc * 2));
  w.rec = reinterpret_cast<bc7::CandRec *>(carve(nc * sizeof(bc7::CandRec)));
  w.qcap = (uint32_t)((size_t)n * bc7::kMaxPerType);
  w.queue = reinterpret_cast<uint32_t *>(carve((size_t)w.qcap * bc7::kNumTypes * 4));
  w.astate = reinterpret_cast<bc7::AState *>(carve(nc * sizeof(bc7::AState)));
  w.astate_cap = (uint32_t)nc;
  uint4 *q0 = reinterpret_cast<uint4 *>(carve((size_t)n * 16));
  const bool learned = p.ranker != nullptr;
  unsigned long long *q0err = nullptr;
  uint32_t *fallback = nullptr;
  unsigned long long *cerr = nullptr;
  w.alist = nullptr;
  w.aid = nullptr;
  w.nu_total = nullptr;
  // the nonuniform metric runs the reference search only (the host entry
  // points reject it with the ranker or statistics)
  const bool nu = p.nonuniform != 0 && !learned && !p.stats;
  if (nu) w.nu_total = reinterpret_cast<double *>(carve(nc * 8));
  uint32_t *alist = nullptr, *chunk_count = nullptr;
  if (learned) {
    q0err = reinterpret_cast<unsigned long long *>(carve((size_t)n * 8));
    cerr = reinterpret_cast<unsigned long long *>(carve(nc * 8));
    alist = reinterpret_cast<uint32_t *>(carve(nc * 4));
    w.aid = reinterpret_cast<uint32_t *>(carve(nc * 4));
    chunk_count = reinterpret_cast<uint32_t *>(carve((nc / bc7::kListChunk + 1) * 4));
    fallback = reinterpret_cast<uint32_t *>(carve((size_t)n * 4));
  }
  uint32_t *fallback_count = w.counters + bc7::kCntFallback;
  const uint32_t nchunks = (n + 255) / 256;
  const uint32_t ngroups = (n + 15) / 16;
  // persistent workgroups of one wave, no more than the candidates could use
  uint32_t persistent = (uint32_t)g_num_cus[dev] * (p.wg_per_cu ? p.wg_per_cu : 16u);
  const uint64_t max_waves = ((uint64_t)n * bc7::kMaxCands + 63) / 64;
  if (persistent > max_waves) persistent = (uint32_t)max_waves;
  const dim3 pack_grid((n + 255) / 256);
  // candidate-error kernel: grid-stride, a few workgroups per CU
  const uint32_t err_grid = (uint32_t)g_num_cus[dev] * 8u;
  const bool guard = p.quality > 0 && p.q0_guard;
  // the type queues are dead once the set-up (and the learned search's first
  // error pass) is done: the annealing hands its tail over through them
  bc7::TailState *tail = reinterpret_cast<bc7::TailState *>(w.queue);
  const size_t tail_cap =
      (size_t)w.qcap * bc7::kNumTypes * sizeof(uint32_t) / sizeof(bc7::TailState);
  int t = timing_begin(stream);
  hipLaunchKernelGGL(bc7::reset_kernel, dim3(1), dim3(bc7::kCntWords), 0, stream, w.counters,
                     (int)bc7::kCntWords);
  hipLaunchKernelGGL(bc7::solid_scan_kernel, dim3(nchunks), dim3(256), 0, stream, r, s);
  hipLaunchKernelGGL(bc7::chunk_scan_kernel, dim3(1), dim3(1024), 0, stream, s);
  timing_end(t, kTagBc7Scan, stream);
  if (learned) {
    // rank every block and keep the confident top-k, then run BoxSelection
    // over the blocks the ranker was not sure about
    const Ranker &rk = *p.ranker;
    t = timing_begin(stream);
    hipLaunchKernelGGL(bc7::rank_select_kernel, dim3((n + mlp::kRankRows - 1) / mlp::kRankRows),
                       dim3(256), 0, stream, r, p, w, (const uint16_t *)rk.w1_oi,
                       (const uint16_t *)rk.w2_oi, (const uint16_t *)rk.w3_oi,
                       (const float *)rk.master, fallback, fallback_count);
    timing_end(t, kTagBc7Rank, stream);
    t = timing_begin(stream);
    hipLaunchKernelGGL(bc7::select_kernel<bc7::kSelBox>, dim3(ngroups), dim3(256), 0, stream,
                       r, p, w, (const uint32_t *)fallback, (const uint32_t *)fallback_count);
    timing_end(t, kTagBc7Select, stream);
  } else if (p.stats) {
    t = timing_begin(stream);
    hipLaunchKernelGGL(bc7::select_kernel<bc7::kSelStats>, dim3(ngroups), dim3(256), 0, stream,
                       r, p, w, (const uint32_t *)nullptr, (const uint32_t *)nullptr);
    timing_end(t, kTagBc7Select, stream);
  } else if (p.selections) {
    t = timing_begin(stream);
    hipLaunchKernelGGL(bc7::select_kernel<bc7::kSelGiven>, dim3(ngroups), dim3(256), 0, stream,
                       r, p, w, (const uint32_t *)nullptr, (const uint32_t *)nullptr);
    timing_end(t, kTagBc7Select, stream);
  } else if (nu) {
    t = timing_begin(stream);
    hipLaunchKernelGGL((bc7::select_kernel<bc7::kSelBox, true>), dim3(ngroups), dim3(256), 0,
                       stream, r, p, w, (const uint32_t *)nullptr, (const uint32_t *)nullptr);
    timing_end(t, kTagBc7Select, stream);
  } else {
    t = timing_begin(stream);
    hipLaunchKernelGGL(bc7::select_kernel<bc7::kSelBox>, dim3(ngroups), dim3(256), 0, stream,
                       r, p, w, (const uint32_t *)nullptr, (const uint32_t *)nullptr);
    timing_end(t, kTagBc7Select, stream);
  }
  t = timing_begin(stream);
  if (n <= (learned ? kSetupAllBlocksLearned : kSetupAllBlocks)) {
    const uint32_t fit = (uint32_t)g_num_cus[dev] * 8u;  // two waves per SIMD
    const uint32_t waves = persistent < fit ? persistent : fit;
    if (nu)
      hipLaunchKernelGGL(bc7::setup_all_kernel<true>, dim3(waves), dim3(64), 0, stream, r, p, w,
                         sct);
    else
      hipLaunchKernelGGL(bc7::setup_all_kernel<false>, dim3(waves), dim3(64), 0, stream, r, p, w,
                         sct);
  } else {
    // the waves that fit at once (setup_waves), as the batches are dealt out
    // evenly: 4096 waves over 3072 places took mode 1's 1.17 ms (learned
    // 4096x4096) to 1.44.  Annealing-state order: modes 0, 2, 3, 7, 6, 1 in
    // front, 4 and 5 behind.
    auto run = [&](auto mode) {
      constexpr int M = decltype(mode)::value;
      const uint32_t fit = (uint32_t)g_num_cus[dev] * bc7::setup_waves(M);
      const dim3 grid(persistent < fit ? persistent : fit);
      if (nu)
        hipLaunchKernelGGL((bc7::setup_kernel<M, true>), grid, dim3(64), 0, stream, r, p, w, sct);
      else
        hipLaunchKernelGGL((bc7::setup_kernel<M, false>), grid, dim3(64), 0, stream, r, p, w, sct);
    };
    run(std::integral_constant<int, 0>{});
    run(std::integral_constant<int, 2>{});
    run(std::integral_constant<int, 3>{});
    run(std::integral_constant<int, 7>{});
    run(std::integral_constant<int, 6>{});
    run(std::integral_constant<int, 1>{});
    run(std::integral_constant<int, 4>{});
    run(std::integral_constant<int, 5>{});
  }
  timing_end(t, kTagBc7Setup, stream);
  if (learned) {
    if (p.quality > 0) {
      t = timing_begin(stream);
      hipLaunchKernelGGL(bc7::cand_error_kernel, dim3(err_grid), dim3(256), 0, stream, r, w,
                         cerr, 0);
      hipLaunchKernelGGL(bc7::pick_kernel, pack_grid, dim3(256), 0, stream, r, s, w, q0, q0err,
                         (const unsigned long long *)cerr, 0, (int)p.q0_guard);
      timing_end(t, kTagBc7Pack, stream);
      bc7::Work wa = w;
      wa.alist = alist;
      t = timing_begin(stream);
      // ordered compaction of the annealing list (grid covers the largest list)
      const uint32_t nlist = (uint32_t)((nc + bc7::kListChunk - 1) / bc7::kListChunk);
      hipLaunchKernelGGL(bc7::list_count_kernel, dim3(nlist), dim3(256), 0, stream, w, cerr,
                         q0err, chunk_count);
      hipLaunchKernelGGL(bc7::list_scan_kernel, dim3(1), dim3(256), 0, stream, w, chunk_count);
      hipLaunchKernelGGL(bc7::list_write_kernel, dim3(nlist), dim3(256), 0, stream, w, cerr,
                         q0err, (const uint32_t *)chunk_count, alist);
      launch_anneal(persistent, g_num_cus[dev], r, p, wa, tail, tail_cap, stream);
      timing_end(t, kTagBc7Anneal, stream);
    }
    t = timing_begin(stream);
    bc7::Work wf = w;
    wf.alist = alist;
    // quality 0: every candidate's error; otherwise the annealed ones
    hipLaunchKernelGGL(bc7::cand_error_kernel, dim3(err_grid), dim3(256), 0, stream, r, wf, cerr,
                       p.quality > 0 ? 1 : 0);
    hipLaunchKernelGGL(bc7::pick_kernel, pack_grid, dim3(256), 0, stream, r, s, w, q0,
                       p.quality > 0 ? q0err : (unsigned long long *)nullptr,
                       (const unsigned long long *)cerr, 1, (int)p.q0_guard);
    timing_end(t, kTagBc7Pack, stream);
    return hipGetLastError();
  }
  if (guard) {
    t = timing_begin(stream);
    hipLaunchKernelGGL(bc7::pack_kernel, pack_grid, dim3(256), 0, stream, r, s, w, q0);
    timing_end(t, kTagBc7Pack, stream);
  }
  if (p.quality > 0) {
    t = timing_begin(stream);
    launch_anneal(persistent, g_num_cus[dev], r, p, w, tail, tail_cap, stream);
    timing_end(t, kTagBc7Anneal, stream);
  }
  t = timing_begin(stream);
  hipLaunchKernelGGL(bc7::pack_kernel, pack_grid, dim3(256), 0, stream, r, s, w,
                     (uint4 *)nullptr);
  timing_end(t, kTagBc7Pack, stream);
  if (guard) {
    t = timing_begin(stream);
    hipLaunchKernelGGL(bc7::guard_kernel, pack_grid, dim3(256), 0, stream, r, q0);
    timing_end(t, kTagBc7Guard, stream);
  }
  if (p.stats)
    hipLaunchKernelGGL(bc7::stats_mode_kernel, pack_grid, dim3(256), 0, stream, r, p.stats);
  return hipGetLastError();
}

hipError_t bc7_exhaustive_labels(const BlockRange &r, unsigned long long *best,
                                 int32_t *labels, unsigned long long *errors,
                                 hipStream_t stream) {
  const uint32_t n = r.num_blocks;
  if (n == 0) return hipSuccess;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  e = bc7_upload_tables(dev);
  if (e != hipSuccess) return e;
  const uint32_t *sct = bc7_single_color_table(dev);
  if (!sct) return hipErrorOutOfMemory;
  hipLaunchKernelGGL(bc7::label_fill_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, best,
                     n);
  static const uint32_t kSlots[8] = {16, 64, 64, 64, 8, 4, 1, 64};
  const int t = timing_begin(stream);
  for (int mode = 0; mode < 8; mode++) {
    const uint64_t items = (uint64_t)n * kSlots[mode];
    uint64_t groups = (items + 63) / 64;
    const uint64_t cap = (uint64_t)g_num_cus[dev] * 64;
    if (groups > cap) groups = cap;
    hipLaunchKernelGGL(bc7::label_kernel<false>, dim3((uint32_t)groups), dim3(64), 0, stream, r,
                       mode, kSlots[mode], sct, best, (float *)nullptr);
  }
  timing_end(t, kTagBc7Labels, stream);
  hipLaunchKernelGGL(bc7::label_finish_kernel, dim3((n + 255) / 256), dim3(256), 0, stream,
                     (const unsigned long long *)best, n, labels, errors);
  return hipGetLastError();
}

hipError_t bc7_candidate_errors(const BlockRange &r, float *errs, hipStream_t stream) {
  const uint32_t n = r.num_blocks;
  if (n == 0) return hipSuccess;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  e = bc7_upload_tables(dev);
  if (e != hipSuccess) return e;
  const uint32_t *sct = bc7_single_color_table(dev);
  if (!sct) return hipErrorOutOfMemory;
  // logits that are no candidate stay +inf
  const uint64_t words = (uint64_t)n * 512;
  hipLaunchKernelGGL(bc7::fill_kernel, dim3((uint32_t)((words + 255) / 256)), dim3(256), 0, stream,
                     reinterpret_cast<uint32_t *>(errs), (uint32_t)words, 0x7F800000u);
  static const uint32_t kSlots[8] = {16, 64, 64, 64, 8, 4, 1, 64};
  const int t = timing_begin(stream);
  for (int mode = 0; mode < 8; mode++) {
    const uint64_t items = (uint64_t)n * kSlots[mode];
    uint64_t groups = (items + 63) / 64;
    const uint64_t cap = (uint64_t)g_num_cus[dev] * 64;
    if (groups > cap) groups = cap;
    hipLaunchKernelGGL(bc7::label_kernel<true>, dim3((uint32_t)groups), dim3(64), 0, stream, r,
                       mode, kSlots[mode], sct, (unsigned long long *)nullptr, errs);
  }
  timing_end(t, kTagBc7Labels, stream);
  return hipGetLastError();
}

}  // namespace fh
