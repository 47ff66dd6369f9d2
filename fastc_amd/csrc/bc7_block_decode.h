// BC7 (BPTC) block decoder shared by the decode kernel and the encoder's
// quality guard: BPTCC::Decompress (BPTCEncoder/src/Decompressor.cpp:32-367).
//
// Like the reference, mode 4 blocks with index mode 1 interpolate with the
// per-mode index widths rather than the swapped ones (Decompressor.cpp:263-295),
// so decoded pixels match the reference decoder byte for byte.  With SPEC the
// widths swap with the indices, as the BC7 specification (and hardware)
// decodes such blocks.  Blocks with the reserved mode (no mode bit in the
// first byte) decode to zero.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace fh {
namespace bc7dec {

struct Attr {
  int8_t subsets, part_bits, rot_bits, idxm_bits, cprec, aprec, pbit, idx_bits, aidx_bits;
};
// pbit: 0 none, 1 shared per subset, 2 one per endpoint
static __constant__ Attr kAttr[8] = {{3, 4, 0, 0, 4, 0, 2, 3, 0}, {2, 6, 0, 0, 6, 0, 1, 3, 0},
                              {3, 6, 0, 0, 5, 0, 0, 2, 0}, {2, 6, 0, 0, 7, 0, 2, 2, 0},
                              {1, 0, 2, 1, 5, 6, 0, 2, 3}, {1, 0, 2, 0, 7, 8, 0, 2, 2},
                              {1, 0, 0, 0, 7, 7, 2, 4, 0}, {2, 6, 0, 0, 5, 5, 2, 2, 0}};
static __constant__ uint16_t kS2[64] = {
    0xcccc, 0x8888, 0xeeee, 0xecc8, 0xc880, 0xfeec, 0xfec8, 0xec80, 0xc800, 0xffec, 0xfe80,
    0xe800, 0xffe8, 0xff00, 0xfff0, 0xf000, 0xf710, 0x008e, 0x7100, 0x08ce, 0x008c, 0x7310,
    0x3100, 0x8cce, 0x088c, 0x3110, 0x6666, 0x366c, 0x17e8, 0x0ff0, 0x718e, 0x399c, 0xaaaa,
    0xf0f0, 0x5a5a, 0x33cc, 0x3c3c, 0x55aa, 0x9696, 0xa55a, 0x73ce, 0x13c8, 0x324c, 0x3bdc,
    0x6996, 0xc33c, 0x9966, 0x0660, 0x0272, 0x04e4, 0x4e40, 0x2720, 0xc936, 0x936c, 0x39c6,
    0x639c, 0x9336, 0x9cc6, 0x817e, 0xe718, 0xccf0, 0x0fcc, 0x7744, 0xee22};
static __constant__ uint16_t kS3[64][2] = {
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
static __constant__ uint8_t kA2[64] = {
    15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 2,  8,  2,  2, 8,
    8,  15, 2,  8,  2,  2,  8,  8,  2,  2,  15, 15, 6,  8,  2,  8,  15, 15, 2,  8,  2, 2,
    2,  15, 15, 6,  6,  2,  6,  8,  15, 15, 2,  2,  15, 15, 15, 15, 15, 2,  2,  15};
static __constant__ uint8_t kA3[2][64] = {
    {3,  3, 15, 15, 8, 3,  15, 15, 8,  8,  6,  6,  6,  5,  3,  3,  3,  3,  8, 15, 3,  3,
     6,  10, 5, 8,  8, 6,  8,  5,  15, 15, 8,  15, 3,  5,  6,  10, 8,  15, 15, 3, 15, 5,
     15, 15, 15, 15, 3, 15, 5,  5,  5,  8,  5,  10, 5,  10, 8,  13, 15, 12, 3,  3},
    {15, 8,  8,  3,  15, 15, 3,  8,  15, 15, 15, 15, 15, 15, 15, 8,  15, 8,  15, 3,  15, 8,
     15, 8,  3,  15, 6,  10, 15, 15, 10, 8,  15, 3,  15, 10, 10, 8,  9,  10, 6,  15, 8,  15,
     3,  6,  6,  8,  15, 3,  15, 15, 15, 15, 15, 15, 15, 15, 15, 15, 3,  15, 15, 8}};
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ u16x2 as_pair(uint32_t v) { return __builtin_bit_cast(u16x2, v); }
__device__ __forceinline__ uint32_t as_word(u16x2 v) { return __builtin_bit_cast(uint32_t, v); }

// The 64 bits of the block from bit pos (< 128) on.
__device__ __forceinline__ uint64_t bits_from(uint64_t lo, uint64_t hi, uint32_t pos) {
  // shift counts masked to 0..63: the branch not taken never shifts out of range
  return pos >= 64 ? (hi >> ((pos - 64) & 63u))
                   : ((lo >> (pos & 63u)) | ((hi << 1) << ((63 - pos) & 63u)));
}

// v with a zero bit put in at bit p (< 64), the bits from p on moved up.
__device__ __forceinline__ uint64_t insert_zero(uint64_t v, uint32_t p) {
  const uint64_t low = (1ull << p) - 1ull;
  return (v & low) | ((v & ~low) << 1);
}

// Interpolation weight of index v for n-bit indices in the word's high half,
// the reference's kInterpolationValues (Compressor.cpp:159-168):
// round(64 v / (2^n - 1)) as ((128 v + m) recip) >> 16 with m = 2^n - 1 and a
// 16-bit reciprocal of 2 m that is exact for these operands, multiplied out.
struct Weight {
  uint32_t mul, add;
};
__device__ __forceinline__ Weight weight_of_width(uint32_t n) {
  const uint32_t recip = n == 2 ? 10923u : (n == 3 ? 4682u : 2185u);
  return {128u * recip, ((1u << n) - 1u) * recip};
}
__device__ __forceinline__ uint32_t weight_hi(Weight w, uint32_t v) {
  // both factors are below 2^24: the full-rate multiply-add
  uint32_t r;
  asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(r) : "v"(v), "v"(w.mul), "v"(w.add));
  return r;
}

// One subset's endpoints for the interpolation: 64 e0 + 32 and e1 - e0 of the
// channel pairs (0, 2) and (1, 3).
struct Line {
  uint32_t a02, a13, d02, d13;
};
__device__ __forceinline__ Line line_of(uint32_t x02, uint32_t x13, uint32_t y02, uint32_t y13) {
  return {(x02 << 6) + 0x00200020u, (x13 << 6) + 0x00200020u,
          as_word(as_pair(y02) - as_pair(x02)), as_word(as_pair(y13) - as_pair(x13))};
}
__device__ __forceinline__ void pick_line(Line &c, bool take, const Line &o) {
  c.a02 = take ? o.a02 : c.a02;
  c.a13 = take ? o.a13 : c.a13;
  c.d02 = take ? o.d02 : c.d02;
  c.d13 = take ? o.d13 : c.d13;
}

// Decodes one 16-byte block (little-endian 128-bit stream), handing its 16
// RGBA8 pixels to put(i, pixel) in raster order (a caller that needs each only
// once keeps 16 registers free).  Every field position is computed from the mode's
// attributes, so lanes holding blocks of different modes run one path and
// nothing is indexed dynamically in private memory.
//
// The kernels that call this are bound by VALU issue, the whole-image decode
// (908 instructions a wave, 24 of its 27 us at 4096x4096) with its stores.  Each channel's
// endpoint fields are one 32-bit chunk of the stream, widened as 16-bit pairs
// of channels; the index streams are taken out once, with the anchors' missing
// top bits put back, and shifted along; and a pixel is one packed
// multiply-add and shift per channel pair and one byte permutation for the
// rotation: about 28 instructions a pixel where a field extraction, four
// scalar interpolations and the rotation took 90.  The pixels' code is there
// once for each number of subsets, and a wave takes the one that its lanes
// need at most, which keeps the decode at 57 VGPRs (134 with the lines picked
// by branches).  4096x4096 BC7 decode: 47.2 -> 26.8 us.
template <bool SPEC, class Put>
__device__ __forceinline__ void decode_pixels(const uint4 raw, Put put) {
  const uint64_t lo = (uint64_t)raw.x | ((uint64_t)raw.y << 32);
  const uint64_t hi = (uint64_t)raw.z | ((uint64_t)raw.w << 32);
  const uint32_t first = raw.x & 0xFFu;
  if (first == 0) {  // reserved mode
#pragma unroll
    for (int i = 0; i < 16; i++) put(i, 0u);
    return;
  }
  const int mode = __builtin_ctz(first);
  const Attr a = kAttr[mode];
  const uint32_t ns = a.subsets, cp = a.cprec, ap = a.aprec;
  uint32_t pos = mode + 1;
  // shape, rotation and index mode lie in the first 14 bits
  const uint32_t shape = (raw.x >> pos) & ((1u << a.part_bits) - 1u);
  pos += a.part_bits;
  const uint32_t rot = (raw.x >> pos) & ((1u << a.rot_bits) - 1u);
  pos += a.rot_bits;
  const bool im = ((raw.x >> pos) & ((1u << a.idxm_bits) - 1u)) != 0;
  pos += a.idxm_bits;
  // endpoints: R, G, B of every subset and endpoint (at most 30 bits a
  // channel), then A, then p-bits
  const uint32_t per = 2 * ns * cp;
  const uint32_t apos = pos + 3 * per, pbpos = apos + 2 * ns * ap;
  const uint32_t npb = a.pbit == 1 ? ns : (a.pbit == 2 ? 2 * ns : 0);
  const uint32_t cr = (uint32_t)bits_from(lo, hi, pos);
  const uint32_t cg = (uint32_t)bits_from(lo, hi, pos + per);
  const uint32_t cb = (uint32_t)bits_from(lo, hi, pos + 2 * per);
  const uint32_t ca = (uint32_t)bits_from(lo, hi, apos);
  // the p-bit of endpoint k in bit k: shared ones (two subsets) twice
  uint32_t pb = (uint32_t)bits_from(lo, hi, pbpos) & ((1u << npb) - 1u);
  if (a.pbit == 1) pb = (pb & 1u) * 3u | ((pb >> 1) & 1u) * 12u;
  const uint32_t ext = a.pbit ? 1u : 0u, cpp = cp + ext, app = ap + ext;
  const uint32_t up02 = (8 - cp) * 0x10001u, up13 = (8 - cp) | ((8 - ap) << 16);
  const uint32_t dn02 = cpp * 0x10001u, dn13 = cpp | (app << 16);
  const uint32_t pc = 1u << (7 - cp);  // used with p-bits only, where cp and ap are below 8
  const uint32_t pb02 = pc * 0x10001u, pb13 = pc | (ap ? (1u << ((7 - ap) & 7u)) << 16 : 0u);
  const uint32_t opaque = ap ? 0u : 0x00FF0000u;
  const uint32_t cmask = (1u << cp) - 1u, amask = (1u << ap) - 1u;
  auto endpoint = [&](uint32_t k, uint32_t &o02, uint32_t &o13) {
    const uint32_t c = k * cp;
    // lanes with fewer subsets read past their fields: never used
    const uint32_t f02 = ((cr >> (c & 31u)) & cmask) | (((cb >> (c & 31u)) & cmask) << 16);
    const uint32_t f13 =
        ((cg >> (c & 31u)) & cmask) | (((ca >> ((k * ap) & 31u)) & amask) << 16);
    const bool bit = (pb >> k) & 1u;
    const u16x2 v02 = (as_pair(f02) << as_pair(up02)) | as_pair(bit ? pb02 : 0u);
    const u16x2 v13 = (as_pair(f13) << as_pair(up13)) | as_pair(bit ? pb13 : 0u);
    o02 = as_word(v02 | (v02 >> as_pair(dn02)));
    o13 = as_word(v13 | (v13 >> as_pair(dn13))) | opaque;
  };
  auto line = [&](uint32_t s) {
    uint32_t x02, x13, y02, y13;
    endpoint(2 * s, x02, x13);
    endpoint(2 * s + 1, y02, y13);
    return line_of(x02, x13, y02, y13);
  };
  const Line l0 = line(0), l1 = line(1), l2 = line(2);
  uint32_t m1 = 0, m2 = 0, a1 = 16, a2 = 16;  // masks (subset 2 lies in m1 too), anchors
  if (ns == 2) {
    m1 = kS2[shape];
    a1 = kA2[shape];
  } else if (ns == 3) {
    m1 = kS3[shape][0];
    m2 = kS3[shape][1];
    const uint32_t b1 = kA3[0][shape], b2 = kA3[1][shape];
    a1 = b1 < b2 ? b1 : b2;
    a2 = b1 < b2 ? b2 : b1;
  }
  // index streams: colour (anchors carry one bit less), then alpha (modes 4
  // and 5); the others' alpha reads the colour indices
  const uint32_t ib = a.idx_bits, aib = a.aidx_bits;
  const uint32_t cstart = pbpos + npb;
  uint64_t cs = insert_zero(bits_from(lo, hi, cstart), ib - 1);
  // (one subset has no further anchor; with more, ib <= 3 and the bit is below 64)
  if (a1 < 16) cs = insert_zero(cs, a1 * ib + ib - 1);
  if (a2 < 16) cs = insert_zero(cs, a2 * ib + ib - 1);
  uint64_t as = aib ? insert_zero(bits_from(lo, hi, cstart + 16 * ib - ns), aib - 1) : cs;
  const uint32_t ab = aib ? aib : ib;
  // the index mode swaps the streams; the reference keeps the per-mode widths
  // for the weights after the swap
  const uint32_t cw = im ? ab : ib, aw = im ? ib : ab;
  if (im) {
    const uint64_t t = as;
    as = cs;
    cs = t;
  }
  const Weight wfc = weight_of_width(SPEC ? cw : ib), wfa = weight_of_width(SPEC ? aw : ab);
  const uint32_t ci_mask = (1u << cw) - 1u, ai_mask = (1u << aw) - 1u;
  // mode 4 with index mode 1: 3-bit colour indices against the 2-bit table row,
  // which is 0 (both weights) past its end
  const bool quirk = !SPEC && im;
  // byte permutation that swaps alpha with channel rot - 1
  const uint32_t perm = rot == 0 ? 0x03020100u
                                 : (rot == 1 ? 0x00020103u : (rot == 2 ? 0x01020300u : 0x02030100u));
  // LINES: the most subsets of the wave's lanes
  auto pixels = [&](auto lines) {
    constexpr int LINES = decltype(lines)::value;
#pragma unroll
    for (uint32_t i = 0; i < 16; i++) {
      const uint32_t ci = (uint32_t)cs & ci_mask, ai = (uint32_t)as & ai_mask;
      cs >>= cw;
      as >>= aw;
      Line c = l0;
      if (LINES > 1) pick_line(c, (m1 >> i) & 1u, l1);
      if (LINES > 2) pick_line(c, (m2 >> i) & 1u, l2);
      const uint32_t wc = weight_hi(wfc, ci), wa = weight_hi(wfa, ai);
      const u16x2 W02 = {as_pair(wc).y, as_pair(wc).y};
      const u16x2 W13 = as_pair(__builtin_amdgcn_perm(wa, wc, 0x07060302u));
      const u16x2 S = {6, 6};
      const u16x2 r02 = (as_pair(c.d02) * W02 + as_pair(c.a02)) >> S;
      const u16x2 r13 = (as_pair(c.d13) * W13 + as_pair(c.a13)) >> S;
      uint32_t pixel = as_word(r02) | (as_word(r13) << 8);
      if (!SPEC) pixel = quirk && ci > 3u ? (as_word(r13) << 8) & 0xFF000000u : pixel;
      put((int)i, __builtin_amdgcn_perm(pixel, pixel, perm));
    }
  };
  if (__ballot(ns > 2)) pixels(std::integral_constant<int, 3>{});
  else if (__ballot(ns > 1)) pixels(std::integral_constant<int, 2>{});
  else pixels(std::integral_constant<int, 1>{});
}

template <bool SPEC = false>
__device__ __forceinline__ void decode_block(const uint4 raw, uint32_t px[16]) {
  decode_pixels<SPEC>(raw, [&](int i, uint32_t pixel) { px[i] = pixel; });
}

}  // namespace bc7dec
}  // namespace fh
