"""Pins for the BC7 CPU oracle (no GPU).

The reference BC7 encoder cannot be built here (its headers need CMake-made
config files) and its own tests do not cover it, so each oracle function is
pinned by golden data the reference tree holds, by a closed form, by an
invariant, or by brute force on small inputs.  Each check is chosen so that a
plausible slip (wrong shift, dropped term, swapped operand) fails it.
"""
import hashlib
import json
import os

import numpy as np
import pytest

from fastc_amd import synth

HERE = os.path.dirname(os.path.abspath(__file__))
REF = "/root/reference"


def _tab(ptr, n):
    return np.ctypeslib.as_array(ptr, shape=(n,)).copy()


def test_lookup_tables_match_reference(oracle):
    """Generator-built tables == the reference's literal tables
    (BPTCEncoder/src/BCLookupTables.h), by hash fixture and, when the tree is
    present, element by element."""
    L = oracle.lib()
    m5 = _tab(L.ora_table_mode5(), 512)
    d6 = _tab(L.ora_table_dxt6(), 1536)
    fx = json.load(open(os.path.join(HERE, "golden", "bc7_tables.json")))
    assert hashlib.sha256(m5.tobytes()).hexdigest() == fx["mode5_sha256"]
    assert hashlib.sha256(d6.tobytes()).hexdigest() == fx["dxt6_sha256"]
    path = os.path.join(REF, "BPTCEncoder", "src", "BCLookupTables.h")
    if os.path.exists(path):
        from tests.golden.make_golden import parse_table
        text = open(path).read()
        assert np.array_equal(m5, parse_table(text, "Optimal7CompressBC7Mode5[256][2]"))
        assert np.array_equal(d6, parse_table(text, "Optimal6CompressDXT1[256][2][3]"))


def _expand(k, prec, pbit):
    """Grid value k (prec bits, optional p-bit appended) replicated to 8 bits."""
    bits = prec + (pbit >= 0)
    v = (k << 1 | pbit) if pbit >= 0 else k
    v <<= 8 - bits
    return (v | (v >> bits)) & 0xFF


@pytest.mark.parametrize("prec", [4, 5, 6, 7])
@pytest.mark.parametrize("pbit", [-1, 0, 1])
def test_quantize_channel_closed_form(oracle, prec, pbit):
    """QuantizeChannel (RGBAEndpoints.cpp:126-165), all 256 inputs.

    Always a value of the endpoint grid, idempotent on the grid and monotone.
    With a p-bit it is the nearest grid value (ties go up).  Without one it
    never rounds below the grid value sharing the input's top `prec` bits: it
    is the nearest grid value among those whose top bits are at least the
    input's (ties go up) -- e.g. 144 -> 153, not the closer 136, at 4 bits."""
    L = oracle.lib()
    mask = (0xFF << (8 - prec)) & 0xFF
    grid = sorted({_expand(k, prec, pbit) for k in range(1 << prec)})
    res = [L.ora_quantize_channel(v, mask, pbit) for v in range(256)]
    assert all(r in grid for r in res)
    assert all(res[g] == g for g in grid)
    assert all(res[i] <= res[i + 1] for i in range(255))
    for val in range(256):
        allowed = grid if pbit >= 0 else [g for g in grid if (g >> (8 - prec)) >= (val >> (8 - prec))]
        d = [abs(val - g) for g in allowed]
        best = min(d)
        want = max(g for g, dd in zip(allowed, d) if dd == best)
        assert res[val] == want, (val, prec, pbit, res[val], want)


def test_quantize_channel_special_masks(oracle):
    L = oracle.lib()
    for v in range(256):
        assert L.ora_quantize_channel(v, 0xFF, -1) == v
        assert L.ora_quantize_channel(v, 0xFF, 1) == v
        assert L.ora_quantize_channel(v, 0x00, -1) == 0xFF


def test_to_pixel_rounds_in_double(oracle):
    """uint32(c + 0.5) is evaluated in double (RGBAEndpoints.cpp:169): the
    float just below 0.5 rounds down, which a float add would round up."""
    L = oracle.lib()
    below = np.nextafter(np.float32(0.5), np.float32(0))
    for c, want in [(below, 0), (0.5, 1), (1.4999999, 1), (254.5, 255), (255.0, 255),
                    (np.float32(127.49999), 127)]:
        v = np.array([c, 0, 0, 0], dtype=np.float32)
        assert L.ora_to_pixel(v.ctypes.data, 0xFFFFFFFF, -1) & 0xFF == want, c


def test_length_is_correctly_rounded_sqrt(oracle):
    """VectorBase::Length takes sqrt in long double then rounds to float; the
    result equals the correctly rounded float sqrt of the float dot product
    (reference test: Base/test/TestVector.cpp:118-129)."""
    L = oracle.lib()
    rng = np.random.default_rng(0)
    v6 = np.array([1, 2, 3, 4], dtype=np.float32)
    assert L.ora_length(v6.ctypes.data) == np.float32(np.sqrt(np.float32(30)))
    for _ in range(20000):
        v = (rng.standard_normal(4) * rng.choice([1e-3, 1, 300])).astype(np.float32)
        s = np.float32(0)
        for x in v:
            s = np.float32(s + np.float32(x * x))
        assert L.ora_length(v.ctypes.data) == np.sqrt(s)


def _power_iter(m, steps):
    b = np.full(4, 0.5)
    for _ in range(steps):
        nb = m @ b
        b = nb / np.linalg.norm(nb)
    return b


def test_power_method(oracle):
    """MatrixSquare::PowerMethod (MatrixSquare.h:44-105): at most 4 products
    starting from (1/2,1/2,1/2,1/2).  A rank-1 matrix converges at once and
    reports its eigenvalue (the reference's own test, TestMatrix.cpp:213-230,
    checks a 2x2 case the same way); a general matrix follows 4 steps of the
    textbook iteration."""
    import ctypes
    L = oracle.lib()
    u = np.array([0.2, -0.5, 0.7, 0.4])
    u /= np.linalg.norm(u)
    m = (3.0 * np.outer(u, u)).astype(np.float32)
    eig = np.zeros(4, np.float32)
    ev = ctypes.c_float(0)
    L.ora_power_method(m.ctypes.data, eig.ctypes.data, ctypes.byref(ev))
    assert np.allclose(np.abs(eig), np.abs(u), atol=1e-6)
    assert abs(ev.value - 3.0) < 1e-5
    rng = np.random.default_rng(1)
    for _ in range(200):
        a = rng.standard_normal((4, 4))
        m = (a @ a.T).astype(np.float32)
        eig = np.zeros(4, np.float32)
        it = L.ora_power_method(m.ctypes.data, eig.ctypes.data, None)
        want = _power_iter(m.astype(np.float64), it - 1 if it < 5 else 4)
        assert np.allclose(eig, want, atol=2e-4), (it, eig, want)


def _interp_err(pix, e1, e2, j, nb):
    w = {4: [0, 21, 43, 64], 8: [0, 9, 18, 27, 37, 46, 55, 64],
         16: [0, 4, 9, 13, 17, 21, 26, 30, 34, 38, 43, 47, 51, 55, 60, 64]}[nb][j]
    e = 0
    for k in range(4):
        a = (e1 >> (8 * k)) & 255
        b = (e2 >> (8 * k)) & 255
        ip = (a * (64 - w) + b * w + 32) >> 6
        e += (((pix >> (8 * k)) & 255) - ip) ** 2
    return e


def test_quantized_error_indices_and_bound(oracle):
    """QuantizedError (RGBAEndpoints.cpp:190-310): the returned error is the sum
    of the errors of the returned indices, and never below the exhaustive
    best-index error (the index search is local)."""
    L = oracle.lib()
    rng = np.random.default_rng(2)
    for trial in range(300):
        px = rng.integers(0, 2**32, 16, dtype=np.uint64).astype(np.uint32)
        if trial % 3 == 0:
            base = rng.integers(0, 200)
            px = (np.uint32(base) + rng.integers(0, 40, 16).astype(np.uint32)) * np.uint32(0x01010101)
        nb = [4, 8, 16][trial % 3]
        p1 = rng.integers(0, 256, 4).astype(np.float32)
        p2 = rng.integers(0, 256, 4).astype(np.float32)
        idx = np.zeros(16, np.uint8)
        err = L.ora_quantized_error(px.ctypes.data, None, 16, p1.ctypes.data, p2.ctypes.data,
                                    nb, 0xFFFFFFFF, None, idx.ctypes.data)
        q1 = int(sum(int(p1[k]) << (8 * k) for k in range(4)))
        q2 = int(sum(int(p2[k]) << (8 * k) for k in range(4)))
        if q1 == q2:
            continue
        tot = sum(_interp_err(int(px[i]), q1, q2, int(idx[i]), nb) for i in range(16))
        assert err == tot
        brute = sum(min(_interp_err(int(px[i]), q1, q2, j, nb) for j in range(nb))
                    for i in range(16))
        assert err >= brute


def _encode_block(oracle, px, **kw):
    out, st = oracle.bc7_compress_block(np.array(px, dtype=np.uint32), **kw)
    return out, st


def _mode_of(blk):
    m = 0
    while m < 8 and not (blk[0] >> m) & 1:
        m += 1
    return m


def test_solid_blocks_decode_exactly(oracle):
    """CompressOptimalColorBC7 (Compressor.cpp:1424-1458): every 8-bit value is
    reproduced exactly by mode 5 with the table endpoints, whatever the
    watermark entry."""
    for v in range(256):
        px = [(v) | ((255 - v) << 8) | (((v * 7) & 255) << 16) | (((v * 13) & 255) << 24)] * 16
        for wm in (0, 4, 8):
            out, st = _encode_block(oracle, px, wm_index=wm)
            assert st.path == 0 and _mode_of(out) == 5
            dec = oracle.bc7_decode_block_spec(out)
            assert np.all(dec == px[0]), (v, wm)


def test_transparent_block(oracle):
    """WriteTransparentBlock (Compressor.cpp:1416-1421): mode 6, all zero."""
    px = [(i * 0x00030507) & 0x00FFFFFF for i in range(16)]
    out, st = _encode_block(oracle, px)
    assert st.path == 1
    assert out[0] == 0x40 and not out[1:].any()
    assert not oracle.bc7_decode_block_spec(out).any()


def test_watermark_sequence_in_raster_order(oracle):
    """gWMVal advances once per solid block in processing order, starting at
    entry 0 in a fresh process (Compressor.cpp:140,1457)."""
    wm_tab = [0x32b92180, 0x32ba3080, 0x31103200, 0x28103c80, 0x32bb3080,
              0x25903600, 0x3530b900, 0x3b32b180, 0x34b5b98]
    img = np.zeros((4, 4 * 12), dtype=np.uint32)
    for b in range(12):
        img[:, 4 * b:4 * b + 4] = 0xFF000000 | (b * 20)
    out, wm = oracle.bc7_compress(img)
    for b in range(12):
        blk = out[16 * b:16 * b + 16]
        bits = int.from_bytes(blk.tobytes(), "little")
        assert (bits >> 97) & 0x7FFFFFFF == wm_tab[b % 9]
    assert wm == 11 % 9


def test_box_selection_known_answers(oracle):
    import ctypes
    L = oracle.lib()
    ns, s2, s3, modes = (ctypes.c_uint32() for _ in range(4))
    # two flat colours split top/bottom = shape 13 (mask 0xff00): early exit
    px = np.array([0xFF102030] * 8 + [0xFF80A0C0] * 8, dtype=np.uint32)
    L.ora_bc7_box_selection(px.ctypes.data, ctypes.byref(ns), ctypes.byref(s2),
                            ctypes.byref(s3), ctypes.byref(modes))
    assert (ns.value, s2.value, modes.value) == (1, 13, 0b10001010)
    # a non-opaque gradient: alpha modes only, one shape
    px = np.array([(i * 16) << 24 | (i * 0x030201) for i in range(16)], dtype=np.uint32)
    L.ora_bc7_box_selection(px.ctypes.data, ctypes.byref(ns), ctypes.byref(s2),
                            ctypes.byref(s3), ctypes.byref(modes))
    assert ns.value == 1 and modes.value == 0b11110000
    # opaque noise: two shapes searched, modes 4 and 5 dropped
    rng = np.random.default_rng(3)
    px = (rng.integers(0, 2**24, 16) | 0xFF000000).astype(np.uint32)
    L.ora_bc7_box_selection(px.ctypes.data, ctypes.byref(ns), ctypes.byref(s2),
                            ctypes.byref(s3), ctypes.byref(modes))
    assert ns.value == 2 and modes.value == 0b11001111


def test_annealing_never_worse_than_q0(oracle):
    """Simulated annealing starts from the quality-0 fit and only keeps
    improvements (Compressor.cpp:583-624): the internal error per block at
    q=50 is at most the q=0 one."""
    img = synth.generate(64, 64, 9)
    blks = synth.blocks(img)
    for b in range(0, blks.shape[0], 3):
        _, s0 = _encode_block(oracle, blks[b], quality=0)
        _, s50 = _encode_block(oracle, blks[b], quality=50, seed=5, block_id=b)
        if s0.path == 2:
            assert s50.best_error <= s0.best_error


def test_decode_matches_spec_except_mode4_index_mode1(oracle):
    """BPTCC::Decompress equals the specification decode except for mode 4
    with index mode 1, where the reference interpolates with the unswapped
    index widths (Decompressor.cpp:263-295)."""
    img = synth.generate(128, 128, 11)
    data, _ = oracle.bc7_compress(img)
    dec = synth.blocks(oracle.bc7_decompress(data, 128, 128))
    blocks = data.reshape(-1, 16)
    for b in range(blocks.shape[0]):
        spec = oracle.bc7_decode_block_spec(blocks[b])
        m = _mode_of(blocks[b])
        idx_mode = (int.from_bytes(blocks[b].tobytes(), "little") >> 7) & 1
        if m == 4 and idx_mode == 1:
            continue
        assert np.array_equal(spec, dec[b]), b


def test_psnr_closed_form(oracle):
    """Image::ComputePSNR (Image.cpp:205-255) on premultiplied RGB."""
    a = np.full((4, 4), 0xFF808080, dtype=np.uint32)
    b = a.copy()
    b[0, 0] = 0xFF808081
    # one channel of one pixel differs by 1 (alpha 1): mse = 1/16
    assert abs(oracle.psnr(a, b) - 10 * np.log10(3 * 255 * 255 * 16)) < 1e-9
    c = a.copy()
    c[:] = 0x00808080  # alpha 0 hides RGB entirely
    d = np.full((4, 4), 0x00000000, dtype=np.uint32)
    assert oracle.premul_sse(c, d) == 0.0


def test_block_premul_err_closed_form(oracle):
    """The guard's block error is Image::ComputePSNR's per-pixel term
    (Base/src/Image.cpp:205-255) times 255^2, exactly."""
    rng = np.random.default_rng(8)
    for _ in range(50):
        a = rng.integers(0, 2**32, 16, dtype=np.uint64).astype(np.uint32)
        b = rng.integers(0, 2**32, 16, dtype=np.uint64).astype(np.uint32)
        want = 0
        for i in range(16):
            pa, pb = int(a[i]) >> 24, int(b[i]) >> 24
            for c in range(3):
                d = pa * ((int(a[i]) >> (8 * c)) & 255) - pb * ((int(b[i]) >> (8 * c)) & 255)
                want += d * d
        assert oracle.block_premul_err(a, b) == want
        assert abs(oracle.premul_sse(a, b) * 255 * 255 - want) <= 1e-6 * max(want, 1)


def _dec_ref(oracle, blk):
    """One block through the reference decoder (BPTCC::Decompress)."""
    return oracle.bc7_decompress(blk, 4, 4).reshape(16)


def test_quality_guard(oracle):
    """With the guard, no block decodes worse than its quality-0 encoding;
    blocks the guard keeps are the unguarded annealed blocks."""
    img = synth.generate(64, 64, 13)
    blks = synth.blocks(img)
    kept = 0
    for b in range(blks.shape[0]):
        o0, _ = _encode_block(oracle, blks[b], quality=0)
        og, sg = _encode_block(oracle, blks[b], quality=50, seed=2, block_id=b, q0_guard=True)
        on, _ = _encode_block(oracle, blks[b], quality=50, seed=2, block_id=b)
        e0 = oracle.block_premul_err(blks[b], _dec_ref(oracle, o0))
        eg = oracle.block_premul_err(blks[b], _dec_ref(oracle, og))
        en = oracle.block_premul_err(blks[b], _dec_ref(oracle, on))
        assert eg <= e0
        if sg.q0_kept:
            assert np.array_equal(og, o0) and en > e0
            kept += 1
        else:
            assert np.array_equal(og, on)
    assert kept > 0


def test_partition_tables_match_reference(oracle):
    """Partition masks, anchors and interpolation weights equal the
    reference's (Shapes.h:23-50, AnchorTables.h:22-45,
    Compressor.cpp:159-168): hash fixture made from the reference text, and
    element by element when the tree is present."""
    L = oracle.lib()
    s2 = np.zeros(64, np.uint16)
    s3 = np.zeros(128, np.uint16)
    a2 = np.zeros(64, np.uint8)
    a3 = np.zeros(128, np.uint8)
    iv = np.zeros(128, np.uint32)
    L.ora_table_partitions(s2.ctypes.data, s3.ctypes.data, a2.ctypes.data, a3.ctypes.data,
                           iv.ctypes.data)
    got = {"shape2": s2, "shape3": s3, "anchor2": a2, "anchor3": a3, "interp": iv}
    fx = json.load(open(os.path.join(HERE, "golden", "bc7_tables.json")))
    for k, v in got.items():
        assert hashlib.sha256(v.tobytes()).hexdigest() == fx[k + "_sha256"], k
    if os.path.exists(os.path.join(REF, "BPTCEncoder", "include", "FasTC", "Shapes.h")):
        from tests.golden.make_golden import partition_tables
        for k, v in partition_tables(REF).items():
            assert np.array_equal(got[k], v), k
    # BC7 specification facts independent of both: subset 0 always holds
    # pixel 0 (the implicit anchor), and each anchor lies in its subset
    s2, s3 = s2.astype(int), s3.astype(int)
    a2, a3 = a2.astype(int), a3.astype(int)
    for sh in range(64):
        assert not (s2[sh] & 1) and (s2[sh] >> a2[sh]) & 1
        m1, m2 = int(s3[2 * sh]), int(s3[2 * sh + 1])
        assert not (m1 & 1) and (m2 & ~m1) == 0
        assert (m1 >> a3[sh]) & 1 and not (m2 >> a3[sh]) & 1
        assert (m2 >> a3[64 + sh]) & 1


# (color bits, alpha bits, p-bit type 0 none / 1 shared / 2 per endpoint,
#  colour index bits, alpha index bits) of the eight BC7 modes (BC7 spec)
_MODES = {0: (4, 0, 2, 3, 0), 1: (6, 0, 1, 3, 0), 2: (5, 0, 0, 2, 0), 3: (7, 0, 2, 2, 0),
          4: (5, 6, 0, 2, 3), 5: (7, 8, 0, 2, 2), 6: (7, 7, 2, 4, 0), 7: (5, 5, 2, 2, 0)}
_W1 = {2: 21, 3: 9, 4: 4}  # weight of index 1 (BC7 spec interpolation tables)


def test_single_color_brute_force(oracle):
    """CompressSingleColor (Compressor.cpp:252-353) against exhaustive
    enumeration: per channel the distance is the minimum over every grid
    pair of |interp(index 1) - value|, the p-bit combination minimises the
    sum of squares (first one on ties) and the endpoints reach the minimum."""
    import ctypes
    L = oracle.lib()
    rng = np.random.default_rng(4)
    cols = [[0, 0, 0, 0], [255, 255, 255, 255], [1, 128, 254, 7]] + \
        [list(rng.integers(0, 256, 4)) for _ in range(25)]
    for mode, (cb, ab, pbt, ib, aib) in _MODES.items():
        for im in ([0, 1] if mode == 4 else [0]):
            nbits_idx = ib if im == 0 else aib
            w = _W1[nbits_idx]
            combos = [(0, 0)] if pbt == 0 else ([(0, 0), (1, 1)] if pbt == 1 else
                                                [(0, 0), (0, 1), (1, 0), (1, 1)])
            for col in cols:
                p = np.array(col, np.float32)
                p1 = np.zeros(4, np.float32)
                p2 = np.zeros(4, np.float32)
                pbc = ctypes.c_int(0)
                err = L.ora_single_color(mode, im, p.ctypes.data, p1.ctypes.data,
                                         p2.ctypes.data, ctypes.byref(pbc))
                best, best_c, best_d = None, None, None
                for ci, (pl, ph) in enumerate(combos):
                    d = []
                    for ch in range(4):
                        bits = cb if ch < 3 else ab
                        val = int(col[ch])
                        if bits == 0:
                            d.append(255 - val)
                            continue
                        pbl, pbh = (pl, ph) if pbt else (-1, -1)
                        lo = np.array([_expand(k, bits, pbl) for k in range(1 << bits)])
                        hi = np.array([_expand(k, bits, pbh) for k in range(1 << bits)])
                        ip = ((64 - w) * lo[:, None] + w * hi[None, :] + 32) >> 6
                        d.append(int(np.abs(ip - val).min()))
                    e = float(sum(x * x for x in d))
                    if best is None or e < best:
                        best, best_c, best_d = e, ci, d
                assert err == best and pbc.value == best_c, (mode, im, col)
                pl, ph = combos[best_c]
                for ch in range(4):
                    bits = cb if ch < 3 else ab
                    if bits == 0:
                        assert p1[ch] == 255 and p2[ch] == 255
                        continue
                    a, b = int(p1[ch]), int(p2[ch])
                    assert a in [_expand(k, bits, pl if pbt else -1) for k in range(1 << bits)]
                    assert b in [_expand(k, bits, ph if pbt else -1) for k in range(1 << bits)]
                    assert abs((((64 - w) * a + w * b + 32) >> 6) - int(col[ch])) == best_d[ch]


def _pbits_equal_per_subset(blk, mode):
    """Whether both endpoints of every subset carry the same p-bit (the p-bits
    follow the endpoint fields: modes 0, 3, 6, 7 at bits 77, 94, 63, 94)."""
    start, nsub = {0: (77, 3), 3: (94, 2), 6: (63, 1), 7: (94, 2)}[mode]
    bits = int.from_bytes(bytes(blk), "little")
    return all(((bits >> (start + 2 * s)) & 1) == ((bits >> (start + 2 * s + 1)) & 1)
               for s in range(nsub))


def test_internal_error_equals_decoded_error(oracle):
    """Under the uniform metric a fit's internal error (its QuantizedError sums,
    Compressor.cpp:538-630) equals the squared error of the packed block as the
    BC7 specification decodes it, wherever the reference's two endpoint quirks
    do not apply:
      * Pack swaps the endpoints of a subset whose anchor index has its top bit
        set but not their p-bits (Compressor.cpp:1149-1170), so with unique
        p-bits (modes 0, 3, 6, 7) the equality holds when both p-bits agree;
      * for modes without p-bits GetPBitCombo returns {0, 0}, not null
        (CompressionMode.h:243-250), so QuantizedError quantises the endpoints
        as if they carried a zero p-bit (RGBAEndpoints.cpp:207-209) while Pack
        writes them without one: mode 2 is left out.
    Mode 1 (shared p-bits) always satisfies it.  A field of Pack's multi-subset
    layout in the wrong place would decode to other colours and break it."""
    from fastc_amd import synth
    rng = np.random.default_rng(21)
    img = synth.generate(64, 64, 9) | np.uint32(0xFF000000)
    blocks = [img[y:y + 4, x:x + 4].reshape(16).copy() for y in range(0, 64, 4)
              for x in range(0, 64, 4)]
    blocks = [b for b in blocks if not (b == b[0]).all()][:60]
    for _ in range(20):
        blocks.append((rng.integers(0, 2**24, 16) | 0xFF000000).astype(np.uint32))
    checked = {m: 0 for m in (0, 1, 3, 6, 7)}
    for px in blocks:
        for mode in checked:
            for slot in ((0, 5, 13) if mode != 6 else (0,)):
                out, err = oracle.bc7_encode_candidate(px, mode, slot)
                if mode != 1 and not _pbits_equal_per_subset(out, mode):
                    continue
                dec = oracle.bc7_decode_block_spec(out)
                sse = sum(int(((int(px[i]) >> (8 * k)) & 255) - ((int(dec[i]) >> (8 * k)) & 255)) ** 2
                          for i in range(16) for k in range(4))
                assert err == sse, (mode, slot, err, sse)
                checked[mode] += 1
    assert checked[1] == 240 and min(checked.values()) >= 20, checked


def test_anneal_point_count(oracle):
    """The oracle's count of annealing QuantizedError point evaluations
    (OptimizeEndpointsForCluster, Compressor.cpp:583-624): none at quality 0;
    with mode 6 alone (one subset of 16 points) a multiple of 16, and at
    least 16 * q for a block whose fit is not exact (a subset anneals for at
    least q steps while its best error stays above 0)."""
    L = oracle.lib()
    rng = np.random.default_rng(3)
    px = (rng.integers(0, 2**24, 16) | 0xFF000000).astype(np.uint32)
    L.ora_anneal_point_count(1)
    oracle.bc7_compress_block(px, quality=0)
    assert L.ora_anneal_point_count(1) == 0
    for q in (1, 7, 30):
        out, st = oracle.bc7_compress_block(px, quality=q, seed=9, block_modes=0x40)
        n = L.ora_anneal_point_count(1)
        assert st.best_error > 0 and n % 16 == 0 and n >= 16 * q, (q, n)
