"""The workloads this framework's speed is measured on.

A case is a dict of plain values; `prepare` makes what a program holds before
the call, `run` makes one pass through the public entry points and `work`
says what a pass cannot do without.  The images are the seeded generator's
(fastc_amd.synth): value noise with alpha ramps and flat blocks, the
distribution the encoders' tests and benchmark use.

BC7 encodes pass a caller-held watermark counter (a device word for batches),
reset before each pass, as a build that has to write the same bytes on every
run does; the process-wide counter would number the flat blocks on from
the previous pass.
"""
import ctypes
import os

import numpy as np
import torch

import fastc_amd
from fastc_amd import batch_workload, synth

DXT1, DXT5, ETC1, BC7 = 0, 1, 2, 3
WATERMARK_START = 0xFFFFFFFF


def listed():
    return [
        # one small texture or the tail of a mip chain while an editor waits:
        # nothing but latency and launches
        {"name": "bc7_q0_64", "kind": "encode", "format": BC7, "width": 64, "height": 64,
         "quality": 0, "learned": False},
        # CompressImageData on a host image at its default quality: the 256 x 256
        # image the reference's command line is tried on, copies both ways included
        {"name": "bc7_q0_256_host", "kind": "host_encode", "format": BC7, "width": 256,
         "height": 256, "quality": 0, "learned": False},
        # a medium texture of odd block counts at the usual annealing quality,
        # with the reference's own search
        {"name": "bc7_q50_508x380", "kind": "encode", "format": BC7, "width": 508, "height": 380,
         "quality": 50, "learned": False},
        # the reference's search on a texture of the largest common size
        {"name": "bc7_q50_4096", "kind": "encode", "format": BC7, "width": 4096, "height": 4096,
         "quality": 50, "learned": False},
        # the learned search on an everyday texture
        {"name": "bc7_learned_1024", "kind": "encode", "format": BC7, "width": 1024,
         "height": 1024, "quality": 50, "learned": True},
        # the benchmark's headline: the learned search at 4096 x 4096
        {"name": "bc7_learned_4096", "kind": "encode", "format": BC7, "width": 4096,
         "height": 4096, "quality": 50, "learned": True},
        # the two DXT formats: a common size, and the largest
        {"name": "dxt1_2048", "kind": "encode", "format": DXT1, "width": 2048, "height": 2048,
         "quality": 0, "learned": False},
        {"name": "dxt5_4096", "kind": "encode", "format": DXT5, "width": 4096, "height": 4096,
         "quality": 0, "learned": False},
        # ETC1 for mobile targets, sides that are no power of two
        {"name": "etc1_2044x1532", "kind": "encode", "format": ETC1, "width": 2044,
         "height": 1532, "quality": 0, "learned": False},
        # loading a compressed texture where the pixels are needed again
        {"name": "decode_bc7_4096", "kind": "decode", "format": BC7, "width": 4096,
         "height": 4096},
        # checking an encode: per-block errors and the total behind the PSNR,
        # on an image whose sides cut through the last blocks
        {"name": "error_bc7_1918x1078", "kind": "error", "format": BC7, "width": 1918,
         "height": 1078},
        # an asset build: textures of uneven sizes with their mip chains, in
        # three formats, planned once and replayed as a graph
        {"name": "batch_32_mips", "kind": "batch", "textures": 32, "min_side": 64,
         "max_side": 1024, "quality": 50, "learned": True},
    ]


def _log_uniform(rng, low, high, step):
    """A multiple of step in [low, high], uniform in its logarithm."""
    v = low * (high / low) ** rng.random()
    return min(high, max(low, int(v / step + 0.5) * step))


def draw(rng):
    kind = rng.choice(["bc7", "bc7", "bc7", "learned", "learned", "simple", "simple", "host",
                       "decode", "error", "batch"])
    if kind == "batch":
        return {"kind": "batch", "textures": _log_uniform(rng, 4, 32, 1), "min_side": 64,
                "max_side": rng.choice([128, 256, 512, 1024]), "quality": rng.choice([0, 8, 50]),
                "learned": rng.random() < 0.5}
    if kind in ("decode", "error"):
        return {"kind": kind, "format": rng.choice([DXT1, DXT5, ETC1, BC7, BC7, BC7]),
                "width": _log_uniform(rng, 61, 4096, 1),
                "height": _log_uniform(rng, 61, 4096, 1)}
    high = 1024 if kind == "host" else 4096
    width, height = _log_uniform(rng, 64, high, 4), _log_uniform(rng, 64, high, 4)
    fmt = BC7 if kind in ("bc7", "learned") else rng.choice(
        [DXT1, DXT5, ETC1] + [BC7] * (kind == "host"))
    quality = rng.choice([0, 8, 20, 50, 50]) if fmt == BC7 else 0
    return {"kind": "host_encode" if kind == "host" else "encode", "format": fmt, "width": width,
            "height": height, "quality": quality, "learned": kind == "learned"}


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _ceil4(n):
    return (n + 3) // 4 * 4


def _upload(img):
    return torch.from_numpy(img.view(np.int32)).cuda()


def _ranker():
    ranker = fastc_amd.Ranker()
    path = os.path.join(os.path.dirname(os.path.abspath(fastc_amd.__file__)), "data",
                        "bc7_ranker.npy")
    ranker.set_params(np.load(path))
    return ranker


def _prepare_encode(case, seed):
    w, h, fmt = case["width"], case["height"], case["format"]
    img = synth.generate(w, h, seed, edges=fmt != BC7)
    state = {"case": case, "wm": ctypes.c_uint32(WATERMARK_START) if fmt == BC7 else None,
             "ranker": _ranker() if case["learned"] else None}
    size = fastc_amd.compressed_size(fmt, w, h)
    if case["kind"] == "host_encode":
        state["img"] = img
        state["out"] = np.zeros(size, dtype=np.uint8)
    else:
        state["img"] = _upload(img)
        state["out"] = torch.zeros(size, dtype=torch.uint8, device="cuda")
    return state


def _prepare_encoded(case, seed):
    """An encoded surface (and its original) of a size whose edge blocks may be cut."""
    w, h, fmt = case["width"], case["height"], case["format"]
    pw, ph = _ceil4(w), _ceil4(h)
    img = synth.generate(pw, ph, seed, edges=fmt != BC7)
    padded = _upload(img)
    enc = torch.zeros(fastc_amd.compressed_size(fmt, w, h), dtype=torch.uint8, device="cuda")
    fastc_amd.compress_device(padded.data_ptr(), enc.data_ptr(), enc.numel(), pw, ph, fmt=fmt,
                              stream=_stream(), wm_counter=ctypes.c_uint32(WATERMARK_START))
    state = {"case": case, "enc": enc}
    if case["kind"] == "decode":
        state["out"] = torch.zeros((h, w), dtype=torch.int32, device="cuda")
    else:
        state["img"] = _upload(np.ascontiguousarray(img[:h, :w]))
        state["errors"] = torch.zeros((ph // 4) * (pw // 4), dtype=torch.int64, device="cuda")
        state["sse"] = torch.zeros(2, dtype=torch.int64, device="cuda")
    return state


def _batch_shapes(case):
    """(format, width, height, opaque) of each texture: power-of-two sides and
    the format mix of batch_workload.make_batch, fixed by the case, so that
    every build of it writes an archive of the same layout."""
    rng = np.random.default_rng(case["textures"] + case["max_side"])
    low, high = int(np.log2(case["min_side"])), int(np.log2(case["max_side"]))
    shapes = []
    for _ in range(case["textures"]):
        w, h = (1 << int(k) for k in rng.integers(low, high + 1, 2))
        opaque = bool(rng.random() < 0.4)
        shapes.append((int(rng.choice([BC7, DXT5, ETC1], p=[0.6, 0.25, 0.15])), w, h, opaque))
    return shapes


def _mip_sizes(w, h):
    sizes = [(w, h)]
    while sizes[-1] != (1, 1):
        w, h = max(1, w // 2), max(1, h // 2)
        sizes.append((w, h))
    return sizes


def _prepare_batch(case, seed):
    # pixels of all levels in one buffer, blocks in another, as an asset
    # build lays its archive out
    surfaces, pixels, in_at, out_at = [], [], 0, 0
    for i, (fmt, w, h, opaque) in enumerate(_batch_shapes(case)):
        top = synth.generate(w, h, ((seed % 1000003) << 20) + i)
        if opaque:
            top = top | np.uint32(0xFF000000)
        for level in map(batch_workload.pad4, batch_workload.mip_chain(top)):
            h, w = level.shape
            surfaces.append((fmt, in_at, out_at, w, h))
            pixels.append(level.reshape(-1))
            in_at += w * h * 4
            out_at += (fastc_amd.compressed_size(fmt, w, h) + 15) // 16 * 16
    img = _upload(np.concatenate(pixels))
    out = torch.zeros(out_at, dtype=torch.uint8, device="cuda")
    wm = torch.full((1,), -1, dtype=torch.int32, device="cuda")
    batch = fastc_amd.Batch(
        [(fmt, img.data_ptr() + i, out.data_ptr() + o, w, h) for fmt, i, o, w, h in surfaces],
        quality=case["quality"], seed=1, ranker=_ranker() if case["learned"] else None,
        wm_counter_ptr=wm.data_ptr())
    return {"case": case, "batch": batch, "img": img, "out": out, "wm": wm}


def prepare(case, seed):
    if case["kind"] == "batch":
        return _prepare_batch(case, seed)
    if case["kind"] in ("decode", "error"):
        return _prepare_encoded(case, seed)
    return _prepare_encode(case, seed)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "batch":
        state["wm"].fill_(-1)
        state["batch"].run(use_graph=True, stream=_stream())
        return state["out"], state["wm"]
    w, h, fmt = case["width"], case["height"], case["format"]
    if kind == "decode":
        fastc_amd.decompress_device(state["enc"].data_ptr(), state["out"].data_ptr(), w, h,
                                    fmt=fmt, stream=_stream())
        return state["out"]
    if kind == "error":
        fastc_amd.block_error_device(state["img"].data_ptr(), state["enc"].data_ptr(), w, h,
                                     state["sse"].data_ptr(), state["errors"].data_ptr(),
                                     fmt=fmt, stream=_stream())
        return state["errors"], state["sse"]
    wm = state["wm"]
    if wm is not None:
        wm.value = WATERMARK_START
    if kind == "host_encode":
        fastc_amd.compress(state["img"], fmt=fmt, quality=case["quality"], seed=1,
                           out=state["out"], wm_counter=wm, ranker=state["ranker"])
    else:
        out = state["out"]
        fastc_amd.compress_device(state["img"].data_ptr(), out.data_ptr(), out.numel(), w, h,
                                  fmt=fmt, quality=case["quality"], seed=1, stream=_stream(),
                                  wm_counter=wm, ranker=state["ranker"])
    return state["out"] if wm is None else (state["out"], wm.value)


# Operations of the searches per 4 x 4 block.  BoxSelection scores the 16
# texels under 64 two-subset and 64 three-subset shapes; a score projects a
# texel, interpolates and squares in four channels.  At quality 50 the
# annealing evaluates about 18,600 texels per block of the generator's images
# in the reference's search and about 1,160 in the learned one; the ranker is
# a 64-256-256-512 network.
_OPS_PER_SCORE = 24
_BOX_SCORES = 2 * 64 * 16
_FIT_SCORES = 16 * 16
_ANNEAL_SCORES = {False: 18600 / 50, True: 1160 / 50}
_RANKER_FLOPS = 2 * (64 * 256 + 256 * 256 + 256 * 512)
_DXT_OPS = 16 * 4 * _OPS_PER_SCORE
_ETC1_OPS = 2 * 16 * 8 * 4 * 8  # two flips, 8 intensity tables, 4 selectors


def _encode_work(fmt, blocks, quality, learned):
    if fmt == BC7:
        scores = (4 * 16 if learned else _BOX_SCORES + _FIT_SCORES)
        scores += quality * _ANNEAL_SCORES[learned]
        flops = _OPS_PER_SCORE * scores + (_RANKER_FLOPS if learned else 0)
    else:
        flops = _ETC1_OPS if fmt == ETC1 else _DXT_OPS
    return {"bytes": blocks * (64 + fastc_amd.BLOCK_BYTES[fmt]), "flops": blocks * flops}


def work(case):
    if case["kind"] == "batch":
        total = {"bytes": 0, "flops": 0}
        for fmt, w, h, _ in _batch_shapes(case):
            for lw, lh in _mip_sizes(w, h):
                one = _encode_work(fmt, (_ceil4(lw) // 4) * (_ceil4(lh) // 4), case["quality"],
                                   case["learned"])
                total = {k: total[k] + one[k] for k in total}
        return total
    w, h, fmt = case["width"], case["height"], case["format"]
    blocks = (_ceil4(w) // 4) * (_ceil4(h) // 4)
    if case["kind"] == "decode":
        return {"bytes": blocks * fastc_amd.BLOCK_BYTES[fmt] + w * h * 4, "flops": w * h * 12}
    if case["kind"] == "error":
        return {"bytes": blocks * (fastc_amd.BLOCK_BYTES[fmt] + 8) + w * h * 4,
                "flops": w * h * 24}
    return _encode_work(fmt, blocks, case["quality"], case["learned"])
