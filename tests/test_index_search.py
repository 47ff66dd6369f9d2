"""The annealing's and BoxSelection's index search at its edges: endpoint
distances up to the largest (black to white in all four channels), where the
quotient that names the neighbouring indices has the least room."""
import ctypes
import os
import subprocess

import numpy as np
import pytest


def _contrast_image(w, h, levels, seed):
    """Texels whose channels take only the given levels: the subsets' axes
    are then as long as they get and many projections fall on an index."""
    rng = np.random.default_rng(seed)
    c = np.asarray(levels, dtype=np.uint32)[rng.integers(0, len(levels), (h, w, 4))]
    return np.ascontiguousarray(c[..., 0] | c[..., 1] << 8 | c[..., 2] << 16 | c[..., 3] << 24)


@pytest.mark.parametrize("kf", [3, 7, 15])
def test_index_arithmetic(kf):
    """floor and ceil of d kf / l by the encoder's float arithmetic (a
    correctly rounded 1 / (64 l), the product clamped to [0, 1], truncations
    of fma(u, kf, 1.9e-6) and fma(u, kf, 1 - 1.9e-6)) against integers, at the
    steps of both functions: the smallest and largest l and a sample."""
    top = 4 * 255 * 255
    rng = np.random.default_rng(kf)
    ls = np.unique(np.concatenate([np.arange(1, 3000), np.arange(top - 3000, top + 1),
                                   rng.integers(1, top, 20000)]))
    rl = (1.0 / (64.0 * ls)).astype(np.float32)
    slack = np.float32(1.9e-6)
    rest = np.float32(1.0) - slack
    for k in range(kf + 1):
        for o in (-2, -1, 0, 1, 2):
            d = k * ls // kf + o
            ok = (d >= 0) & (d <= ls)
            u = np.clip((64 * d).astype(np.float32) * rl, np.float32(0), np.float32(1))
            # u * kf is exact in double; the sum rounds once to float
            j1 = (u.astype(np.float64) * kf + np.float64(slack)).astype(np.float32).astype(int)
            j2 = (u.astype(np.float64) * kf + np.float64(rest)).astype(np.float32).astype(int)
            assert np.array_equal(j1[ok], (d * kf // ls)[ok])
            assert np.array_equal(j2[ok], (-(-d * kf // ls))[ok])


def test_index_arithmetic_of_the_encoder(tmp_path):
    """The encoder's own header (bc7_index.h) compiled for the host: every
    distance, every start of the reciprocal within 2 ulp, every step."""
    here = os.path.dirname(os.path.abspath(__file__))
    exe = str(tmp_path / "index_test")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off",
                    os.path.join(here, "cpp", "index_test.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0 and int(r.stdout.split()[0]) > 260100 * 145, r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("levels", [(0, 255), (0, 1, 254, 255), (0, 85, 170, 255)])
@pytest.mark.parametrize("opaque", [False, True])
@pytest.mark.parametrize("metric", [0, 1])
def test_contrast_bit_exact(fh, oracle, levels, opaque, metric):
    img = _contrast_image(48, 32, levels, len(levels))
    if opaque:
        img |= np.uint32(0xFF000000)
    for q in (0, 8):
        print(f"contrast {levels} opaque={opaque} metric={metric} q={q}", flush=True)
        ref, _ = oracle.bc7_compress(img, quality=q, seed=5, q0_guard=True, metric=metric)
        got = fh.compress(img, quality=q, seed=5, wm_counter=ctypes.c_uint32(0xFFFFFFFF),
                          metric=metric)
        bad = np.nonzero((got.reshape(-1, 16) != ref.reshape(-1, 16)).any(axis=1))[0]
        assert bad.size == 0, f"{bad.size} blocks differ, first {bad[:8]}"
