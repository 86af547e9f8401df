"""The detection chain's outputs bit for bit.

A detection is a comparison with a threshold, so a kernel that rounds otherwise
moves cells that lie on it: on 16 x 128 x 9000 cubes an equally exact transform
flips one cell in two hundred cubes.  The digests pin the compressed cube, the
power, the averages and the detections on gfx950 over the block sizes of the
pulse compression (1024 to 16384 points, out of place and in place) and the
Doppler sizes of the fused and of the separate pulse-axis and CFAR kernels.
Inputs are whole numbers over 64 from numpy's generator.
"""
import hashlib
import json
import os

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "radar_bits.json")

FUSED = [  # C, P, S, L, nd, tpc
    (2, 34, 1000, 64, 32, "valid"),       # blocks of 1024
    (1, 130, 3306, 128, 128, "valid"),    # 1024, five to a row
    (2, 66, 2000, 100, 64, "valid"),      # 2048
    (1, 18, 5003, 487, 16, "valid"),      # 2048, three to a row
    (2, 128, 4000, 500, 128, "same"),     # 4096
    (1, 128, 9000, 1000, 128, "valid"),   # 4096, three to a row
    (1, 64, 8000, 1000, 64, "none"),      # 8192
    (1, 40, 20000, 3000, 64, "same"),     # 8192, four to a row
    (1, 20, 16000, 9000, 32, "valid"),    # 16384
    (1, 8, 1500, 200, 8, "same"),
    (1, 200, 2500, 300, 256, "same"),     # separate pulse-axis pass and CFAR
    (1, 900, 1200, 100, 1024, "valid"),
]
STAGES = [  # C, P, S, L
    (2, 20, 1000, 64), (2, 77, 5003, 487), (1, 33, 7000, 875), (1, 16, 9000, 1000), (1, 100, 2700, 300),
]


def _inputs(seed, C, P, S, L):
    rng = np.random.default_rng(seed)
    c64 = lambda *s: (rng.integers(-256, 257, s + (2,)) / 64).astype(np.float32).view(np.complex64)[..., 0]  # noqa: E731
    return torch.from_numpy(c64(C, P, S)).cuda(), torch.from_numpy(c64(L)).cuda()


def _digest(t):
    return hashlib.sha256(t.contiguous().cpu().numpy().tobytes()).hexdigest()[:16]


def fused(mx, C, P, S, L, nd, tpc):
    x, w = _inputs(S, C, P, S, L)
    pipe = mx.FusedRadarPipeline(C, P, S, L, nd=nd, tpc=tpc, pfa=0.02, want_pow=True, want_ba=True)
    pipe.step(x, w)
    assert int(pipe.dets.sum()) > 0
    return {k: _digest(t) for k, t in (("y", pipe.y), ("pow", pipe.pw), ("ba", pipe.ba), ("dets", pipe.dets))}


def stages(mx, C, P, S, L):
    x, w = _inputs(S, C, P, S, L)
    pipe = mx.RadarPipeline(P, S, L, C)
    pipe.GetInputView()[:, :, :S].copy_(x)
    pipe.GetwaveformView()[:L].copy_(w)
    pipe.run()
    return {k: _digest(t) for k, t in (("w", pipe.waveformView), ("y", pipe.inputView), ("tpc", pipe.tpcView),
                                       ("pow", pipe.xPow), ("ba", pipe.ba), ("dets", pipe.dets))}


@pytest.fixture(scope="module")
def mx():
    import matx_amd
    return matx_amd


@pytest.fixture(scope="module")
def bits():
    with open(GOLDEN) as f:
        return json.load(f)


@pytest.mark.parametrize("case", FUSED, ids=str)
def test_fused_pipeline_bits(mx, bits, case):
    assert fused(mx, *case) == bits[f"fused {case}"]


@pytest.mark.parametrize("case", STAGES, ids=str)
def test_stage_pipeline_bits(mx, bits, case):
    assert stages(mx, *case) == bits[f"stages {case}"]
