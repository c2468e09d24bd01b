"""Float32 I/O contracts on bf16 matrix cores with every operand split in three bf16
parts: the result has float32 accuracy, at the edges of the kernel's 32-token chunk and
16-row tiles, for operands of very different magnitude, and in the carry it leaves."""
import numpy as np
import pytest
import torch

from oracle import inputs as I
from oracle import mamba3_ref as M

pytestmark = pytest.mark.gpu

# Each product of two split operands drops terms below 2^-24 of it (random sign), and an
# output is a float32 sum of at most 128 + 32 products: sqrt(160) 2^-24 = 7.5e-7 in the
# 2-norm.
REL = 7.5e-7


def _rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("N,P,R,L", [(128, 64, 32, 1), (128, 64, 32, 31), (128, 64, 32, 33), (128, 64, 64, 47),
                                     (64, 64, 16, 65), (64, 64, 32, 16), (64, 32, 16, 49), (32, 32, 8, 96),
                                     (32, 64, 8, 17)])
@pytest.mark.parametrize("spread", [1.0, 1e4])
def test_float32_accuracy(N, P, R, L, spread):
    from mamba3_rocm import mamba3_siso_hip_carry
    B, H = 2, 2
    d = I.scan_inputs(B, L, H, N, P, R, seed=L + N)
    if spread != 1.0:      # columns of Q and rows of V over eight decades, products of order one
        s = np.geomspace(1.0 / spread, spread, N).astype(np.float32)
        d["Q"], d["K"] = d["Q"] * s, d["K"] / s
        d["V"] = d["V"] * np.geomspace(1.0 / spread, spread, L).astype(np.float32)[None, :, None, None]
        d["Q_bias"], d["K_bias"] = d["Q_bias"] * s, d["K_bias"] / s
    t = [torch.from_numpy(d[k]).cuda() for k in ("Q", "K", "V", "ADT", "DT", "Trap", "Q_bias", "K_bias", "Angles", "D",
                                                 "Z")]
    y, (_, ssm, k, v) = mamba3_siso_hip_carry(*t, chunk_size=32, seq_split=False)
    ref = M.mamba3_ssd_chunked_batched(*(d[k] for k in ("Q", "K", "V", "ADT", "DT", "Trap", "Angles", "Q_bias",
                                                        "K_bias", "D", "Z")), chunk_size=32)
    # rope turns pairs of columns of neighbouring magnitude, so a row's largest product
    # sets the scale of its rounding: compare rows by their own norm
    err = np.linalg.norm(y.cpu().numpy() - ref, axis=-1) / np.linalg.norm(ref, axis=-1).clip(1e-30)
    assert float(np.sqrt(np.mean(err ** 2))) < REL * (1 if spread == 1.0 else 8), err.max()
    assert _rel(v.cpu().numpy(), d["V"][:, -1]) == 0.0
    assert np.isfinite(ssm.cpu().numpy()).all()
