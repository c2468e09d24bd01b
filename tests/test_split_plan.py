"""The sequence split's choice of segments: when it splits, the workspace it asks for, and
the split result against one pass at the rule's edges (segments of one kernel chunk, a
ragged last segment, d_state 64, few tokens)."""
import numpy as np
import pytest

from oracle import inputs as I


def _lib():
    from mamba3_rocm import _lib
    return _lib.load()


def test_plan_workspace():
    lib = _lib()
    plan, ws = lib.m3_scan_split_plan_bytes, lib.m3_chunk_scan_ws_bytes
    for io in (0, 1):
        assert plan(1, 127, 2, 128, 64, 32, 64, io) == 0              # under two segments of 64 tokens
        assert plan(1, 8192, 129, 128, 64, 32, 64, io) == 0           # over half the compute units
        assert plan(1, 8192, 8, 128, 64, 32, 48, io) == 0             # generic kernel
        assert plan(1, 8192, 8, 32, 32, 8, 64, io) == 0               # no state-only pass
        assert plan(2, 1024, 8, 64, 64, 16, 64, io) > 0               # d_state 64
        for B, L, H in ((1, 613, 24), (4, 1500, 24), (1, 32768, 32), (1, 4096, 2), (4, 12288, 24), (3, 5000, 8)):
            p, w = plan(B, L, H, 128, 64, 32, 64, io), ws(B, L, H, 128, 64, 32, 64, io)
            assert w >= p, (B, L, H)                                  # the public size holds the choice
            slots = 1024 * (2 * (64 * 128 + 128 + 64 + 32) + 1) * 4 + 9 * 256
            assert p <= slots                                         # at most 1024 carry slots
    assert plan(4, 1500, 24, 128, 64, 32, 64, 1) == 0                 # 96 pairs: one pass is faster


@pytest.mark.gpu
@pytest.mark.parametrize("bf16", [True, False])
@pytest.mark.parametrize("B,L,H,N,P,R", [(1, 1024, 16, 64, 64, 16), (2, 1025, 4, 64, 32, 16), (1, 700, 3, 128, 64, 32),
                                         (1, 4097, 24, 128, 64, 64), (1, 833, 1, 128, 64, 32)])
def test_split_equals_one_pass(B, L, H, N, P, R, bf16):
    import torch
    from mamba3_rocm import mamba3_siso_hip_carry, _lib as m3lib
    io = m3lib.DTYPE_BF16 if bf16 else m3lib.DTYPE_F32
    assert _lib().m3_scan_split_plan_bytes(B, L, H, N, P, R, 64, io) > 0
    d = I.scan_inputs(B, L, H, N, P, R, seed=L, bf16=bf16)
    dt = torch.bfloat16 if bf16 else torch.float32
    t = {k: torch.from_numpy(v).cuda() for k, v in d.items()}
    args = [t[k].to(dt) if k in "QKVZ" else t[k] for k in ("Q", "K", "V", "ADT", "DT", "Trap", "Q_bias", "K_bias",
                                                           "Angles", "D", "Z")]
    g = np.random.default_rng(L)
    carry = tuple(torch.from_numpy(g.standard_normal(s).astype(np.float32)).cuda()
                  for s in ((B, H, R), (B, H, P, N), (B, H, N), (B, H, P)))
    a, (_, ha, ka, va) = mamba3_siso_hip_carry(*args, initial_carry=carry)
    b, (_, hb, kb, vb) = mamba3_siso_hip_carry(*args, initial_carry=carry, seq_split=False)
    # the carries are float32 on both paths; bf16 operands are rounded from states that
    # differ by float32 rounding, so a few of them differ by one bf16 ulp (2^-8)
    rel = lambda x, y: float((x.float() - y.float()).norm() / y.float().norm())  # noqa: E731
    tol = 4e-3 if bf16 else 5e-6
    assert rel(a, b) < tol and rel(ha, hb) < tol, (rel(a, b), rel(ha, hb))
    assert rel(ka, kb) < 1e-5 and torch.equal(va, vb)
