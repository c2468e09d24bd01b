"""The final carry is written whole by every scan kernel: its buffers aren't cleared first."""
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("io", ["bf16", "f32"])
@pytest.mark.parametrize("B,L,H,N,P,R", [(1, 1, 2, 128, 64, 32), (2, 65, 3, 128, 64, 64), (1, 3000, 2, 128, 64, 32),
                                         (1, 700, 2, 64, 64, 16), (1, 130, 2, 64, 32, 16), (2, 70, 3, 48, 24, 8),
                                         (1, 40, 2, 16, 16, 3), (0, 65, 3, 128, 64, 32)])
def test_final_carry_written_whole(io, B, L, H, N, P, R):
    import torch
    from mamba3_rocm import mamba3_siso_hip_carry
    dt = torch.bfloat16 if io == "bf16" else torch.float32
    g = torch.Generator(device="cuda")
    g.manual_seed(L)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    args = (rand(B, L, H, N).to(dt), rand(B, L, H, N).to(dt), rand(B, L, H, P).to(dt), -rand(B, H, L).abs(),
            rand(B, H, L).abs(), rand(B, H, L).to(dt), rand(H, N), rand(H, N), rand(B, L, H, R))
    shapes = [(B, H, R), (B, H, P, N), (B, H, N), (B, H, P)]
    # leave NaN in the blocks that the carry's allocations take next
    poison = [torch.full(s, float("nan"), device="cuda") for s in shapes * 4]
    del poison
    _, fin = mamba3_siso_hip_carry(*args)
    for t, s in zip(fin, shapes):
        assert tuple(t.shape) == s and bool(torch.isfinite(t).all())
