"""The generation step's fused Dense layers (m3_step_gemm): each against torch with the
separate kernels' rounding points, at the edges of the 16-row and 16-column tiles and of
the tile choice, their argument checks, and a stack's step with them against the step
with library GEMMs."""
import numpy as np
import pytest


def _lib():
    from mamba3_rocm import _lib
    return _lib.load()


def test_argument_checks():
    lib = _lib()
    p = 4096          # a non-null aligned address that is never read: every call below is refused
    f = lambda *a: lib.m3_step_gemm(*a, 1e-6, None)  # noqa: E731
    assert f(4, p, p, p, p, p, p, p, 1, 256, 256) == 1            # M3_E_ARG: no such mode
    assert f(0, p, p, p, p, p, p, p, 1, 300, 256) == 3            # M3_E_UNSUPPORTED: K
    assert f(0, p, p, p, p, p, p, p, 1, 256, 260) == 3            # N not a multiple of 8
    assert f(2, p, p, p, p, p, p, p, 1, 256, 512) == 3            # the gate's product is square
    assert f(0, p, p, p, None, p, p, p, 1, 256, 256) == 1         # no scale
    assert f(2, p, p, p, None, None, None, p, 1, 256, 256) == 1   # no bias
    assert f(0, p + 4, p, p, p, p, p, p, 1, 256, 256) == 2        # M3_E_ALIGN
    assert f(0, p, p, p, p, p, p, p, 0, 256, 256) == 0            # empty batch
    rows = lib.m3_step_rows_max
    assert rows(768, 1536, 3432) >= 64 and rows(256, 512, 1336) >= 64 and rows(1024, 2048, 4480) >= 64
    assert rows(800, 1600, 3528) == 0 and rows(768, 768, 3432) == 0 and rows(2048, 4096, 8704) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("K,N", [(256, 264), (512, 512), (768, 3432), (1024, 1024)])
@pytest.mark.parametrize("M", [1, 15, 16, 17, 33, 64, 65, 129, 257])
def test_products(M, K, N):
    import torch
    lib = _lib()
    g = torch.Generator(device="cuda")
    g.manual_seed(M * K + N)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    bf = lambda t: t.to(torch.bfloat16)  # noqa: E731
    r64 = lambda t: bf(t.float()).double()  # noqa: E731
    st = torch.cuda.current_stream().cuda_stream
    p = lambda t: None if t is None else t.data_ptr()  # noqa: E731

    def call(mode, x, wt, out, scale, bias, b2, skip, k, n, eps):
        assert lib.m3_step_gemm(mode, p(x), p(wt), p(out), p(scale), p(bias), p(b2), p(skip), M, k, n, eps, st) == 0
        torch.cuda.synchronize()
        return out.double()

    # a result is rounded to bf16 (2^-9 of it at most, 1.2e-3 in the 2-norm); an operand that
    # float32 and float64 statistics round differently moves by one bf16 ulp
    rel = lambda a, b: float((a - b).norm() / b.norm())  # noqa: E731
    x, wt, sc, bi = rand(M, K) + 0.5, bf(rand(K, N) / K ** 0.5), 1 + 0.1 * rand(K), 0.1 * rand(K)
    xn = torch.nn.functional.layer_norm(x.double(), (K,), sc.double(), bi.double(), 1e-6)
    got = call(0, x, wt, torch.empty(M, N, device="cuda", dtype=torch.bfloat16), sc, bi, None, None, K, N, 1e-6)
    assert rel(got, r64(xn) @ wt.double()) < 2.5e-3

    if K <= 512:
        y, wo = bf(rand(M, 2 * K)), bf(rand(2 * K, K) / K ** 0.5)
        ns = 1 + 0.1 * rand(2 * K)
        rs = r64(torch.rsqrt((y.double() ** 2).mean(-1, keepdim=True) + 1e-6))
        v = r64(r64(r64(y.double() * rs) * ns.double()) @ wo.double())
        got = call(1, y, wo, torch.empty(M, K, device="cuda", dtype=torch.bfloat16), ns, None, None, None, 2 * K, K, 1e-6)
        want = torch.nn.functional.gelu(v, approximate="tanh")
        assert rel(got, want) < 4e-3                      # two roundings

    gg, w2, b2, skip = bf(rand(M, K)), bf(rand(K, K) / K ** 0.5), bf(0.1 * rand(K)), rand(M, K)
    for mode in (2, 3):
        got = call(mode, gg, w2, torch.empty(M, K, device="cuda"), None, None, b2, skip, K, K, 0.0)
        v = gg.double() if mode == 2 else r64(torch.nn.functional.gelu(gg.double(), approximate="tanh"))
        gate = r64(v * r64(torch.sigmoid(r64(v @ w2.double().t() + b2.double()))))
        assert rel(got, skip.double() + gate) < 1.5e-3    # the float32 residual carries most of it


@pytest.mark.gpu
@pytest.mark.parametrize("d_model", [256, 512, 768, 1024])
@pytest.mark.parametrize("B", [31, 32, 33, 64, 100])
def test_stack_step_equals_library_route(d_model, B):
    import torch
    from mamba3_rocm import Mamba3Stack
    from mamba3_rocm.stack import init_params
    p = init_params(96, d_model, 3, 11, "cuda")
    for lp in p["layers"]:                            # norms and biases that are not ones and zeros
        for k in ("ln_scale", "ln_bias", "out2_b"):
            lp[k] = lp[k] + 0.1 * torch.randn_like(lp[k])
        lp["mixer"]["out_norm"] = lp["mixer"]["out_norm"] + 0.1 * torch.randn_like(lp["mixer"]["out_norm"])
    s = Mamba3Stack(p, d_model, dtype=torch.bfloat16)
    fused, s.step_rows_max = s.step_rows_max, 0
    assert fused >= 64
    ids = torch.from_numpy(np.random.default_rng(B).integers(0, 96, (B, 5))).cuda()
    _, a = s.prefill(ids)
    b = [tuple(t.clone() for t in c) for c in a]
    nxt = ids[:, 0]
    for _ in range(3):
        s.step_rows_max = fused
        la, _ = s.step(nxt, a)
        s.step_rows_max = 0
        lb, _ = s.step(nxt.reshape(B, 1), b)
        assert tuple(la.shape) == (B, 96) and torch.equal(la, lb)
        nxt = lb.argmax(-1)
    assert all(torch.equal(ta, tb) for ca, cb in zip(a, b) for ta, tb in zip(ca, cb))
    s.step_rows_max = fused
    with pytest.raises(ValueError):
        s.step(nxt, [tuple(t.double() for t in c) for c in a])
