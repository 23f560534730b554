"""GPU tests of the surrogate network kernels (pr_mlp_*) against the CPU FP64 oracle.

* the BF16 matrix-core product in all four operand layouts, ragged sizes, bias and GELU
  epilogue, against float64 products of the same bf16 values;
* forward, loss and backward of a 23-64-64-22 network against torch CPU float64 autograd
  (bf16 rounding of weights, inputs and activations bounds the agreement);
* Adam against its float64 closed form.
"""
import numpy as np
import pytest

from oracle import mlp_oracle as mo

pytestmark = pytest.mark.gpu


def _bf16(t):
    import torch
    return torch.as_tensor(np.asarray(t, np.float32)).to(torch.bfloat16)


@pytest.mark.parametrize("a_kfast,b_kfast", [(True, False), (True, True), (False, False), (False, True)])
@pytest.mark.parametrize("M,N,K", [(77, 45, 50), (128, 64, 256), (5, 130, 23)])
def test_gemm_layouts(gpu, a_kfast, b_kfast, M, N, K):
    import torch
    from pelelmex_amd import surrogate as sg
    rng = np.random.default_rng(M * 1000 + N + K)
    A = rng.normal(size=(M, K)).astype(np.float32)
    B = rng.normal(size=(K, N)).astype(np.float32)
    bias = rng.normal(size=N).astype(np.float32)
    Ab, Bb = mo.bf16_round(A), mo.bf16_round(B)
    ref = Ab @ Bb + bias
    # store A as [M, K] (k fastest) or [K, M] (m fastest); B as [K, N] or [N, K]
    Ad = (_bf16(A) if a_kfast else _bf16(A.T.copy())).to(gpu).contiguous()
    Bd = (_bf16(B.T.copy()) if b_kfast else _bf16(B)).to(gpu).contiguous()
    sam, sak = (K, 1) if a_kfast else (1, M)
    sbk, sbn = (1, K) if b_kfast else (N, 1)
    C = torch.full((M, N), float("nan"), dtype=torch.float32, device=gpu)
    Z = torch.full((M, N), float("nan"), dtype=torch.float32, device=gpu)
    Cb = torch.zeros((M, N), dtype=torch.bfloat16, device=gpu)
    bd = torch.as_tensor(bias).to(gpu)
    sg.gemm(M, N, K, Ad, sam, sak, Bd, sbk, sbn, bias=bd, gelu=True, Cf=C, ldc=N, Cb=Cb, ldcb=N, Z=Z, ldz=N)
    torch.cuda.synchronize()
    scale = np.abs(Ab) @ np.abs(Bb) + np.abs(bias)
    z = Z.cpu().numpy()
    assert np.all(np.abs(z - ref) <= 2e-6 * scale + 1e-6)
    import torch.nn.functional as F
    g = F.gelu(torch.as_tensor(ref)).numpy()
    assert np.all(np.abs(C.cpu().numpy() - g) <= 2e-6 * scale + 1e-5)
    assert np.all(np.abs(Cb.float().cpu().numpy() - g) <= 1e-2 * np.abs(g) + 1e-5 * scale + 1e-5)
    # accumulate mode adds the raw product
    C2 = torch.ones((M, N), dtype=torch.float32, device=gpu)
    sg.gemm(M, N, K, Ad, sam, sak, Bd, sbk, sbn, Cf=C2, ldc=N, accumulate=True)
    torch.cuda.synchronize()
    assert np.all(np.abs(C2.cpu().numpy() - (1.0 + Ab @ Bb)) <= 2e-6 * scale + 1e-6)


def test_forward_backward_against_autograd(gpu):
    import torch
    from pelelmex_amd import surrogate as sg
    dims = [23, 64, 64, 22]
    mlp = sg.MLP(dims, device=gpu, seed=3)
    rng = np.random.default_rng(4)
    for b in mlp.b:
        b.copy_(torch.as_tensor(rng.normal(0, 0.1, b.numel()).astype(np.float32)))
    B = 300
    X = rng.normal(size=(B, 23)).astype(np.float32)
    T = rng.normal(size=(B, 22)).astype(np.float32)
    Xd = _bf16(X).to(gpu).contiguous()
    Td = torch.as_tensor(T).to(gpu)
    out = mlp.forward(Xd, keep=True)
    loss, dY = mlp.mse(out, Td)
    mlp.backward(dY)
    torch.cuda.synchronize()
    Wr = [mo.bf16_round(w.cpu().numpy()) for w in mlp.W]
    br = [b.cpu().numpy().astype(np.float64) for b in mlp.b]
    Xr = mo.bf16_round(X)
    ref_out = mo.forward(Wr, br, Xr, bf16_activations=True)
    np.testing.assert_allclose(out.cpu().numpy(), ref_out, rtol=0, atol=1e-3 * np.abs(ref_out).max())
    l_ref, gW_ref, gb_ref = mo.loss_and_grads(Wr, br, Xr, T)
    assert abs(float(loss.item()) - l_ref) <= 1e-2 * l_ref
    for l in range(len(dims) - 1):
        for got, ref in ((mlp.gW[l].cpu().numpy(), gW_ref[l]), (mlp.gb[l].cpu().numpy(), gb_ref[l])):
            rel = np.linalg.norm(got - ref) / np.linalg.norm(ref)
            cos = np.sum(got * ref) / (np.linalg.norm(got) * np.linalg.norm(ref))
            assert rel <= 3e-2 and cos >= 0.999, (l, rel, cos)


def test_adam_against_closed_form(gpu):
    import torch
    from pelelmex_amd import surrogate as sg
    rng = np.random.default_rng(5)
    dims = [23, 40, 22]
    mlp = sg.MLP(dims, device=gpu, seed=1)
    p0 = [w.cpu().numpy().astype(np.float64) for w in mlp.W + mlp.b]
    grads = [rng.normal(size=w.shape).astype(np.float32) for w in mlp.W + mlp.b]
    for g, t in zip(grads, mlp.gW + mlp.gb):
        t.copy_(torch.as_tensor(g))
    mlp.adam(lr=1e-2)
    for g, t in zip(grads, mlp.gW + mlp.gb):
        t.copy_(torch.as_tensor(-0.5 * g))
    mlp.adam(lr=1e-2)
    torch.cuda.synchronize()
    for k, (p, g) in enumerate(zip(p0, grads)):
        m = np.zeros_like(p)
        v = np.zeros_like(p)
        p1, m, v = mo.adam(p, g.astype(np.float64), m, v, 1, 1e-2)
        p2, m, v = mo.adam(p1, -0.5 * g.astype(np.float64), m, v, 2, 1e-2)
        got = (mlp.W + mlp.b)[k].cpu().numpy()
        np.testing.assert_allclose(got, p2, rtol=1e-5, atol=1e-6)
    # the bf16 copies follow the fp32 parameters
    for w, wb in zip(mlp.W, mlp.Wb):
        np.testing.assert_array_equal(wb.float().cpu().numpy(), mo.bf16_round(w.cpu().numpy()).astype(np.float32))


def test_hidden_layer_forward_kernel_bits(gpu):
    """pr_surrogate_forward (the learned path's forward: the tiled 128 x 128 kernel with
    transposed weights for the hidden layers) gives the bits of the same network run layer by
    layer through pr_mlp_gemm, on a row count that is not a multiple of the tile."""
    import torch
    from pelelmex_amd import surrogate as sg
    from pelelmex_amd.reactor import Reactor
    model = sg.load(sg.WEIGHTS)
    dims = [int(d) for d in model["dims"]]
    mlp = sg.MLP(dims, device=gpu)
    mlp.set_flat_params(torch.as_tensor(model["params"], dtype=torch.float32))
    r = Reactor.create("ReactorCvode", "drm19", {"ode.rtol": 1e-10, "ode.atol": 1e-10})
    r.init(2, 1)
    sg.attach(r, model)
    g = torch.Generator(device="cpu").manual_seed(3)
    X = (torch.randn((1000, dims[0]), generator=g) * 1.5).to(torch.bfloat16).to(gpu)
    Y1 = r.surrogate_forward(X)
    Y2 = mlp.forward(X)
    torch.cuda.synchronize()
    assert torch.isfinite(Y1).all()
    assert torch.equal(Y1, Y2)
    r.close()


# gradients' products: K split over a block's waves from 256 on when it is the longest side; the
# smallest split, ragged tiles and K steps, odd extents and strides, both sides of 64 x 64
@pytest.mark.parametrize("a_kfast,b_kfast", [(True, False), (True, True), (False, False), (False, True)])
@pytest.mark.parametrize("M,N,K", [(255, 33, 256), (23, 256, 4096), (256, 22, 1031), (1, 1, 511), (34, 66, 520)])
def test_gemm_long_k(gpu, a_kfast, b_kfast, M, N, K):
    import torch
    from pelelmex_amd import surrogate as sg
    rng = np.random.default_rng(M + N + K)
    A, B = rng.normal(size=(M, K)).astype(np.float32), rng.normal(size=(K, N)).astype(np.float32)
    Ab, Bb = mo.bf16_round(A), mo.bf16_round(B)
    Ad = (_bf16(A) if a_kfast else _bf16(A.T.copy())).to(gpu).contiguous()
    Bd = (_bf16(B.T.copy()) if b_kfast else _bf16(B)).to(gpu).contiguous()
    sam, sak = (K, 1) if a_kfast else (1, M)
    sbk, sbn = (1, K) if b_kfast else (N, 1)
    # fp32 additions of one element: 32 inside an MFMA, one per K step of a wave, one per wave; each
    # may be off by 2^-23 of the running sum, which the sum of magnitudes bounds
    tol = (32 + K / 512 + 1 + 16) * 2.0 ** -23 * (np.abs(Ab) @ np.abs(Bb))
    for off in (0, 1):  # the second pass from an odd element, so that no wide load is aligned
        Ao = torch.cat([Ad.flatten()[:off], Ad.flatten()])[off:]
        Bo = torch.cat([Bd.flatten()[:off], Bd.flatten()])[off:]
        C = torch.full((M, N), float("nan"), dtype=torch.float32, device=gpu)
        sg.gemm(M, N, K, Ao, sam, sak, Bo, sbk, sbn, Cf=C, ldc=N)
        torch.cuda.synchronize()
        assert np.all(np.abs(C.cpu().numpy() - Ab @ Bb) <= tol)


# rows of k at any alignment: every remainder of a 16-byte load, one and several K steps, split and not
@pytest.mark.parametrize("a_rows,b_rows", [(True, True), (True, False), (False, True)])
@pytest.mark.parametrize("M,N,K", [(65, 33, k) for k in (1, 7, 8, 9, 15, 23, 25, 33, 63)] + [(64, 66, 259), (33, 1, 1029)])
def test_gemm_rows_at_any_alignment(gpu, a_rows, b_rows, M, N, K):
    """The bits of the same product with rows padded by zeros to whole aligned 16 bytes, for rows from
    an even or odd element at an even or odd pitch; what lies between and behind the rows is NaN."""
    import torch
    from pelelmex_amd import surrogate as sg
    g = torch.Generator().manual_seed(K)
    bias = torch.randn(N, generator=g).to(gpu)
    pad = (K + 7) // 8 * 8

    def operand(x, rows, ld, off):  # (tensor, stride of x's rows, stride of k); columns of x: x contiguous
        if not rows:
            return x.t().contiguous().to(torch.bfloat16).to(gpu), 1, x.shape[0]
        buf = torch.full((off + x.shape[0] * ld + 8,), float("nan"), dtype=torch.bfloat16)
        buf[off:off + x.shape[0] * ld].view(x.shape[0], ld)[:, :x.shape[1]] = x.to(torch.bfloat16)
        return buf.to(gpu)[off:], ld, 1

    def products(a, b, k, ld, off):
        (A, sam, sak), (B, sbn, sbk) = operand(a, a_rows, ld, off), operand(b, b_rows, ld, off)
        out = []
        for bi in (bias, None):
            C = torch.full((M, N), float("nan"), dtype=torch.float32, device=gpu)
            sg.gemm(M, N, k, A, sam, sak, B, sbk, sbn, bias=bi, Cf=C, ldc=N)
            out.append(C)
        return out

    a, b = torch.randn(M, K, generator=g), torch.randn(N, K, generator=g)
    zeros = lambda x: torch.cat([x, torch.zeros(x.shape[0], pad - K)], 1)
    want = products(zeros(a), zeros(b), pad, pad, 0)
    assert all(torch.isfinite(w).all() for w in want)
    for off, odd in ((0, 0), (0, 1), (1, 0), (1, 1), (2, 1)):
        for got, w in zip(products(a, b, K, K + (K + odd) % 2, off), want):
            assert torch.equal(got, w), (off, odd)


def test_gemm_odd_rows_cost_no_multiple(gpu):
    """A product of odd rows takes about the time of the aligned one (0.9; 2.4 by single elements)."""
    import time
    import torch
    from pelelmex_amd import surrogate as sg
    took = []
    for M, N, K in ((2048, 2048, 2048), (2048, 2047, 2049)):
        A, B = (torch.randn(n * K, device=gpu).to(torch.bfloat16) for n in (M, N))
        C, bias, ts = torch.empty((M, N), device=gpu), torch.zeros(N, device=gpu), []
        for _ in range(20):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            sg.gemm(M, N, K, A, K, 1, B, 1, K, bias=bias, Cf=C, ldc=N)
            torch.cuda.synchronize()
            ts.append(time.perf_counter() - t0)
        took.append(float(np.median(ts)))
    assert took[1] < 1.6 * took[0]


@pytest.mark.parametrize("rows,cols", [(1, 1), (511, 15), (512, 16), (513, 17), (4097, 22), (1030, 256)])
def test_column_sum(gpu, rows, cols):
    """Four partial sums over rows r, r + 4, .. in row order, then (0 + 1) + (2 + 3): bit for bit."""
    import torch
    from pelelmex_amd import surrogate as sg
    from pelelmex_amd.reactor import lib
    d = torch.randn((rows, cols + 3), generator=torch.Generator().manual_seed(rows))
    p = np.zeros((4, cols), dtype=np.float32)
    for r in range(rows):
        p[r % 4] += d[r, :cols].numpy()
    ref = (p[0] + p[1]) + (p[2] + p[3])
    out = torch.full((cols,), 2.0, dtype=torch.float32, device=gpu)
    dg = d.to(gpu)
    for acc, want in ((0, ref), (1, ref + ref)):
        assert lib().pr_mlp_column_sum(rows, cols, sg._ptr(dg), cols + 3, sg._ptr(out), acc, sg._stream()) == 0
        torch.cuda.synchronize()
        np.testing.assert_array_equal(out.cpu().numpy(), want)


def test_adam_on_replaced_tensors(gpu):
    """A network whose lists hold a caller's own tensors steps like one that keeps its buffers."""
    import torch
    from pelelmex_amd import surrogate as sg
    nets = [sg.MLP([5, 7, 3], device=gpu, seed=2) for _ in range(2)]
    nets[1].W[0], nets[1].b[1] = nets[1].W[0].clone(), nets[1].b[1].clone()
    for net in nets:
        for i, g in enumerate(net.gW + net.gb):
            g.copy_(torch.linspace(-1.0, 1.0 + i, g.numel()).reshape(g.shape))
        net.adam()
        net.adam(lr=1e-2)
    for a, b in zip(nets[0].W + nets[0].b + nets[0].Wb, nets[1].W + nets[1].b + nets[1].Wb):
        assert torch.equal(a, b)
