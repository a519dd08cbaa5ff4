"""GPU tests of the surrogate's kernels through the C-ABI: the bf16 MFMA GEMM
(bit-exact on integer-valued operands, where FP32 accumulation is exact in
any order, so the check pins the matrix-core lane layout), and the
elementwise training kernels against PyTorch FP32."""
import numpy as np
import pytest
import torch

from digital_twin_brain_amd import _native as nat

pytestmark = pytest.mark.gpu


def ctypes_stream():
    return torch.cuda.current_stream().cuda_stream


def _bits(x):
    """bf16 tensor -> its raw uint16 storage (int16 view)."""
    return x.contiguous().view(torch.int16)


def gemm(A, B, bias=None, act=0, want_bf16=False, lda=None, ldb=None):
    """A [M,K] / B [N,K] bf16 on the device (may be column slices of wider buffers)."""
    L = nat.lib()
    M, K = A.shape
    N = B.shape[0]
    C = torch.empty((M, N), dtype=torch.float32, device="cuda")
    Cb = torch.empty((M, N), dtype=torch.bfloat16, device="cuda") if want_bf16 else None
    nat.check(L.dtb_mlp_gemm_bf16_nt(M, N, K, A.data_ptr(), lda or A.stride(0), B.data_ptr(), ldb or B.stride(0),
                                      nat.ptr(bias), act, C.data_ptr(), N, nat.ptr(Cb), N, ctypes_stream()))
    torch.cuda.synchronize()
    return (C, Cb) if want_bf16 else C


# the first four take 32x32 tiles with K split over the wavefronts (K = 16 gives
# three wavefronts an empty range); 1024x1024 takes 64x64 tiles; the next two
# take 128x128 tiles (at least 256 of them), with a 32-row and a 64-column edge band;
# the last three take LDS-staged 256x256 tiles (64, 72 and 81 tiles: the tile map
# deals workgroups eight at a time, so 81 leaves seven idle)
@pytest.mark.parametrize("M,N,K", [(32, 32, 16), (96, 160, 48), (256, 512, 384), (64, 96, 1040), (1024, 1024, 48),
                                   (2080, 2080, 64), (2048, 2112, 48), (2048, 2048, 128), (2304, 2048, 64),
                                   (2304, 2304, 192)])
def test_gemm_bit_exact_on_integer_operands(M, N, K):
    g = torch.Generator().manual_seed(M * 7 + N + K)
    A = torch.randint(-4, 5, (M, K), generator=g).to(torch.bfloat16)
    B = torch.randint(-4, 5, (N, K), generator=g).to(torch.bfloat16)
    bias = torch.randint(-8, 9, (N,), generator=g).float()
    want = A.double() @ B.double().T + bias.double()
    C = gemm(A.cuda(), B.cuda(), bias.cuda())
    assert torch.equal(C.cpu().double(), want)
    C, Cb = gemm(A.cuda(), B.cuda(), bias.cuda(), act=1, want_bf16=True)
    assert torch.equal(C.cpu().double(), want.clamp_min(0))
    assert torch.equal(Cb.cpu().float(), want.clamp_min(0).float().to(torch.bfloat16).float())


@pytest.mark.parametrize("M,N,K", [(128, 64, 96), (2048, 2048, 256)])
def test_gemm_strided_operands_and_random_values(M, N, K):
    g = torch.Generator().manual_seed(5)
    Abuf = torch.randn((M, K + 24), generator=g).to(torch.bfloat16).cuda()
    Bbuf = torch.randn((N, K + 8), generator=g).to(torch.bfloat16).cuda()
    A, B = Abuf[:, :K], Bbuf[:, :K]
    C = gemm(A, B)
    want = A.float().cpu() @ B.float().cpu().T
    torch.testing.assert_close(C.cpu(), want, rtol=1e-5, atol=1e-5 * K ** 0.5)


# edges of the LDS-staged tiles (256, 128, 64, and 64 with K in four ranges) with
# ragged last rows and columns of tiles; K from less than one 64-wide slice over
# one, two and three slices to a slice ring used more than once, whole and short
# last slices.  Integers: every partial sum is exact.  The columns and rows
# around C stay untouched.
@pytest.mark.parametrize("K", [16, 48, 64, 112, 128, 144, 192, 208, 256, 400, 704])
@pytest.mark.parametrize("M,N", [(3808, 3104), (2080, 2144), (1056, 992), (736, 800)])
def test_gemm_tile_edges(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    A = torch.randint(-4, 5, (M, K + 8), generator=g, device="cuda").to(torch.bfloat16)
    B = torch.randint(-4, 5, (N, K + 16), generator=g, device="cuda").to(torch.bfloat16)
    bias = torch.randint(-8, 9, (N,), generator=g, device="cuda").float()
    C = torch.full((M + 1, N + 4), 0.5, device="cuda")
    nat.check(nat.lib().dtb_mlp_gemm_bf16_nt(M, N, K, A.data_ptr(), K + 8, B.data_ptr(), K + 16, bias.data_ptr(), 0,
                                             C.data_ptr(), N + 4, None, 0, ctypes_stream()))
    want = torch.full_like(C, 0.5)
    want[:M, :N] = A[:, :K].float() @ B[:, :K].float().T + bias
    assert torch.equal(C, want)


# both sides of the rules that choose by K and by the number of 32x32 tiles (256: one a CU)
@pytest.mark.parametrize("M,N,K,kernel", [
    (4096, 4128, 192, "tile_kernel<1>"), (4096, 4128, 256, "tile_kernel<1>"), (4096, 4128, 272, "tile_kernel<2>"),
    (4096, 4064, 272, "tile_kernel<4>"), (12320, 12288, 192, "tile_kernel<1>"), (12320, 12288, 208, "tile_kernel<4>"),
    (32, 8192, 1040, "splitk"), (8192, 32, 1040, "splitk"), (32, 8224, 1040, "tile_kernel<1>"),
    (64, 8192, 1040, "tile_kernel<1>")])
def test_gemm_on_both_sides_of_the_tile_rules(M, N, K, kernel):
    from digital_twin_brain_amd.surrogate import gemm_kernel_name

    assert kernel in gemm_kernel_name(M, N, K)
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    A = torch.randint(-4, 5, (M, K), generator=g, device="cuda").to(torch.bfloat16)
    B = torch.randint(-4, 5, (N, K), generator=g, device="cuda").to(torch.bfloat16)
    C = torch.empty((M, N), device="cuda")
    nat.check(nat.lib().dtb_mlp_gemm_bf16_nt(M, N, K, A.data_ptr(), K, B.data_ptr(), K, None, 0, C.data_ptr(), N, None,
                                             0, ctypes_stream()))
    assert torch.equal(C, A.float() @ B.float().T)


def test_gemm_rejects_bad_shapes():
    L = nat.lib()
    A = torch.zeros((32, 16), dtype=torch.bfloat16, device="cuda")
    C = torch.zeros((32, 32), dtype=torch.float32, device="cuda")
    assert L.dtb_mlp_gemm_bf16_nt(33, 32, 16, A.data_ptr(), 16, A.data_ptr(), 16, None, 0, C.data_ptr(), 32, None,
                                  0, None) == nat.DTB_INVALID_PARAMETER
    assert L.dtb_mlp_gemm_bf16_nt(32, 32, 12, A.data_ptr(), 16, A.data_ptr(), 16, None, 0, C.data_ptr(), 32, None,
                                  0, None) == nat.DTB_INVALID_PARAMETER
    assert L.dtb_mlp_gemm_bf16_nt(32, 32, 16, A.data_ptr(), 16, A.data_ptr(), 16, None, 2, C.data_ptr(), 32, None,
                                  0, None) == nat.DTB_INVALID_PARAMETER


def test_transpose_and_convert():
    L = nat.lib()
    g = torch.Generator().manual_seed(2)
    x = torch.randn((70, 45), generator=g)
    xb = x.to(torch.bfloat16).cuda()
    out = torch.empty((45, 70), dtype=torch.bfloat16, device="cuda")
    nat.check(L.dtb_mlp_transpose_bf16(70, 45, xb.data_ptr(), out.data_ptr(), ctypes_stream()))
    cb = torch.empty((70, 45), dtype=torch.bfloat16, device="cuda")
    xs = x.cuda()
    nat.check(L.dtb_mlp_f32_to_bf16(x.numel(), xs.data_ptr(), cb.data_ptr(), ctypes_stream()))
    torch.cuda.synchronize()
    assert torch.equal(_bits(out.cpu()), _bits(xb.cpu().T))
    # round to nearest even, as torch's conversion
    assert torch.equal(_bits(cb.cpu()), _bits(x.to(torch.bfloat16)))


def test_elementwise_training_kernels():
    L = nat.lib()
    g = torch.Generator().manual_seed(3)
    M, N = 64, 96
    dY = torch.randn((M, N), generator=g).cuda()
    Z = torch.randn((M, N), generator=g).cuda()
    dZ = torch.empty_like(dY)
    nat.check(L.dtb_mlp_relu_backward(M * N, dY.data_ptr(), Z.data_ptr(), dZ.data_ptr(), None, ctypes_stream()))
    db = torch.empty(N, device="cuda")
    nat.check(L.dtb_mlp_bias_grad(M, N, dZ.data_ptr(), db.data_ptr(), ctypes_stream()))
    out = torch.randn((M, N), generator=g).cuda()
    tgt = torch.randn((M, N), generator=g).cuda()
    mask = (torch.rand((M, N), generator=g) > 0.3).float().cuda()
    grad = torch.empty_like(out)
    nb = (M * N + 255) // 256
    lsum = torch.empty(nb, device="cuda")
    nat.check(L.dtb_mlp_mse_grad(M * N, out.data_ptr(), tgt.data_ptr(), mask.data_ptr(), 0.5, grad.data_ptr(), None,
                                 lsum.data_ptr(), ctypes_stream()))
    torch.cuda.synchronize()
    assert torch.equal(dZ, torch.where(Z > 0, dY, torch.zeros_like(dY)))
    torch.testing.assert_close(db, dZ.sum(0), rtol=1e-5, atol=1e-5)
    d = (out - tgt) * mask
    torch.testing.assert_close(grad, 0.5 * d, rtol=1e-6, atol=1e-7)
    torch.testing.assert_close(lsum.sum(), (d * d).sum(), rtol=1e-5, atol=1e-5)


def test_adam_matches_torch_optimizer():
    L = nat.lib()
    g = torch.Generator().manual_seed(4)
    n = 1000
    w0 = torch.randn(n, generator=g)
    p = torch.nn.Parameter(w0.clone())
    opt = torch.optim.Adam([p], lr=1e-3, betas=(0.9, 0.999), eps=1e-8)
    w = w0.clone().cuda()
    m = torch.zeros(n, device="cuda")
    v = torch.zeros(n, device="cuda")
    wb = torch.empty(n, dtype=torch.bfloat16, device="cuda")
    for t in range(1, 6):
        gr = torch.randn(n, generator=g)
        p.grad = gr.clone()
        opt.step()
        gc = gr.cuda()
        nat.check(L.dtb_mlp_adam(n, w.data_ptr(), gc.data_ptr(), m.data_ptr(), v.data_ptr(), 1e-3, 0.9, 0.999, 1e-8,
                                 t, wb.data_ptr(), ctypes_stream()))
    torch.cuda.synchronize()
    torch.testing.assert_close(w.cpu(), p.detach(), rtol=1e-5, atol=1e-6)
    assert torch.equal(_bits(wb.cpu()), _bits(w.cpu().to(torch.bfloat16)))


def _rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


def test_surrogate_gradients_match_fp64_oracle():
    """One forward + backward of a 3-hidden-layer MLP on the GPU against the
    FP64 oracle with bf16 rounding at the same points; remaining differences
    are FP32 accumulation order (and rare bf16 rounding flips)."""
    from digital_twin_brain_amd.surrogate import MLPSurrogate
    from oracle import mlp_oracle as mo

    rng = np.random.default_rng(7)
    n_in, n_out, r = 70, 45, 50
    sur = MLPSurrogate(n_in, n_out, hidden=(96, 128, 64), max_batch=64, seed=3)
    # non-zero biases so every term of the backward is exercised
    for b in sur.b:
        b.copy_(torch.from_numpy(rng.normal(size=b.shape[0]) * 0.1).float())
    X = rng.normal(size=(r, n_in))
    Y = rng.normal(size=(r, n_out))
    mask = (rng.random((r, n_out)) > 0.2).astype(np.float64)
    ls = sur.gradients(torch.from_numpy(X), torch.from_numpy(Y), torch.from_numpy(mask))
    torch.cuda.synchronize()
    P = sur.params_numpy()
    Xp = np.zeros((r, sur.sizes[0])); Xp[:, :n_in] = X
    Tp = np.zeros((r, sur.sizes[-1])); Tp[:, :n_out] = Y
    Mp = np.zeros((r, sur.sizes[-1])); Mp[:, :n_out] = mask
    Yo, hs = mo.forward(P, Xp, bf16=True)
    loss, gY = mo.loss_and_grad(Yo, Tp, Mp, 1.0 / r)
    grads = mo.backward(P, hs, gY, bf16=True)
    np.testing.assert_allclose(sur.H[-1][:r].cpu().double().numpy(), Yo, rtol=1e-4, atol=1e-4)
    assert abs(float(ls.sum()) / r / 2 - loss) <= 1e-4 * loss
    for l, (dW, db) in enumerate(grads):
        assert _rel(sur.dW[l].cpu().double().numpy(), dW) < 2e-3, l
        assert _rel(sur.db[l].cpu().double().numpy(), db) < 2e-3, l


def test_surrogate_predict_matches_oracle_and_training_fits():
    from digital_twin_brain_amd.surrogate import MLPSurrogate
    from oracle import mlp_oracle as mo

    rng = np.random.default_rng(8)
    n_in, n_out, n = 20, 12, 2048
    A = rng.normal(size=(n_in, n_out)) / np.sqrt(n_in)
    X = rng.normal(size=(n, n_in))
    Y = np.tanh(X @ A) + 0.5 * (X[:, :n_out] ** 2)
    sur = MLPSurrogate(n_in, n_out, hidden=(128, 128), max_batch=256, seed=1, lr=2e-3)
    sur.set_normalization(X, Y)
    hist = sur.fit(torch.from_numpy(X), torch.from_numpy(Y), epochs=40, batch=256)
    assert hist[-1] < 0.1 * hist[0], hist
    pred = sur.predict(torch.from_numpy(X[:300])).cpu().double().numpy()
    # the same prediction from the oracle with the trained weights
    P = sur.params_numpy()
    xs, xh = sur.x_scale.cpu().double().numpy(), sur.x_shift.cpu().double().numpy()
    Xn = np.zeros((300, sur.sizes[0]))
    Xn[:, :n_in] = (X[:300].astype(np.float32) * xs.astype(np.float32) + xh.astype(np.float32))
    Yn, _ = mo.forward(P, Xn, bf16=True)
    want = Yn[:, :n_out] * sur._y_std.cpu().double().numpy() + sur._y_mean.cpu().double().numpy()
    np.testing.assert_allclose(pred, want, rtol=1e-3, atol=1e-3 * np.abs(want).max())
    nrmse = np.linalg.norm(pred - Y[:300]) / np.sqrt(pred.size) / (Y.max() - Y.min())
    assert nrmse < 0.05, nrmse


def test_loss_partial_sums_cover_only_the_current_batch():
    """After a full-size batch fills the loss buffer, a smaller batch's
    returned partial sums add up to that batch's own squared error (the
    buffer's tail belongs to the earlier batch)."""
    from digital_twin_brain_amd.surrogate import GRUSurrogate, MLPSurrogate

    rng = np.random.default_rng(5)
    sur = MLPSurrogate(20, 10, hidden=(64, 64), max_batch=256, seed=1)
    sur.gradients(torch.randn(256, 20), torch.randn(256, 10) * 100.0)
    X, Y = rng.normal(size=(40, 20)), rng.normal(size=(40, 10)).astype(np.float32)
    ls = sur.gradients(torch.from_numpy(X), torch.from_numpy(Y))
    out = sur.H[-1][:40, :10].cpu().double().numpy()
    want = ((out - Y) ** 2).sum()
    assert abs(float(ls.sum()) - want) <= 1e-4 * want

    gru = GRUSurrogate(10, 6, hidden=32, max_batch=64, max_steps=8, seed=1)
    gru.gradients(torch.randn(8, 64, 10), torch.randn(8, 64, 6) * 100.0)
    T, r = 3, 20
    X, Y = rng.normal(size=(T, r, 10)), rng.normal(size=(T, r, 6)).astype(np.float32)
    ls = gru.gradients(torch.from_numpy(X), torch.from_numpy(Y))
    B = (r + 31) // 32 * 32  # rows padded to a multiple of 32
    out = gru.Y[:T * B].cpu().double().numpy().reshape(T, B, -1)[:, :r, :6]
    want = ((out - Y) ** 2).sum()
    assert abs(float(ls.sum()) - want) <= 1e-4 * want


def test_gru_gradients_match_fp64_oracle():
    """BPTT of the GRU surrogate on the GPU against the FP64 oracle (itself
    pinned to torch.nn.GRU) with bf16 rounding at the same points."""
    from digital_twin_brain_amd.surrogate import GRUSurrogate
    from oracle import mlp_oracle as mo

    rng = np.random.default_rng(11)
    T, r, n_in, n_out, H = 6, 40, 50, 30, 64
    sur = GRUSurrogate(n_in, n_out, hidden=H, max_batch=64, max_steps=8, seed=2)
    sur.p["b_o"].copy_(torch.from_numpy(rng.normal(size=sur.O) * 0.1).float())
    X = rng.normal(size=(T, r, n_in))
    Y = rng.normal(size=(T, r, n_out))
    h0 = rng.normal(size=(r, H)) * 0.3
    ls = sur.gradients(torch.from_numpy(X), torch.from_numpy(Y), h0=torch.from_numpy(h0))
    torch.cuda.synchronize()
    P = sur.params_numpy()
    Xp = np.zeros((T, r, sur.I)); Xp[:, :, :n_in] = X
    Tp = np.zeros((T, r, sur.O)); Tp[:, :, :n_out] = Y
    Mp = np.zeros((T, r, sur.O)); Mp[:, :, :n_out] = 1.0
    h0f = h0.astype(np.float32).astype(np.float64)
    Yo, cache = mo.gru_forward(P, Xp, h0f, bf16=True)
    loss, gY = mo.loss_and_grad(Yo, Tp, Mp, 1.0 / (T * r))
    g = mo.gru_backward(P, cache, gY, bf16=True)
    B = 64  # 40 rows padded to a multiple of 32
    Yg = sur.Y[:T * B].cpu().double().numpy().reshape(T, B, -1)[:, :r]
    np.testing.assert_allclose(Yg, Yo, rtol=1e-3, atol=1e-3)
    assert abs(float(ls.sum()) / (T * r) / 2 - loss) <= 1e-3 * loss
    for k in ("W_ih", "b_ih", "W_hh", "b_hh", "W_o", "b_o"):
        assert _rel(sur.grad[k].cpu().double().numpy(), g[k]) < 5e-3, k


def test_gru_training_fits_a_delayed_sequence_task():
    """y_t = x_{t-1} (a one-step memory): only the recurrence can fit it."""
    from digital_twin_brain_amd.surrogate import GRUSurrogate

    rng = np.random.default_rng(12)
    T, n, d = 8, 512, 8
    X = rng.normal(size=(T, n, d))
    Y = np.concatenate([np.zeros((1, n, d)), X[:-1]], axis=0)
    sur = GRUSurrogate(d, d, hidden=64, max_batch=64, max_steps=T, seed=1, lr=3e-3)
    hist = sur.fit(torch.from_numpy(X), torch.from_numpy(Y), epochs=30, batch=64)
    assert hist[-1] < 0.2 * hist[0], hist
    pred, hT = sur.predict(torch.from_numpy(X[:, :64]))
    err = pred.cpu().double().numpy()[1:] - Y[1:, :64]
    assert np.sqrt((err ** 2).mean()) < 0.4
    assert hT.shape == (64, 64)


@pytest.mark.parametrize("M,N", [(1, 1), (15, 63), (16, 64), (127, 65), (128, 33), (129, 512), (2048, 2080)])
def test_bias_grad_adds_in_row_order(M, N):
    """Column sums at the edges of the 64-column workgroups, the 16-row runs and
    the 128-row stages, bit for bit against a loop over rows."""
    g = torch.Generator().manual_seed(M + N)
    dZ = torch.randn((M, N), generator=g)
    d = dZ.cuda()
    db = torch.full((N + 1,), 7.0, device="cuda")
    nat.check(nat.lib().dtb_mlp_bias_grad(M, N, d.data_ptr(), db.data_ptr(), ctypes_stream()))
    torch.cuda.synchronize()
    want = torch.zeros(N)
    for row in dZ:
        want += row
    assert torch.equal(db[:N].cpu(), want)
    assert float(db[N]) == 7.0


# the kernel stages 256 rows at a time: one stage short of, at and past full, ragged ones
# after full ones, beside column counts off its 64
@pytest.mark.parametrize("M,N", [(255, 63), (256, 65), (257, 33), (300, 100), (511, 7), (512, 129), (513, 64)])
def test_bias_grad_over_several_stages_of_rows(M, N):
    g = torch.Generator().manual_seed(M * 3 + N)
    dZ = torch.randn((M, N), generator=g)
    d = dZ.cuda()
    db = torch.full((N + 1,), 7.0, device="cuda")
    nat.check(nat.lib().dtb_mlp_bias_grad(M, N, d.data_ptr(), db.data_ptr(), ctypes_stream()))
    want = torch.zeros(N)
    for row in dZ:
        want += row
    assert torch.equal(db[:N].cpu(), want)
    assert float(db[N]) == 7.0


# one layer; one 32-wide tile; widths of one, two and more tiles per wavefront; a batch whose
# products are one chain over K (2048 x 512) beside ones split in four; wide inputs and outputs
# (two output tiles a wavefront and a half-empty second round); rows at the edges of the 32-row tiles
@pytest.mark.parametrize("n_in,n_out,hidden,rows,batch", [
    (18, 6, (), 5, 32), (18, 6, (32,), 31, 32), (40, 70, (64, 96), 33, 64), (18, 6, (512, 512, 512), 2048, 2048),
    (18, 6, (512, 256), 2047, 2048), (720, 540, (512, 512, 512), 64, 64), (100, 300, (544, 32), 130, 256),
    (8, 600, (128,), 96, 96), (33, 5, (64, 64, 64, 64, 64, 64, 64), 40, 64)])
def test_whole_network_kernels_equal_the_layer_by_layer_launches(n_in, n_out, hidden, rows, batch):
    """Prediction and weight gradients bit for bit; the bias gradients and loss
    sums, FP32 sums in another order, to (terms) roundings."""
    from digital_twin_brain_amd.surrogate import MLPSurrogate

    g = torch.Generator().manual_seed(rows + n_in)
    X = torch.randn((rows, n_in), generator=g)
    Y = torch.randn((rows, n_out), generator=g)
    mask = (torch.rand((rows, n_out), generator=g) > 0.3).float()
    Xp = torch.randn((batch + 70, n_in), generator=g)  # a whole batch and a part
    sur = [MLPSurrogate(n_in, n_out, hidden=hidden, max_batch=batch, seed=4) for _ in range(2)]
    for s in sur:
        assert s.chain and s.chain_train
        for b in s.b:
            b.copy_(torch.linspace(-0.1, 0.2, b.shape[0]))
        s.set_normalization(X, Y + 0.3)
    sur[1].chain = sur[1].chain_train = False
    sur[1]._alloc_layers()
    sur[1]._refresh_bf16()
    for m in (None, mask):
        for step in range(2):
            a, b = (s.gradients(X, Y, m).clone() for s in sur)
            B = (rows + 31) // 32 * 32
            assert a.shape == b.shape
            torch.testing.assert_close(a, b, rtol=256 * 2.0 ** -23, atol=0)
            assert torch.equal(sur[0].H[-1][:B], sur[1].H[-1][:B])
            for l in range(len(hidden) + 1):
                assert torch.equal(sur[0].dW[l], sur[1].dW[l]), l
                G = sur[1].G[l][:B].double()
                bound = B * 2.0 ** -23 * G.abs().sum(0)
                assert ((sur[0].db[l].double() - G.sum(0)).abs() <= bound).all(), l
            for s in sur:
                for l in range(len(hidden) + 1):
                    s.db[l].copy_(sur[1].db[l])  # the same bias step on both sides
                s.step()
            for l in range(len(hidden) + 1):
                assert torch.equal(sur[0].W[l], sur[1].W[l]) and torch.equal(sur[0].b[l], sur[1].b[l])
                assert torch.equal(_bits(sur[1].Wb[l]), _bits(sur[1].W[l].to(torch.bfloat16)))
                assert torch.equal(_bits(sur[1].WbT[l]), _bits(sur[1].Wb[l].T))
    assert torch.equal(sur[0].predict(Xp), sur[1].predict(Xp))


def test_networks_beyond_the_whole_network_kernels_run_layer_by_layer():
    from digital_twin_brain_amd.surrogate import MLPSurrogate

    for hidden in ((2560,), (32,) * 8):  # wider than 160 KB of activations; nine layers
        sur = MLPSurrogate(10, 4, hidden=hidden, max_batch=32, seed=1)
        assert not sur.chain and not sur.chain_train
        sur.gradients(torch.randn(20, 10), torch.randn(20, 4))
        sur.step()
        assert sur.predict(torch.randn(40, 10)).isfinite().all()
    mixed = MLPSurrogate(10, 4, hidden=(1184, 1184), max_batch=32, seed=1)  # the sign masks do not fit beside 1,184 columns
    assert mixed.chain and not mixed.chain_train
    mixed.gradients(torch.randn(20, 10), torch.randn(20, 4))
    mixed.step()
    assert mixed.predict(torch.randn(40, 10)).isfinite().all()


# hidden sizes whose split of K falls between, on and inside the 32-column instructions, one unit
# tile to all wavefronts, weights in registers alone and partly in LDS; ragged batches; one step
@pytest.mark.parametrize("H,T,rows,n_in,n_out", [(32, 3, 5, 4, 3), (64, 5, 64, 18, 6), (96, 4, 33, 40, 70),
                                                 (128, 1, 32, 7, 5), (160, 3, 31, 8, 33), (192, 6, 40, 18, 6),
                                                 (224, 2, 64, 20, 6), (256, 7, 50, 18, 6), (256, 2, 100, 70, 100)])
def test_gru_sequence_kernels_equal_the_launch_per_step_path(H, T, rows, n_in, n_out):
    """Outputs, states and gradients bit for bit."""
    from digital_twin_brain_amd.surrogate import GRUSurrogate

    g = torch.Generator().manual_seed(H + T)
    X, Y = torch.randn((T, rows, n_in), generator=g), torch.randn((T, rows, n_out), generator=g)
    mask = (torch.rand((T, rows, n_out), generator=g) > 0.3).float()
    h0 = 0.3 * torch.randn((rows, H), generator=g)
    sur = [GRUSurrogate(n_in, n_out, hidden=H, max_batch=rows + 20, max_steps=T, seed=2) for _ in range(2)]
    assert all(s.sequence for s in sur)
    sur[1].sequence = False
    sur[1]._alloc_steps()
    for s in sur:
        s.set_normalization(X, Y + 0.2)
    B = (rows + 31) // 32 * 32
    for h, m in ((None, None), (h0, mask)):
        a, b = (s.gradients(X, Y, m, h).clone() for s in sur)
        assert torch.equal(a, b)
        assert torch.equal(sur[0].Y[:T * B], sur[1].Y[:T * B])
        assert torch.equal(sur[0].Hs[:(T + 1) * B], sur[1].Hs[:(T + 1) * B])
        for k in sur[0].grad:
            assert torch.equal(sur[0].grad[k], sur[1].grad[k]), k
        for s in sur:
            s.step()
        for k in sur[0].p:
            assert torch.equal(sur[0].p[k], sur[1].p[k]), k
    (ya, ha), (yb, hb) = (s.predict(X, h0) for s in sur)
    assert torch.equal(ya, yb) and torch.equal(ha, hb)


def test_gru_beyond_the_sequence_kernels():
    """Hidden sizes past 256 keep the launch per step; the gradients are checked against the FP64 oracle."""
    from digital_twin_brain_amd.surrogate import GRUSurrogate
    from oracle import mlp_oracle as mo

    rng = np.random.default_rng(3)
    T, r = 3, 32
    sur = GRUSurrogate(8, 4, hidden=288, max_batch=32, max_steps=T, seed=2)
    assert not sur.sequence
    X, Y = rng.normal(size=(T, r, 8)), rng.normal(size=(T, r, 4))
    sur.gradients(torch.from_numpy(X), torch.from_numpy(Y))
    Xp = np.zeros((T, r, sur.I)); Xp[:, :, :8] = X
    Tp = np.zeros((T, r, sur.O)); Tp[:, :, :4] = Y
    Mp = np.zeros((T, r, sur.O)); Mp[:, :, :4] = 1.0
    P = sur.params_numpy()
    Yo, cache = mo.gru_forward(P, Xp, np.zeros((r, sur.H)), bf16=True)
    _, gY = mo.loss_and_grad(Yo, Tp, Mp, 1.0 / (T * r))
    g = mo.gru_backward(P, cache, gY, bf16=True)
    for k in g:
        if k in sur.grad:
            assert _rel(sur.grad[k].cpu().double().numpy(), g[k]) < 5e-3, k


def test_gru_targets_and_masks_broadcast_as_in_an_assignment():
    from digital_twin_brain_amd.surrogate import GRUSurrogate

    T, r = 3, 5
    g = torch.Generator().manual_seed(1)
    m = GRUSurrogate(4, 6, hidden=32, max_batch=8, max_steps=T)
    X, Y = torch.randn((T, r, 4), generator=g), torch.randn((T, r, 6), generator=g)
    mask = (torch.rand((r, 1), generator=g) > 0.4).float()

    def grads(y, k):
        loss = m.gradients(X, y, mask=k).clone()
        return [loss] + [v.clone() for v in m.grad.values()]

    want = grads(Y, mask.expand(T, r, 6))
    for y, k in ((Y[None], mask), (Y, mask[None, None]), (Y[None, None], mask.expand(1, 1, T, r, 6))):
        for a, b in zip(grads(y, k), want):
            assert torch.equal(a, b)
    with pytest.raises(RuntimeError):
        m.gradients(X, Y[None].expand(2, T, r, 6))


# wide networks on both sides of the rule that sends few rows to a launch per product
@pytest.mark.parametrize("n_in,n_out,hidden,rows,chain,chain_train", [
    (18, 6, (512, 512, 512), 90, True, True), (18, 6, (1024, 1024, 1024), 90, False, True),
    (720, 540, (512, 512, 512), 40, False, True), (720, 540, (512, 512, 512), 2048, True, True),
    (720, 540, (1024, 1024, 1024), 32, False, False), (1100, 900, (1024, 1024, 1024), 33, False, True)])
def test_few_rows_of_wide_networks_go_layer_by_layer(n_in, n_out, hidden, rows, chain, chain_train):
    """The same predictions and weight gradients bit for bit, before and after
    an update, and with a first layer-by-layer call after it."""
    from digital_twin_brain_amd.surrogate import MLPSurrogate

    g = torch.Generator().manual_seed(rows + n_in)
    X, Y = torch.randn((rows, n_in), generator=g), torch.randn((rows, n_out), generator=g)
    a, b, late = (MLPSurrogate(n_in, n_out, hidden=hidden, max_batch=max(rows, 64), seed=4) for _ in range(3))
    assert a.chain and a.chain_train
    assert a._chain_pays(rows) == chain and a._chain_pays(rows, train=True) == chain_train
    assert a._chain_pays(a.max_batch + 1)
    b._chain_pays = lambda rows, train=False: True
    for _ in range(2):
        assert torch.equal(a.predict(X), b.predict(X))
        for s in (a, b, late):
            s.gradients(X, Y)
        for l in range(len(hidden) + 1):
            assert torch.equal(a.dW[l], b.dW[l]), l
            for s in (a, late):  # FP32 sums in another order
                s.db[l].copy_(b.db[l])
        for s in (a, b, late):
            s.step()
    assert torch.equal(a.predict(X), b.predict(X)) and torch.equal(late.predict(X), b.predict(X))
    assert (a.Wb is not None) == (not chain or not chain_train)
