"""Learned surrogate of a data-assimilation window (no counterpart in the
reference: new in this library).

`MLPSurrogate` is a ReLU multilayer perceptron trained and evaluated with the
library's own kernels (bf16 matrix-core GEMM with FP32 accumulation, fused
bias + ReLU, ReLU backward, bias gradient, masked MSE gradient, Adam on FP32
master weights, normalise/pad).  PyTorch provides only device memory and the
stream.

Layer l computes Z = H W_l^T + b_l with W_l stored [out, in]; widths are
padded to multiples of 32 and the batch to a multiple of 32 (padded rows
carry zero loss weight).  Backward per layer, with G the bf16 gradient of Z:
dW = G^T H (GEMM of the two transposes), db = column sums of G (FP32),
dH = G W (GEMM against the transposed weights), masked by H > 0.
"""
from __future__ import annotations

import numpy as np
import torch

from . import _native as nat


def _pad(n, m=32):
    return (int(n) + m - 1) // m * m


def _params(rows):
    """dtb_adam_param table of (rows, cols, w, g, m, v, and the bf16 copies wb, wt, wf, wtf) tensors."""
    return np.array([(r, c, *(0 if x is None else x.data_ptr() for x in ts)) for r, c, *ts in rows], dtype=np.int64)


def _broadcast(x, shape, dev):
    """x as contiguous FP32 on the device, broadcast to `shape` as an assignment
    to a tensor of that shape broadcasts it (leading ones beyond its rank go)."""
    x = torch.as_tensor(x).to(dev, torch.float32)
    while x.dim() > len(shape) and x.shape[0] == 1:
        x = x[0]
    return x.expand(shape).contiguous()


class MLPSurrogate:
    def __init__(self, n_in, n_out, hidden=(512, 512, 512), max_batch=256, device=0, seed=0, lr=1e-3,
                 betas=(0.9, 0.999), eps=1e-8):
        nat.require_gpu()
        self.lib = nat.lib()
        self.dev = torch.device("cuda", device)
        self.n_in, self.n_out = int(n_in), int(n_out)
        self.sizes = [_pad(n_in)] + [_pad(h) for h in hidden] + [_pad(n_out)]
        self.max_batch = _pad(max_batch)
        self.lr, self.b1, self.b2, self.eps = float(lr), float(betas[0]), float(betas[1]), float(eps)
        self.t = 0
        g = torch.Generator().manual_seed(seed)
        f32, bf = dict(dtype=torch.float32, device=self.dev), dict(dtype=torch.bfloat16, device=self.dev)
        # bf16 weights and their transposes in fragment order (dtb_adam_param)
        self.W, self.b, self.Wf, self.WTf = [], [], [], []
        self.Wb = self.WbT = None  # row-major copies of the launch-per-product path
        self.mW, self.vW, self.mb, self.vb, self.dW, self.db = [], [], [], [], [], []
        for l, (i, o) in enumerate(zip(self.sizes[:-1], self.sizes[1:])):
            w = torch.randn((o, i), generator=g) * np.sqrt(2.0 / i)  # He initialisation
            if l == 0:
                w[:, self.n_in:] = 0.0
            self.W.append(w.to(self.dev))
            self.b.append(torch.zeros(o, **f32))
            self.Wf.append(torch.empty((o, i), **bf))
            self.WTf.append(torch.empty((i, o), **bf))
            for lst in (self.mW, self.vW, self.dW):
                lst.append(torch.zeros((o, i), **f32))
            for lst in (self.mb, self.vb, self.db):
                lst.append(torch.zeros(o, **f32))
        B = self.max_batch
        self.HbT = [torch.empty((s, B), **bf) for s in self.sizes[:-1]]  # bf16 layer inputs, transposed
        self.GbT = [torch.empty((s, B), **bf) for s in self.sizes[1:]]   # bf16 gradient of each layer's Z, transposed
        self.dbp = [torch.empty((B // 32, s), **f32) for s in self.sizes[1:]]
        # the whole-network kernels, unless the network is too wide or deep for
        # them: then a launch per product, whose activations live in memory
        # (H: layer inputs, H[0] = X, and the output)
        table = self._table()
        self.chain = self.lib.dtb_mlp_chain_fits(len(self.W), table.ctypes.data, 0) == nat.DTB_OK
        self.chain_train = self.lib.dtb_mlp_chain_fits(len(self.W), table.ctypes.data, 1) == nat.DTB_OK
        self.H = [None] * len(self.W) + [torch.empty((B, self.sizes[-1]), **f32)]
        if not (self.chain and self.chain_train):
            self._alloc_layers()
        self.lsum = torch.empty(((B * self.sizes[-1] + 255) // 256,), **f32)
        self.x_scale = torch.ones(self.n_in, **f32)
        self.x_shift = torch.zeros(self.n_in, **f32)
        self.y_scale = torch.ones(self.n_out, **f32)
        self.y_shift = torch.zeros(self.n_out, **f32)
        self._y_std = torch.ones(self.n_out, **f32)
        self._y_mean = torch.zeros(self.n_out, **f32)
        self._refresh_bf16()

    # -- helpers -----------------------------------------------------------
    def _stream(self):
        return torch.cuda.current_stream(self.dev).cuda_stream

    def _alloc_layers(self):
        """Buffers of the launch-per-product path."""
        B = self.max_batch
        f32, bf = dict(dtype=torch.float32, device=self.dev), dict(dtype=torch.bfloat16, device=self.dev)
        self.Wb = [torch.empty(w.shape, **bf) for w in self.W]
        self.WbT = [torch.empty((w.shape[1], w.shape[0]), **bf) for w in self.W]
        self.H[:-1] = [torch.empty((B, s), **f32) for s in self.sizes[:-1]]
        self.Hb = [torch.empty((B, s), **bf) for s in self.sizes[:-1]]
        self.G = [torch.empty((B, s), **f32) for s in self.sizes[1:]]    # gradient of each layer's Z
        self.Gb = [torch.empty((B, s), **bf) for s in self.sizes[1:]]
        self.dH = torch.empty((B, max(self.sizes)), **f32)
        self.T = torch.empty((B, self.sizes[-1]), **f32)
        self.M = torch.empty((B, self.sizes[-1]), **f32)

    def _chain_pays(self, rows, train=False):
        """Whether the whole-network kernel is the faster way to take `rows` rows
        (else a launch per product, the same results bit for bit).

        It is, by far, for many rows.  But up to max_batch rows of a wide
        network leave most of the device idle while each workgroup streams
        every weight (10.5 us a MB) and walks wide inputs and outputs, where
        the launches cost 4.5 us each more than its layers and spread over the
        device.  us, launches : whole network, four layers with hidden widths h:
            18 -> h -> 6, 90 rows         h = 512 52:39, 768 56:50, 1,024 59:74
            18 -> h -> 1,000, 256 rows    h = 128 47:57, 512 48:71; 2,048 rows 55:58, 78:73
            720 -> h -> 540, 256 rows     h = 128 49:61, 512 50:74; 2,048 rows 54:61, 86:77
            1,100 -> h -> 900, 256 rows   h = 128 48:77, 1,024 59:164; 8,192 rows 104:97, 302:170
        and 18 -> 768 x 6 -> 6, 90 rows 81:98.  Training has more to gain
        (43 launches) and loses only for a single tile of rows of the widest:
        32 rows of 1,100 -> 1,024 x 3 -> 900 224:304, of 720 -> 1,024 x 3 -> 540
        214:252, but of 18 -> 1,024 x 3 -> 6 199:156."""
        n_in, n_out = self.sizes[0], self.sizes[-1]
        mb = 2e-6 * sum(w.numel() for w in self.W)  # bf16
        if train:
            return rows > 32 or mb < 6 or n_in + n_out < 1000
        if rows > self.max_batch:
            return True
        return 10.5 * mb + 0.02 * n_in + 0.03 * n_out <= 11 + 4.5 * len(self.W) + 0.006 * rows * mb

    def _use_chain(self, rows, train=False):
        if not (self.chain_train if train else self.chain):
            return False
        if self._chain_pays(rows, train):
            return True
        if self.Wb is None:
            self._alloc_layers()
            self._refresh_bf16()
        return False

    def _table(self):
        """dtb_mlp_layer [layers] (ten 8-byte fields each) of the current buffers."""
        return np.array([(w.shape[1], w.shape[0], wf.data_ptr(), wt.data_ptr(), b.data_ptr(), dw.data_ptr(),
                          db.data_ptr(), ht.data_ptr(), gt.data_ptr(), dbp.data_ptr())
                         for w, wf, wt, b, dw, db, ht, gt, dbp in zip(self.W, self.Wf, self.WTf, self.b, self.dW,
                                                                      self.db, self.HbT, self.GbT, self.dbp)],
                        dtype=np.int64)

    def _weights(self):
        none = [None] * len(self.W)
        return [(w.shape[0], w.shape[1], w, *r) for w, *r in
                zip(self.W, self.dW, self.mW, self.vW, self.Wb or none, self.WbT or none, self.Wf, self.WTf)]

    def _refresh_bf16(self):
        table = _params(self._weights())
        nat.check(self.lib.dtb_mlp_refresh_bf16(len(table), table.ctypes.data, self._stream()))

    def set_normalization(self, X, Y):
        """Per-feature standardisation from training data (host or device arrays)."""
        X = torch.as_tensor(X, dtype=torch.float64)
        Y = torch.as_tensor(Y, dtype=torch.float64)
        xs = X.std(0).clamp_min(1e-12)
        ys = Y.std(0).clamp_min(1e-12)
        self.x_scale = (1.0 / xs).float().to(self.dev)
        self.x_shift = (-X.mean(0) / xs).float().to(self.dev)
        self.y_scale = (1.0 / ys).float().to(self.dev)
        self.y_shift = (-Y.mean(0) / ys).float().to(self.dev)
        self._y_std = ys.float().to(self.dev)
        self._y_mean = Y.mean(0).float().to(self.dev)

    def _load_x(self, X, rows):
        X = X.to(self.dev, torch.float32).contiguous()
        nat.check(self.lib.dtb_mlp_affine(rows, self.n_in, self.sizes[0], X.data_ptr(), X.stride(0),
                                          self.x_scale.data_ptr(), self.x_shift.data_ptr(), self.H[0].data_ptr(),
                                          self.Hb[0].data_ptr(), self.sizes[0], self._stream()))

    def _forward(self, B):
        s = self._stream()
        L = len(self.W)
        for l in range(L):
            o, i = self.W[l].shape
            last = l == L - 1
            nat.check(self.lib.dtb_mlp_gemm_bf16_nt(B, o, i, self.Hb[l].data_ptr(), i, self.Wb[l].data_ptr(), i,
                                                    self.b[l].data_ptr(), 0 if last else 1, self.H[l + 1].data_ptr(),
                                                    o, None if last else self.Hb[l + 1].data_ptr(), o, s))

    # -- public API --------------------------------------------------------
    def predict(self, X):
        """X [rows, n_in] -> [rows, n_out] FP32 on the device (denormalised)."""
        X = torch.as_tensor(X)
        n = X.shape[0]
        out = torch.empty((n, self.n_out), dtype=torch.float32, device=self.dev)
        if self._use_chain(n):
            X = X.to(self.dev, torch.float32).contiguous()
            table = self._table()
            nat.check(self.lib.dtb_mlp_predict(len(self.W), table.ctypes.data, n, self.max_batch, X.data_ptr(),
                                               X.stride(0), self.n_in, self.x_scale.data_ptr(),
                                               self.x_shift.data_ptr(), self._y_std.data_ptr(),
                                               self._y_mean.data_ptr(), self.n_out, out.data_ptr(), self.n_out,
                                               self._stream()))
            return out
        for r0 in range(0, n, self.max_batch):
            r = min(self.max_batch, n - r0)
            B = _pad(r)
            self._load_x(X[r0:r0 + r], r)
            if B > r:
                self.Hb[0][r:B].zero_()
            self._forward(B)
            nat.check(self.lib.dtb_mlp_affine(r, self.n_out, self.n_out, self.H[-1].data_ptr(), self.sizes[-1],
                                              self._y_std.data_ptr(), self._y_mean.data_ptr(),
                                              out[r0:r0 + r].data_ptr(), None, self.n_out, self._stream()))
        return out

    def gradients(self, X, Y, mask=None):
        """Forward + backward on one batch (rows <= max_batch); leaves dW, db
        and returns the device loss partial sums.  The loss is
        sum(mask*(Yn - Tn)^2) / (2*rows) on standardised outputs."""
        s = self._stream()
        X = torch.as_tensor(X)
        r = X.shape[0]
        assert r <= self.max_batch
        B = _pad(r)
        no = self.sizes[-1]
        Yd = torch.as_tensor(Y).to(self.dev, torch.float32).contiguous()
        if self._use_chain(r, train=True):
            X = X.to(self.dev, torch.float32).contiguous()
            Md = None if mask is None else \
                torch.as_tensor(mask).to(self.dev, torch.float32).expand(r, self.n_out).contiguous()
            table = self._table()
            nat.check(self.lib.dtb_mlp_train_gradients(
                len(self.W), table.ctypes.data, r, X.data_ptr(), X.stride(0), self.n_in, self.x_scale.data_ptr(),
                self.x_shift.data_ptr(), Yd.data_ptr(), Yd.stride(0), self.n_out, self.y_scale.data_ptr(),
                self.y_shift.data_ptr(), nat.ptr(Md), self.n_out, 1.0 / max(r, 1), self.H[-1].data_ptr(),
                self.lsum.data_ptr(), s))
            return self.lsum[: (B * no + 255) // 256]
        self._load_x(X, r)
        nat.check(self.lib.dtb_mlp_affine(r, self.n_out, no, Yd.data_ptr(), Yd.stride(0), self.y_scale.data_ptr(),
                                          self.y_shift.data_ptr(), self.T.data_ptr(), None, no, s))
        self.M[:B].zero_()
        if mask is None:
            self.M[:r, :self.n_out].fill_(1.0)
        else:
            self.M[:r, :self.n_out].copy_(torch.as_tensor(mask).to(self.dev, torch.float32))
        if B > r:
            self.Hb[0][r:B].zero_()
            self.T[r:B].zero_()
        self._forward(B)
        L = len(self.W)
        nat.check(self.lib.dtb_mlp_mse_grad(B * no, self.H[L].data_ptr(), self.T.data_ptr(), self.M.data_ptr(),
                                            1.0 / r, self.G[L - 1].data_ptr(), self.Gb[L - 1].data_ptr(),
                                            self.lsum.data_ptr(), s))
        for l in range(L - 1, -1, -1):
            o, i = self.W[l].shape
            nat.check(self.lib.dtb_mlp_transpose_bf16(B, o, self.Gb[l].data_ptr(), self.GbT[l].data_ptr(), s))
            nat.check(self.lib.dtb_mlp_transpose_bf16(B, i, self.Hb[l].data_ptr(), self.HbT[l].data_ptr(), s))
            # dW[o, i] = sum_b G[b, o] H[b, i]
            nat.check(self.lib.dtb_mlp_gemm_bf16_nt(o, i, B, self.GbT[l].data_ptr(), B, self.HbT[l].data_ptr(), B,
                                                    None, 0, self.dW[l].data_ptr(), i, None, 0, s))
            nat.check(self.lib.dtb_mlp_bias_grad(B, o, self.G[l].data_ptr(), self.db[l].data_ptr(), s))
            if l > 0:
                # dH[b, i] = sum_o G[b, o] W[o, i], then the ReLU mask of layer l-1
                nat.check(self.lib.dtb_mlp_gemm_bf16_nt(B, i, o, self.Gb[l].data_ptr(), o, self.WbT[l].data_ptr(), o,
                                                        None, 0, self.dH.data_ptr(), i, None, 0, s))
                nat.check(self.lib.dtb_mlp_relu_backward(B * i, self.dH.data_ptr(), self.H[l].data_ptr(),
                                                         self.G[l - 1].data_ptr(), self.Gb[l - 1].data_ptr(), s))
        # the partial sums this batch wrote (the buffer is sized for the largest batch)
        return self.lsum[: (B * no + 255) // 256]

    def step(self):
        """One Adam step on every parameter from the last `gradients` call."""
        self.t += 1
        table = _params(self._weights() + [(1, b.shape[0], b, g, m, v, None, None, None, None) for b, g, m, v in
                                           zip(self.b, self.db, self.mb, self.vb)])
        nat.check(self.lib.dtb_mlp_adam_multi(len(table), table.ctypes.data, self.lr, self.b1, self.b2, self.eps,
                                              self.t, self._stream()))

    def fit(self, X, Y, epochs=50, batch=None, seed=0, verbose=False):
        """Mini-batch Adam over (X, Y) kept on the device; returns the mean
        standardised loss per epoch."""
        X = torch.as_tensor(X).to(self.dev, torch.float32)
        Y = torch.as_tensor(Y).to(self.dev, torch.float32)
        n = X.shape[0]
        batch = min(self.max_batch, n) if batch is None else int(batch)
        g = torch.Generator().manual_seed(seed)
        hist = []
        for ep in range(epochs):
            perm = torch.randperm(n, generator=g).to(self.dev)
            tot = torch.zeros((), dtype=torch.float64, device=self.dev)
            for r0 in range(0, n - batch + 1, batch):
                idx = perm[r0:r0 + batch]
                ls = self.gradients(X.index_select(0, idx), Y.index_select(0, idx))
                tot += ls.sum().double() / batch
                self.step()
            hist.append(float(tot) / max(1, n // batch) / self.n_out)
            if verbose:
                print(f"epoch {ep}: loss {hist[-1]:.4e}")
        return hist

    def params_numpy(self):
        """[(W, b)] in FP32, unpadded widths dropped only for clarity of tests."""
        return [(w.cpu().double().numpy(), b.cpu().double().numpy()) for w, b in zip(self.W, self.b)]


class GRUSurrogate:
    """Single-layer GRU (gate order r, z, n as torch.nn.GRU) with a linear
    readout per step, trained by backpropagation through time on the
    library's kernels.

    Forward over a sequence X [T, B, n_in]: one GEMM for every step's input
    projection, one kernel for all steps of the recurrence, one GEMM for every
    step's readout.  Backward: the loss and its gradient, one GEMM to the
    hidden states, one kernel for all steps in reverse, then all weight
    gradients over the T*B rows together.  Hidden sizes past 256 (or batches
    whose products the sequence kernels do not take) run a recurrent GEMM and
    a gate kernel per step instead."""

    def __init__(self, n_in, n_out, hidden=256, max_batch=64, max_steps=32, device=0, seed=0, lr=1e-3,
                 betas=(0.9, 0.999), eps=1e-8):
        nat.require_gpu()
        self.lib = nat.lib()
        self.dev = torch.device("cuda", device)
        self.n_in, self.n_out = int(n_in), int(n_out)
        self.I, self.H, self.O = _pad(n_in), _pad(hidden), _pad(n_out)
        self.max_batch, self.max_steps = _pad(max_batch), int(max_steps)
        self.lr, self.b1, self.b2, self.eps = float(lr), float(betas[0]), float(betas[1]), float(eps)
        self.t = 0
        g = torch.Generator().manual_seed(seed)
        f32, bf = dict(dtype=torch.float32, device=self.dev), dict(dtype=torch.bfloat16, device=self.dev)
        H, I, O = self.H, self.I, self.O
        s = 1.0 / np.sqrt(H)
        w_ih = (torch.rand((3 * H, I), generator=g) * 2 - 1) * s
        w_ih[:, self.n_in:] = 0.0
        init = dict(W_ih=w_ih, b_ih=(torch.rand(3 * H, generator=g) * 2 - 1) * s,
                    W_hh=(torch.rand((3 * H, H), generator=g) * 2 - 1) * s,
                    b_hh=(torch.rand(3 * H, generator=g) * 2 - 1) * s,
                    W_o=torch.randn((O, H), generator=g) * s, b_o=torch.zeros(O))
        self.p = {k: v.float().to(self.dev) for k, v in init.items()}
        self.grad = {k: torch.zeros_like(v) for k, v in self.p.items()}
        self.m = {k: torch.zeros_like(v) for k, v in self.p.items()}
        self.v = {k: torch.zeros_like(v) for k, v in self.p.items()}
        self.pb = {k: torch.empty(self.p[k].shape, **bf) for k in ("W_ih", "W_hh", "W_o")}
        self.pbT = {k: torch.empty(tuple(reversed(self.p[k].shape)), **bf) for k in ("W_hh", "W_o")}
        B, T = self.max_batch, self.max_steps
        self.Xb = torch.empty((T * B, I), **bf)
        self.XbT = torch.empty((I, T * B), **bf)
        self.Gi = torch.empty((T * B, 3 * H), **f32)
        self.Gh = torch.empty((T * B, 3 * H), **f32)
        self.Hs = torch.empty(((T + 1) * B, H), **f32)
        self.Hb = torch.empty(((T + 1) * B, H), **bf)
        self.HbT = torch.empty((H, (T + 1) * B), **bf)
        self.Y = torch.empty((T * B, O), **f32)
        self.Gy = torch.empty((T * B, O), **f32)
        self.Gyb = torch.empty((T * B, O), **bf)
        self.GybT = torch.empty((O, T * B), **bf)
        self.dHo = torch.empty((T * B, H), **f32)
        self.dGib = torch.empty((T * B, 3 * H), **bf)
        self.dGhb = torch.empty((T * B, 3 * H), **bf)
        self.dGiT = torch.empty((3 * H, T * B), **bf)
        self.dGhT = torch.empty((3 * H, T * B), **bf)
        # every batch up to max_batch takes the sequence kernels, or none does
        self.sequence = self.lib.dtb_gru_sequence_fits(B, H) == nat.DTB_OK
        if self.sequence:
            self.dG = torch.empty((T * B, 4 * H), **f32)
        else:
            self._alloc_steps()
        self.lsum = torch.empty(((T * B * O + 255) // 256,), **f32)
        self.x_scale = torch.ones(self.n_in, **f32)
        self.x_shift = torch.zeros(self.n_in, **f32)
        self.y_scale = torch.ones(self.n_out, **f32)
        self.y_shift = torch.zeros(self.n_out, **f32)
        self._y_std = torch.ones(self.n_out, **f32)
        self._y_mean = torch.zeros(self.n_out, **f32)
        self._refresh_bf16()

    def _stream(self):
        return torch.cuda.current_stream(self.dev).cuda_stream

    def _alloc_steps(self):
        """Buffers of the launch-per-step path."""
        B, T, H = self.max_batch, self.max_steps, self.H
        f32 = dict(dtype=torch.float32, device=self.dev)
        self.dGi = torch.empty((T * B, 3 * H), **f32)
        self.dGh = torch.empty((T * B, 3 * H), **f32)
        self.dhz = torch.empty((B, H), **f32)
        self.dhg = torch.empty((B, H), **f32)

    def _refresh_bf16(self):
        table = _params([(w.shape[0], w.shape[1], w, None, None, None, self.pb[k], self.pbT.get(k), None, None)
                         for k, w in self.p.items() if k in self.pb])
        nat.check(self.lib.dtb_mlp_refresh_bf16(len(table), table.ctypes.data, self._stream()))

    def set_normalization(self, X, Y):
        """Per-feature standardisation over every step and sequence."""
        X = torch.as_tensor(X)
        Y = torch.as_tensor(Y)
        MLPSurrogate.set_normalization(self, X.reshape(-1, X.shape[-1]), Y.reshape(-1, Y.shape[-1]))

    def _gemm(self, M, N, K, A, lda, Bm, ldb, bias, C, ldc, Cb=None, ldcb=0):
        nat.check(self.lib.dtb_mlp_gemm_bf16_nt(M, N, K, A.data_ptr(), lda, Bm.data_ptr(), ldb, nat.ptr(bias), 0,
                                                nat.ptr(C), ldc, nat.ptr(Cb), ldcb, self._stream()))

    def _forward(self, X, h0):
        """X [T, r, n_in] (r <= max_batch rows, padded to B); h0 [r, H] or None."""
        s = self._stream()
        T, r = X.shape[0], X.shape[1]
        assert T <= self.max_steps and r <= self.max_batch
        B = _pad(r)
        H, I, O = self.H, self.I, self.O
        X = torch.as_tensor(X).to(self.dev, torch.float32)
        Xp = X.expand(T, r, self.n_in).contiguous()
        if r < B:
            Xp = torch.zeros((T, B, self.n_in), dtype=torch.float32, device=self.dev)
            Xp[:, :r] = X
        nat.check(self.lib.dtb_mlp_affine(T * B, self.n_in, I, Xp.data_ptr(), self.n_in, self.x_scale.data_ptr(),
                                          self.x_shift.data_ptr(), None, self.Xb.data_ptr(), I, s))
        self._gemm(T * B, 3 * H, I, self.Xb, I, self.pb["W_ih"], I, self.p["b_ih"], self.Gi, 3 * H)
        if h0 is not None:
            h0 = torch.as_tensor(h0).to(self.dev, torch.float32).expand(r, H).contiguous()
        if self.sequence:
            nat.check(self.lib.dtb_gru_sequence_forward(T, B, H, self.Gi.data_ptr(), self.pb["W_hh"].data_ptr(),
                                                        self.p["b_hh"].data_ptr(), nat.ptr(h0), r, self.Gh.data_ptr(),
                                                        self.Hs.data_ptr(), self.Hb.data_ptr(), s))
        else:
            self.Hs[:B].zero_()
            if h0 is not None:
                self.Hs[:r].copy_(h0)
            nat.check(self.lib.dtb_mlp_f32_to_bf16(B * H, self.Hs.data_ptr(), self.Hb.data_ptr(), s))
            for t in range(T):
                hb = self.Hb[t * B:(t + 1) * B]
                gh = self.Gh[t * B:(t + 1) * B]
                self._gemm(B, 3 * H, H, hb, H, self.pb["W_hh"], H, self.p["b_hh"], gh, 3 * H)
                nat.check(self.lib.dtb_gru_forward(B, H, self.Gi[t * B:].data_ptr(), gh.data_ptr(),
                                                   self.Hs[t * B:].data_ptr(), self.Hs[(t + 1) * B:].data_ptr(),
                                                   self.Hb[(t + 1) * B:].data_ptr(), s))
        self._gemm(T * B, O, H, self.Hb[B:], H, self.pb["W_o"], H, self.p["b_o"], self.Y, O)
        return T, r, B

    def predict(self, X, h0=None):
        """X [T, rows, n_in] -> (Y [T, rows, n_out] denormalised, h_T [rows, H])."""
        T, r, B = self._forward(X, h0)
        out = torch.empty((T * B, self.n_out), dtype=torch.float32, device=self.dev)
        nat.check(self.lib.dtb_mlp_affine(T * B, self.n_out, self.n_out, self.Y.data_ptr(), self.O,
                                          self._y_std.data_ptr(), self._y_mean.data_ptr(), out.data_ptr(), None,
                                          self.n_out, self._stream()))
        return out.reshape(T, B, -1)[:, :r], self.Hs[T * B:T * B + r].clone()

    def gradients(self, X, Y, mask=None, h0=None):
        """BPTT over one batch of sequences; loss sum(mask (Yn-Tn)^2) / (2 T rows)."""
        s = self._stream()
        T, r, B = self._forward(X, h0)
        H, I, O = self.H, self.I, self.O
        TB = T * B
        Yd = _broadcast(Y, (T, r, self.n_out), self.dev)
        Md = None if mask is None else _broadcast(mask, (T, r, self.n_out), self.dev)
        nat.check(self.lib.dtb_mlp_sequence_loss(T, B, O, r, self.n_out, self.Y.data_ptr(), Yd.data_ptr(),
                                                 self.y_scale.data_ptr(), self.y_shift.data_ptr(), nat.ptr(Md),
                                                 1.0 / (T * r), self.Gy.data_ptr(), self.Gyb.data_ptr(),
                                                 self.lsum.data_ptr(), s))
        self._gemm(TB, H, O, self.Gyb, O, self.pbT["W_o"], O, None, self.dHo, H)
        # recurrence, last step first
        if self.sequence:
            nat.check(self.lib.dtb_gru_sequence_backward(
                T, B, H, self.Gi.data_ptr(), self.Gh.data_ptr(), self.Hs.data_ptr(), self.dHo.data_ptr(),
                self.pbT["W_hh"].data_ptr(), self.dGib.data_ptr(), self.dGhb.data_ptr(), self.dG.data_ptr(),
                s))
            dg = self.dG.data_ptr()
            sums = np.array([(2 * H, 4 * H, dg, self.grad["b_ih"].data_ptr(), self.grad["b_hh"].data_ptr()),
                             (H, 4 * H, dg + 8 * H, self.grad["b_ih"].data_ptr() + 8 * H, 0),
                             (H, 4 * H, dg + 12 * H, self.grad["b_hh"].data_ptr() + 8 * H, 0),
                             (O, O, self.Gy.data_ptr(), self.grad["b_o"].data_ptr(), 0)], dtype=np.int64)
            nat.check(self.lib.dtb_mlp_column_sums(len(sums), sums.ctypes.data, TB, s))
        else:
            for t in range(T - 1, -1, -1):
                last = t == T - 1
                nat.check(self.lib.dtb_gru_backward(
                    B, H, self.Gi[t * B:].data_ptr(), self.Gh[t * B:].data_ptr(), self.Hs[t * B:].data_ptr(),
                    self.dHo[t * B:].data_ptr(), None if last else self.dhz.data_ptr(),
                    None if last else self.dhg.data_ptr(), self.dGi[t * B:].data_ptr(), self.dGib[t * B:].data_ptr(),
                    self.dGh[t * B:].data_ptr(), self.dGhb[t * B:].data_ptr(), self.dhz.data_ptr(), s))
                if t > 0:
                    self._gemm(B, H, 3 * H, self.dGhb[t * B:(t + 1) * B], 3 * H, self.pbT["W_hh"], 3 * H, None,
                               self.dhg, H)
            nat.check(self.lib.dtb_mlp_bias_grad(TB, 3 * H, self.dGi.data_ptr(), self.grad["b_ih"].data_ptr(), s))
            nat.check(self.lib.dtb_mlp_bias_grad(TB, 3 * H, self.dGh.data_ptr(), self.grad["b_hh"].data_ptr(), s))
            nat.check(self.lib.dtb_mlp_bias_grad(TB, O, self.Gy.data_ptr(), self.grad["b_o"].data_ptr(), s))
        # weight gradients over all T*B rows, from transposed operands in fragment order
        KH = (T + 1) * B  # the states before (first T*B) and after (last T*B) every step
        pack = np.array([(TB, O, O, self.Gyb.data_ptr(), self.GybT.data_ptr()),
                         (KH, H, H, self.Hb.data_ptr(), self.HbT.data_ptr()),
                         (TB, I, I, self.Xb.data_ptr(), self.XbT.data_ptr()),
                         (TB, 3 * H, 3 * H, self.dGib.data_ptr(), self.dGiT.data_ptr()),
                         (TB, 3 * H, 3 * H, self.dGhb.data_ptr(), self.dGhT.data_ptr())], dtype=np.int64)
        nat.check(self.lib.dtb_mlp_pack_transposed(len(pack), pack.ctypes.data, s))
        dw = np.array([(H, O, KH, TB, 0, self.HbT.data_ptr() + 2 * 32 * B, self.GybT.data_ptr(), 0,
                        self.grad["W_o"].data_ptr(), 0),
                       (I, 3 * H, TB, TB, 0, self.XbT.data_ptr(), self.dGiT.data_ptr(), 0,
                        self.grad["W_ih"].data_ptr(), 0),
                       (H, 3 * H, KH, TB, 0, self.HbT.data_ptr(), self.dGhT.data_ptr(), 0,
                        self.grad["W_hh"].data_ptr(), 0)], dtype=np.int64)
        nat.check(self.lib.dtb_mlp_weight_gradients(len(dw), dw.ctypes.data, TB, s))
        # the partial sums this batch wrote (the buffer is sized for the longest, largest batch)
        return self.lsum[: (TB * O + 255) // 256]

    def step(self):
        self.t += 1
        table = _params([(w.shape[0] if w.dim() == 2 else 1, w.shape[-1], w, self.grad[k], self.m[k], self.v[k],
                          self.pb.get(k), self.pbT.get(k), None, None) for k, w in self.p.items()])
        nat.check(self.lib.dtb_mlp_adam_multi(len(table), table.ctypes.data, self.lr, self.b1, self.b2, self.eps,
                                              self.t, self._stream()))

    def fit(self, X, Y, epochs=50, batch=None, seed=0):
        """X [T, n, n_in], Y [T, n, n_out] sequences; mini-batches over n."""
        X = torch.as_tensor(X).to(self.dev, torch.float32)
        Y = torch.as_tensor(Y).to(self.dev, torch.float32)
        n = X.shape[1]
        batch = min(self.max_batch, n) if batch is None else int(batch)
        g = torch.Generator().manual_seed(seed)
        hist = []
        for _ in range(epochs):
            perm = torch.randperm(n, generator=g).to(self.dev)
            tot = torch.zeros((), dtype=torch.float64, device=self.dev)
            nb = 0
            for r0 in range(0, n - batch + 1, batch):
                idx = perm[r0:r0 + batch]
                ls = self.gradients(X.index_select(1, idx), Y.index_select(1, idx))
                tot += ls.sum().double() / (batch * X.shape[0])
                self.step()
                nb += 1
            hist.append(float(tot) / max(1, nb) / self.n_out)
        return hist

    def params_numpy(self):
        return {k: v.cpu().double().numpy() for k, v in self.p.items()}


def gemm_kernel_name(M, N, K):
    """The kernel dtb_mlp_gemm_bf16_nt dispatches an M x N x K product to:
    LDS-staged square tiles of 256, 128 or 64 (the fewest rounds of
    workgroups, weighed by a round's time, and smaller ones for a short K; 64
    with K in four ranges where there are fewer than 256 such tiles), or below
    128 tiles of 64, or up to 256 of 32, the 32x32 tiles with K split over the
    four wavefronts."""
    def tiles(t):
        return -(-M // t) * -(-N // t)

    if tiles(64) < 128 or (tiles(64) < 256 and tiles(32) <= 256):
        return "gemm_nt_splitk_kernel (32x32 tiles, K split over 4 wavefronts, bf16 MFMA, FP32 accumulate)"
    if tiles(64) < 256:
        return "gemm_nt_tile_kernel<1> (64x64 LDS-staged tiles, K in 4 ranges, bf16 MFMA, FP32 accumulate)"
    if tiles(128) < 256 or K <= 192 or (K <= 256 and tiles(256) <= 2304):
        t = 1
    else:
        t = 4 if 7 * -(-tiles(256) // 256) <= 4 * -(-tiles(128) // 512) else 2
    return f"gemm_nt_tile_kernel<{t}> ({64 * t}x{64 * t} LDS-staged tiles, bf16 MFMA, FP32 accumulate)"


def gemm_throughput(M, N, K, reps=50, warmup=5, device=0):
    """Time dtb_mlp_gemm_bf16_nt (C = A·Bᵀ, bf16 operands, FP32 out) on
    random operands: HIP events on the stream the kernel is launched on.
    The product is first checked against torch in FP32 (bf16 inputs are
    exact in FP32; only the summation order differs).  Returns a dict with
    the average microseconds per launch and TFLOP/s (2·M·N·K per launch)."""
    nat.require_gpu()
    if M % 32 or N % 32 or K % 16 or min(M, N, K) <= 0:
        raise ValueError("M and N must be positive multiples of 32 and K of 16")
    lib = nat.lib()
    dev = torch.device("cuda", device)
    g = torch.Generator(device="cpu").manual_seed(0)
    A = torch.randn(M, K, generator=g).to(torch.bfloat16).to(dev)
    B = torch.randn(N, K, generator=g).to(torch.bfloat16).to(dev)
    C = torch.empty(M, N, dtype=torch.float32, device=dev)
    s = torch.cuda.current_stream(dev)

    def launch():
        nat.check(lib.dtb_mlp_gemm_bf16_nt(M, N, K, A.data_ptr(), K, B.data_ptr(), K, None, 0, C.data_ptr(), N, None,
                                           0, s.cuda_stream))

    launch()
    ref = A.float() @ B.float().T
    err = float((C - ref).abs().max() / ref.abs().max())
    if not err < 1e-5:
        raise RuntimeError(f"GEMM {M}x{N}x{K} differs from torch: relative error {err:.3g}")
    for _ in range(warmup):
        launch()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record(s)
    for _ in range(reps):
        launch()
    e1.record(s)
    e1.synchronize()
    us = e0.elapsed_time(e1) * 1e3 / reps
    return {"M": M, "N": N, "K": K, "us": us, "tflops": 2.0 * M * N * K / us * 1e-6, "max_rel_err": err}


if __name__ == "__main__":
    import argparse
    import json

    ap = argparse.ArgumentParser(description="surrogate GEMM throughput")
    ap.add_argument("--gemm", type=int, nargs=3, action="append", metavar=("M", "N", "K"), required=True)
    ap.add_argument("--reps", type=int, default=50)
    for shape in ap.parse_args().gemm:
        print(json.dumps(gemm_throughput(*shape, reps=ap.parse_args().reps)), flush=True)
