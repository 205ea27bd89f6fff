"""Dense MLP trained and evaluated with the library's BF16 MFMA GEMM (gh_gemm_bf16).

Every matrix product of the forward and backward passes runs in hand-written kernels with
FP32 accumulation: networks with equal hidden widths of 128 or 256 take one launch forward
and three backward (csrc/mlp_train.hip), any other a GEMM launch per product (csrc/mlp.hip)
with bias, ReLU and the ReLU derivative in its epilogues. PyTorch holds the tensors (device
memory, the FP32 master weights, the Adam state and the loss), nothing more.

Layer l: Z_l = X_l W_l + b_l (FP32), X_{l+1} = bf16(relu(Z_l)) for hidden layers,
the last layer is linear. Backward: G_L = dLoss/dZ_L, dW_l = X_l^T G_l,
db_l = sum_m G_l, G_{l-1} = (G_l W_l^T) * relu'(Z_{l-1}).
"""
import ctypes as C
import struct

import numpy as np

from .. import _abi as A

EPI_STORE, EPI_BIAS_RELU, EPI_BIAS, EPI_DRELU = 0, 1, 2, 3


def _torch():
    import torch

    return torch


# the C layouts of gh_adam_tensor and gh_adam_pack
_ADAM = struct.Struct("=5Q4ifi")
_PACK = struct.Struct("=2Q2i")


def _pointers(tensors):
    """Device addresses of tensors as a C array of pointers."""
    return struct.pack(f"={len(tensors)}Q", *[0 if t is None else t.data_ptr() for t in tensors])


def pad(n, q):
    return (n + q - 1) // q * q


def pad8(n):
    return pad(n, 8)


def fragment_order(w, out):
    """Matrix w [N][K] into out, a flat bf16 buffer in fragment order (include/gatehip.h): N
    padded to 16, K to 32 with zeros. Returns out."""
    torch = _torch()
    n, k = w.shape
    t = torch.zeros(pad(n, 16), pad(k, 32), device=w.device, dtype=torch.bfloat16)
    t[:n, :k] = w
    # (n tile, n, k step, k group, k) -> (n tile, k step, k group, n, k)
    out.view(t.shape[0] // 16, t.shape[1] // 32, 4, 16, 8).copy_(
        t.view(t.shape[0] // 16, 16, t.shape[1] // 32, 4, 8).permute(0, 2, 3, 1, 4))
    return out


class MLP:
    """sizes = [in, hidden..., out]; inputs/outputs padded to multiples of 8 internally."""

    def __init__(self, sizes, device="cuda", seed=0, lr=1e-3, betas=(0.9, 0.999), eps=1e-8, weight_decay=0.0):
        torch = _torch()
        self.lib = A.load_library()
        self.sizes = list(sizes)
        self.dev = torch.device(device)
        self.f32 = torch.float32
        self.psizes = [pad8(s) for s in sizes]
        g = torch.Generator(device="cpu").manual_seed(seed)
        self.W, self.b = [], []
        for k, n, pk, pn in zip(self.sizes[:-1], self.sizes[1:], self.psizes[:-1], self.psizes[1:]):
            w = torch.zeros(pk, pn)
            w[:k, :n] = torch.randn(k, n, generator=g) * np.sqrt(2.0 / k)
            self.W.append(w.to(self.dev))
            self.b.append(torch.zeros(pn, device=self.dev))
        self.lr, self.betas, self.eps, self.wd = lr, betas, eps, weight_decay
        self.m = [torch.zeros_like(t) for t in self.W + self.b]
        self.v = [torch.zeros_like(t) for t in self.W + self.b]
        self.t = 0
        self._refresh()

    # ------------------------------------------------------------------ helpers
    PACK_MAX_TENSORS = 32  # of one gh_pack_weights or gh_adam_step_packed call

    def _refresh(self):
        """bf16 copies of the weights (kept in place: the optimiser kernel writes them): row-major
        and, for the fused kernels, the forward (W^T) and backward (W) copies in fragment order."""
        torch = _torch()
        if getattr(self, "W16", None) is None or [t.shape for t in self.W16] != [w.shape for w in self.W]:
            self.W16 = [torch.empty(w.shape, device=self.dev, dtype=torch.bfloat16) for w in self.W]
            self.Wf = self.Wb = None
            if self.fused_ok():
                sizes = [pad(w.shape[1], 16) * pad(w.shape[0], 32) for w in self.W16]
                sizes += [pad(w.shape[0], 16) * pad(w.shape[1], 32) for w in self.W16[1:]]
                copies = torch.zeros(sum(sizes), device=self.dev, dtype=torch.bfloat16).split(sizes)
                L = len(self.W16)
                self.Wf, self.Wb = list(copies[:L]), [None, *copies[L:]]
        # one launch for tensors that it can read as they are: FP32 rows of full width where it is launched
        if self.dev.type == "cuda" and 0 < len(self.W) <= self.PACK_MAX_TENSORS and all(
                w.is_contiguous() and w.dtype == torch.float32 and w.shape[0] % 8 == 0 and
                w.device.index == torch.cuda.current_device() for w in self.W):
            tab = [_ADAM.pack(w.data_ptr(), 0, 0, 0, t.data_ptr(), *w.shape, 0, 0, 0.0, 0)
                   for w, t in zip(self.W, self.W16)]
            rc = self.lib.gh_pack_weights(b"".join(tab), b"".join(map(self._pack, range(len(tab)))), len(tab),
                                          self._stream())
            if rc != 0:
                raise RuntimeError(f"gh_pack_weights failed ({rc})")
            return
        for t, w in zip(self.W16, self.W):
            t.copy_(w)
        if self.Wf is not None:
            for l, w in enumerate(self.W16):
                fragment_order(w.t(), self.Wf[l])
                if l:
                    fragment_order(w, self.Wb[l])

    def _pack(self, l):
        """gh_adam_pack of weight l."""
        if self.Wf is None:
            return _PACK.pack(0, 0, 0, 0)
        return _PACK.pack(self.Wf[l].data_ptr(), self.Wb[l].data_ptr() if l else 0, pad(self.W[l].shape[0], 32),
                          pad(self.W[l].shape[1], 32))

    def _stream(self):
        return C.c_void_p(_torch().cuda.current_stream().cuda_stream)

    def _gemm(self, a, sam, sak, b, sbk, sbn, M, N, K, bias=None, zprev=None, ldz=0, c32=None, c16=None, ldc=0,
              mode=EPI_STORE):
        p = lambda t: C.c_void_p(t.data_ptr()) if t is not None else C.c_void_p()  # noqa: E731
        rc = self.lib.gh_gemm_bf16(p(a), sam, sak, p(b), sbk, sbn, M, N, K, p(bias), p(zprev), ldz, p(c32), p(c16),
                                   ldc, mode, self._stream())
        if rc != 0:
            raise RuntimeError(f"gh_gemm_bf16 failed ({rc})")

    def n_params(self):
        return sum(int(np.prod(s)) for s in zip(self.sizes[:-1], self.sizes[1:])) + sum(self.sizes[1:])

    def flops_forward(self, batch):
        return 2.0 * batch * sum(k * n for k, n in zip(self.sizes[:-1], self.sizes[1:]))

    # ------------------------------------------------------------------ passes
    def forward(self, x, keep=True):
        """x: (M, in) float tensor on the device, or an already padded contiguous
        (M, in padded) bf16 tensor. Returns (M, out) FP32."""
        torch = _torch()
        M = x.shape[0]
        if x.dtype == torch.bfloat16 and x.shape[1] == self.psizes[0] and x.is_contiguous():
            X = x
        else:
            X = torch.zeros(M, self.psizes[0], device=self.dev, dtype=torch.bfloat16)
            X[:, : self.sizes[0]] = x.to(torch.bfloat16)
        if self._train_fused(X):
            return self._forward_fused(X, keep)
        xs, zs = [X], []
        L = len(self.W)
        for l in range(L):
            K, N = self.psizes[l], self.psizes[l + 1]
            Z = torch.empty(M, N, device=self.dev, dtype=torch.float32)
            if l < L - 1:
                Y = torch.empty(M, N, device=self.dev, dtype=torch.bfloat16)
                self._gemm(xs[-1], K, 1, self.W16[l], N, 1, M, N, K, bias=self.b[l], c32=Z, c16=Y, ldc=N,
                           mode=EPI_BIAS_RELU)
                xs.append(Y)
            else:
                self._gemm(xs[-1], K, 1, self.W16[l], N, 1, M, N, K, bias=self.b[l], c32=Z, ldc=N, mode=EPI_BIAS)
            zs.append(Z)
        if keep:
            self._xs, self._zs = xs, zs
        return zs[-1][:, : self.sizes[-1]]

    def infer(self, X, out, bufs):
        """Inference without keeping activations: X (M, in padded) bf16, out (M, out padded)
        FP32, bufs two bf16 buffers of at least (M, widest hidden layer). Hidden layers write
        only their bf16 activations."""
        M = X.shape[0]
        cur = X
        L = len(self.W)
        for l in range(L):
            K, N = self.psizes[l], self.psizes[l + 1]
            if l < L - 1:
                Y = bufs[l % 2].view(-1)[: M * N].view(M, N)
                self._gemm(cur, K, 1, self.W16[l], N, 1, M, N, K, bias=self.b[l], c16=Y, ldc=N, mode=EPI_BIAS_RELU)
                cur = Y
            else:
                self._gemm(cur, K, 1, self.W16[l], N, 1, M, N, K, bias=self.b[l], c32=out, ldc=out.stride(0),
                           mode=EPI_BIAS)
        return out

    # ------------------------------------------------------------------ fused inference
    FUSED_K_IN, FUSED_N_OUT, FUSED_MAX_LAYERS = 32, 16, 8
    TRAIN_MAX_ROWS = 4194240  # GH_MLP_TRAIN_MAX_ROWS
    COLUMN_SUMS_MAX_ROWS = 65536  # GH_COLUMN_SUMS_MAX_ROWS

    def fused_ok(self):
        """gh_mlp_forward_packed_bf16 handles 2..8 layers with equal hidden widths of 128 or 256,
        at most 32 inputs and 16 outputs."""
        hidden = set(self.psizes[1:-1])
        return (2 <= len(self.W) <= self.FUSED_MAX_LAYERS and len(hidden) == 1 and hidden <= {128, 256}
                and self.psizes[0] <= self.FUSED_K_IN and self.psizes[-1] <= self.FUSED_N_OUT)

    def _fused_args(self):
        """Pointer arrays (bytes) of the forward weight copies and the biases; what was made for
        them stays referenced by the returned list."""
        if len(self.b) < len(self.W):
            raise IndexError("a bias for every layer is needed")
        f32, hold, at = self.f32, [], []
        for b in self.b:
            p = b.data_ptr()
            if p & 15 or b.dtype is not f32 or not b.is_contiguous():
                b = b.to(f32, copy=True).contiguous()
                hold.append(b)
                p = b.data_ptr()
            at.append(p)
        return _pointers(self.Wf), struct.pack(f"={len(at)}Q", *at), hold

    def _train_fused(self, X):
        """gh_mlp_train_* take the network and this batch."""
        return self.Wf is not None and 1 <= X.shape[0] <= self.TRAIN_MAX_ROWS and X.data_ptr() % 16 == 0

    def _forward_fused(self, X, keep):
        torch = _torch()
        M, L = X.shape[0], len(self.W)
        Z = torch.empty(M, self.psizes[-1], device=self.dev, dtype=torch.float32)
        if not keep:
            return self.infer_fused(X, Z)[:, : self.sizes[-1]]
        Xt = torch.empty(pad(M, 32), self.FUSED_K_IN, device=self.dev, dtype=torch.bfloat16)
        Y = torch.empty(L - 1, pad(M, 32), self.psizes[1], device=self.dev, dtype=torch.bfloat16)
        wp, bp, hold = self._fused_args()
        rc = self.lib.gh_mlp_train_forward_bf16(X.data_ptr(), M, L, self.psizes[0], self.psizes[1], self.sizes[-1],
                                                wp, bp, Xt.data_ptr(), _pointers(Y), Z.data_ptr(), Z.stride(0),
                                                self._stream())
        del hold
        if rc != 0:
            raise RuntimeError(f"gh_mlp_train_forward_bf16 failed ({rc})")
        self._xs, self._zs = (M, Xt, Y), None
        return Z[:, : self.sizes[-1]]

    def _backward_fused(self, grad_out, tensor_sums):
        torch = _torch()
        (M, Xt, Y), L = self._xs, len(self.W)
        k_in, hidden, n_out, n_pad = self.psizes[0], self.psizes[1], self.sizes[-1], self.psizes[-1]
        G, G32 = grad_out, None
        # (rows that overlap, as those of an expanded gradient, are laid out: the kernels take a row pitch)
        if (G.dtype != torch.float32 or G.shape != (M, n_out) or G.device != Xt.device or G.stride(1) != 1 or
                G.stride(0) < n_out):
            G = torch.empty(M, n_out, device=self.dev, dtype=torch.float32)
            G[:] = grad_out
        if tensor_sums:
            G32 = torch.empty(L - 1, M, hidden, device=self.dev, dtype=torch.float32)
        shapes = [tuple(w.shape) for w in self.W]
        flat = torch.empty(sum(k * n for k, n in shapes), device=self.dev, dtype=torch.float32)
        dbf = torch.empty((L - 1) * hidden + n_pad, device=self.dev, dtype=torch.float32)
        size = C.c_int64()
        rc = self.lib.gh_mlp_train_workspace(M, L, k_in, hidden, n_pad, C.byref(size))
        if rc != 0:
            raise RuntimeError(f"gh_mlp_train_workspace failed ({rc})")
        ws = torch.empty(size.value, device=self.dev, dtype=torch.uint8)
        rc = self.lib.gh_mlp_train_backward_bf16(Xt.data_ptr(), M, L, k_in, hidden, n_out, n_pad, _pointers(self.Wb),
                                                 _pointers(Y), G.data_ptr(), G.stride(0), flat.data_ptr(),
                                                 dbf.data_ptr(), None if G32 is None else _pointers(G32),
                                                 ws.data_ptr(), size.value, self._stream())
        if rc != 0:
            raise RuntimeError(f"gh_mlp_train_backward_bf16 failed ({rc})")
        dW, o = [], 0
        for k, n in shapes:
            dW.append(flat[o:o + k * n].view(k, n))
            o += k * n
        db = list(dbf.split([n for _, n in shapes]))
        if tensor_sums and M <= self.COLUMN_SUMS_MAX_ROWS and n_pad <= 256 and n_pad & (n_pad - 1) == 0:
            grads, widths, pads = [*G32, G], [hidden] * (L - 1) + [n_out], [hidden] * (L - 1) + [n_pad]
            work = torch.empty(256 * sum(pads), device=self.dev, dtype=torch.float32)
            rc = self.lib.gh_column_sums(_pointers(grads), struct.pack(f"={L}q", *[g.stride(0) for g in grads]),
                                         struct.pack(f"={L}i", *widths), struct.pack(f"={L}i", *pads), L, M,
                                         _pointers(db), work.data_ptr(), work.numel(), self._stream())
            if rc != 0:
                raise RuntimeError(f"gh_column_sums failed ({rc})")
        elif tensor_sums:
            Gp = torch.zeros(M, n_pad, device=self.dev, dtype=torch.float32)
            Gp[:, :n_out] = G
            db = [g.sum(0) for g in (*G32, Gp)]
        return dW, db

    def infer_fused(self, X, out):
        """All layers in one kernel (gh_mlp_forward_packed_bf16): X (M, in padded) bf16 with row
        pitch X.stride(0), out (M, >= out) FP32 with row pitch out.stride(0); only the
        first sizes[-1] columns of out are written. Same values as infer()."""
        wp, bp, hold = self._fused_args()
        rc = self.lib.gh_mlp_forward_packed_bf16(X.data_ptr(), X.stride(0), X.shape[0], len(self.W), self.psizes[0],
                                          self.psizes[1], self.sizes[-1], wp, bp, out.data_ptr(), out.stride(0),
                                          self._stream())
        del hold
        if rc != 0:
            raise RuntimeError(f"gh_mlp_forward_packed_bf16 failed ({rc})")
        return out

    def backward(self, grad_out, tensor_sums=False):
        """grad_out: dLoss/dOutput (M, out) FP32. Returns [dW...], [db...] (FP32, padded).
        tensor_sums: take the bias gradients as column sums of the FP32 gradients in the order of
        gh_column_sums (that of PyTorch 2.10.0's sum), the bits of the layer-by-layer path, instead of the kernels' own sums (2e-7 apart)."""
        torch = _torch()
        if self._zs is None:
            return self._backward_fused(grad_out, tensor_sums)
        M = grad_out.shape[0]
        L = len(self.W)
        G32 = torch.zeros(M, self.psizes[-1], device=self.dev, dtype=torch.float32)
        G32[:, : self.sizes[-1]] = grad_out
        G16 = G32.to(torch.bfloat16)
        dW, db = [None] * L, [None] * L
        for l in range(L - 1, -1, -1):
            K, N = self.psizes[l], self.psizes[l + 1]
            dw = torch.empty(K, N, device=self.dev, dtype=torch.float32)
            # dW = X^T G : (K x M) (M x N)
            self._gemm(self._xs[l], 1, K, G16, N, 1, K, N, M, c32=dw, ldc=N, mode=EPI_STORE)
            dW[l] = dw
            db[l] = G32.sum(0)
            if l > 0:
                Gp32 = torch.empty(M, K, device=self.dev, dtype=torch.float32)
                Gp16 = torch.empty(M, K, device=self.dev, dtype=torch.bfloat16)
                # G_{l-1} = (G W^T) * relu'(Z_{l-1}) : (M x N) (N x K)
                self._gemm(G16, N, 1, self.W16[l], 1, N, M, K, N, zprev=self._zs[l - 1], ldz=K, c32=Gp32, c16=Gp16,
                           ldc=K, mode=EPI_DRELU)
                G32, G16 = Gp32, Gp16
        return dW, db

    def step(self, dW, db):
        """Adam update of the FP32 master weights and biases in one kernel (gh_adam_step),
        which also keeps the padding at zero and writes the bf16 weight copies (both layouts)."""
        params = self.W + self.b
        grads = list(dW) + list(db)
        if len(grads) < len(params):
            raise RuntimeError("a gradient for every weight and bias is needed")
        self.t += 1
        valid = [(k, n) for k, n in zip(self.sizes[:-1], self.sizes[1:])] + [(1, n) for n in self.sizes[1:]]
        tab, packs = [], []
        L = len(self.W)
        for i, (p, g, (vr, vc)) in enumerate(zip(params, grads, valid)):
            if g.shape != p.shape or not g.is_contiguous() or g.dtype != p.dtype:
                raise ValueError("gradient shape / layout differs from its parameter")
            rows, cols = (p.shape[0], p.shape[1]) if p.dim() == 2 else (1, p.shape[0])
            is_w = i < L
            tab.append(_ADAM.pack(p.data_ptr(), g.data_ptr(), self.m[i].data_ptr(), self.v[i].data_ptr(),
                                  self.W16[i].data_ptr() if is_w else 0, rows, cols, vr, vc,
                                  float(self.wd) if is_w else 0.0, 0))
            packs.append(self._pack(i) if is_w else _PACK.pack(0, 0, 0, 0))
        b1, b2 = self.betas
        rc = self.lib.gh_adam_step_packed(b"".join(tab), b"".join(packs), len(params), float(self.lr), float(b1),
                                          float(b2), float(self.eps), self.t, self._stream())
        if rc != 0:
            raise RuntimeError(f"gh_adam_step_packed failed ({rc})")

    def state_dict(self):
        return {"sizes": self.sizes, "W": [w.cpu() for w in self.W], "b": [b.cpu() for b in self.b]}

    def load_state_dict(self, d):
        """Weights and biases of any floating type, with or without the padding."""
        self.W = [self._filled(w, self.sizes[l:l + 2], self.psizes[l:l + 2]) for l, w in enumerate(d["W"])]
        self.b = []
        for l, b in enumerate(d["b"]):
            b = self._filled(b.reshape(-1), self.sizes[l + 1:l + 2], self.psizes[l + 1:l + 2])
            self.b.append(b.expand(self.W[l].shape[1]).contiguous() if b.numel() == 1 and l < len(self.W) else b)
        self._refresh()

    def _filled(self, t, sizes, full):
        """t in FP32 on the device, padded with zeros if it has the network's own sizes."""
        t = t.to(self.dev, _torch().float32)
        if list(t.shape) != sizes or sizes == full:
            return t
        out = _torch().zeros(full, device=self.dev)
        out[tuple(slice(n) for n in sizes)] = t
        return out
