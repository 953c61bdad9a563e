"""``QuantLinear`` with the reference's constructor, buffers and ``forward`` contract
(auto_gptq/nn_modules/qlinear.py:20-75,177-247; selected by ``make_quant(..., use_tvm=True)`` in
auto_gptq/modeling/_utils.py:59-89), computing on hand-written HIP kernels.

Differences from the reference's TVM-backed module (auto_gptq/nn_modules/qlinear_tvm.py), on
purpose: the buffers are the standard AutoGPTQ ones (int32 ``qweight``/``qzeros``, ``g_idx``), the
constructor compiles nothing and touches no GPU (so it works under ``init_empty_weights``), and
``forward`` neither pads M nor allocates a padded output.
"""
from __future__ import annotations

import math

import numpy as np
import torch
import torch.nn as nn

from . import _lib, ops
from .pack import pack_qweight, pack_qzeros, tiled_qualifies


class _ProductWithInputGrad(torch.autograd.Function):
    """The product with a gradient for x (the packed weights are constants): grad_x = grad_y @ W^T, which
    is what the reference's Triton back end offers for training on top of quantised layers
    (auto_gptq/nn_modules/qlinear_triton.py:195-273,298-336): fused on the transposed tiled copy
    (``QuantLinear.grad_input``), or the HIP dequant kernel and the library GEMM for long batches and
    layers the format does not cover."""

    @staticmethod
    def forward(ctx, x2, layer):
        ctx.layer = layer
        return layer._product(x2)

    @staticmethod
    def backward(ctx, grad_out):
        return ctx.layer.grad_input(grad_out), None


class QuantLinear(nn.Module):
    SUPPORTED_BITS = (2, 3, 4, 8)   # the widths of the format (qlinear.py:31-32)
    FUSED_BITS = (3, 4)             # those the kernels on the checkpoint layout cover; 2 and 8 run fused on the
                                    # tiled format only (else as dequant + library GEMM)

    SWITCH_ROWS, GRAD_SWITCH_ROWS = 1152, 384   # the measured defaults of the two switches to the library GEMM

    def __init__(self, bits, groupsize, infeatures, outfeatures, bias, kernel_switch_threshold=SWITCH_ROWS,
                 sort_for_decode=True, tile_for_prefill=True):
        super().__init__()
        if bits not in self.SUPPORTED_BITS:
            raise NotImplementedError("Only 2,3,4,8 bits are supported.")
        if infeatures % 32 != 0 or outfeatures % 32 != 0:
            raise ValueError("infeatures and outfeatures must be multiples of 32")
        self.infeatures = infeatures
        self.outfeatures = outfeatures
        self.bits = bits
        self.groupsize = groupsize if groupsize != -1 else infeatures
        self.maxq = 2 ** self.bits - 1
        # Rows of x from which forward() materialises W (HIP dequant kernel) and calls the library
        # GEMM instead of the fused kernels, as the reference does (qlinear.py:25,198: default 128
        # there).  Measured on MI355X, fused against dequant + library GEMM, weights cold:
        #   * tiled kernels (act-order or not), 4096x11008 int4 / int3: 117 / 117 vs 148 / 135 us at 768 rows,
        #     125 / 118 vs 141 / 140 at 1024, 165 / 152 vs 152 / 148 at 1280; 4096x4096: 54 vs 67 at 1024, 86 vs
        #     73 at 1280; 8192x8192: 172 vs 193 at 1024, 226 vs 219 at 1280.  Hence 1152 (nine row blocks);
        #   * kernels on the checkpoint layout (layers off the tiled route): contiguous groups 124 vs 139 us
        #     at 768 rows, 152 vs 146 at 1024; activation order 126 vs 130 at 640 rows, 139 vs 133 at 768.
        #     Hence 1024 and 640 there.
        # 0 or None disables the switch.  The measured default stands between the kernels above and the library: calls
        # that the panel kernel is the fastest for run there on both sides of it.  Any other value sends every
        # call of that many rows to the library, as in the reference.
        self.kernel_switch_threshold = kernel_switch_threshold
        self.plain_switch_threshold = 1024
        self.act_order_switch_threshold = 640

        groups = math.ceil(infeatures / self.groupsize)
        self.register_buffer("qweight", torch.zeros((infeatures // 32 * bits, outfeatures), dtype=torch.int32))
        self.register_buffer("qzeros", torch.zeros((groups, outfeatures // 32 * bits), dtype=torch.int32))
        self.register_buffer("scales", torch.zeros((groups, outfeatures), dtype=torch.float16))
        self.register_buffer("g_idx", (torch.arange(infeatures, dtype=torch.int64) // self.groupsize).to(torch.int32))
        if bias:
            self.register_buffer("bias", torch.zeros((outfeatures,), dtype=torch.float16))
        else:
            self.bias = None
        self._g_state = None  # (g_idx identity, contiguous?, groups of equal size?) cached by _kernel_g_idx
        # Activation-order layers: on the first decode-size call (up to 16 rows of x), keep a second
        # copy of qweight with the input channels sorted by group (plus a [K] int32 map), which the
        # decode kernel reads faster than it can follow g_idx.  Costs the layer's packed size again in
        # device memory; False keeps only the checkpoint's tensors.
        self.sort_for_decode = sort_for_decode
        self._sorted = None   # (key, (qweight_sorted, kmap) or None)
        # Every fused layer whose groups are whole multiples of 32 channels: on the first call with a row count
        # the tiled kernels are faster at (the library's routing rule, gptq_hip_select_route), keep a copy of the layer in
        # the order the matrix instructions consume (gptq_hip_tile_prepare); the first gradient for x adds the transposed
        # one.  Each costs the layer's packed size again, and the call that builds it its preparation (prepare_tiled /
        # prepare_transposed do it up front); False keeps the checkpoint's tensors (and the sorted copy) only, and long
        # batches then run as dequant + library GEMM.  compact() makes the tiled copy the only one.
        self.tile_for_prefill = tile_for_prefill
        self._tiled = None    # (key, (qtile, sz, xsrc, kinv) or None)
        self._tiled_t = None  # (key, (qtile_t, szt, xsrc) or None): the copy the gradient for x runs on
        # rows of grad_y from which the gradient for x takes the library GEMM (default and own values as above)
        self.grad_switch_threshold = self.GRAD_SWITCH_ROWS
        self._compact = False
        self._routes = {}     # M -> (watched buffers, sum of their versions, path name, fn(x2)): see _route

    # ------------------------------------------------------------------ packing
    def pack(self, linear, scales, zeros, g_idx=None):
        """Quantises ``linear.weight`` with the given per-group ``scales``/``zeros`` ([N, G], as the
        reference passes them) and fills the packed buffers.  Follows qlinear.py:77-175:
        ``q = round((W + s*z) / s)`` per input channel, codes packed along K, ``z - 1`` along N."""
        W = linear.weight.data.clone()
        if isinstance(linear, nn.Conv2d):
            W = W.flatten(1)
        elif type(linear).__name__ == "Conv1D":  # transformers.pytorch_utils.Conv1D keeps [in, out]
            W = W.t()
        if g_idx is not None:
            self.g_idx = g_idx.clone().to(torch.int32)
        scales = scales.t().contiguous()
        zeros = zeros.t().contiguous()
        scale_zeros = zeros * scales
        self.scales = scales.clone().half()
        if linear.bias is not None:
            self.bias = linear.bias.clone().half()
        g = self.g_idx.long().cpu()
        # same arithmetic as the reference's per-column loop: (W[:, k] + (s*z)[g]) / half(s)[g]
        num = W.t().cpu() + scale_zeros[g].cpu()
        intweight = torch.round(num / self.scales[g].cpu()).to(torch.int32)
        self.qweight = torch.from_numpy(pack_qweight(intweight.numpy().astype(np.uint32), self.bits))
        self.qzeros = torch.from_numpy(pack_qzeros(zeros.cpu().numpy().astype(np.int64), self.bits))
        self._g_state = None

    # ------------------------------------------------------------------ forward
    def _kernel_g_idx(self):
        """``None`` when ``g_idx`` is the contiguous ``k // groupsize`` (lets the kernels skip the
        gather), else the tensor.  Checked once per distinct g_idx storage: the first call of a layer waits for the GPU
        here, once for all that its routes and copies want to know of g_idx."""
        g = self.g_idx
        key = (g.data_ptr(), g._version, g.device)
        if self._g_state is None or self._g_state[0] != key:
            K, gs = self.infeatures, self.groupsize
            groups = math.ceil(K / gs)
            host = g.detach().cpu().numpy()     # (some tens of KB; a dozen small kernels for the same answers take longer)
            contiguous = np.array_equal(host, np.repeat(np.arange(groups, dtype=np.int32), gs)[:K])
            whole = K % gs == 0
            if not contiguous:
                lo, hi = int(host.min()), int(host.max())
                if lo < 0 or hi >= groups:
                    raise ValueError(f"g_idx values must lie in [0, {groups}), found [{lo}, {hi}]")
                whole = bool((np.bincount(host, minlength=groups) == gs).all())
            self._g_state = (key, contiguous, whole)
        if self._g_state[1]:
            return None
        if not g.is_contiguous() or g.data_ptr() % 16 != 0 or g.dtype != torch.int32:
            # the kernels read g_idx four entries at a time
            self.g_idx = g.to(torch.int32).contiguous().clone()
            self._g_state = None
            return self._kernel_g_idx()
        return g

    def prepare_decode(self):
        """Builds (once per distinct qweight / g_idx storage) the sorted copy used by decode-size
        calls; returns ``(qweight_sorted, kmap)`` or None when the layer has no activation order or
        does not qualify.  ``forward`` calls this lazily; loaders may call it up front."""
        g = self._kernel_g_idx()
        q = self.qweight
        key = (q.data_ptr(), q._version, None if g is None else (g.data_ptr(), g._version))
        if self._sorted is None or self._sorted[0] != key:
            tensors = None
            if g is not None and q.device.type == "cuda":
                tensors = self._sort_on_gpu(q, g)
            self._sorted = (key, tensors)
        return self._sorted[1]

    def _whole_groups(self):
        """The one check the preparation kernels cannot make: every group holds exactly ``groupsize`` channels."""
        self._kernel_g_idx()
        return self._g_state[2]

    def _sort_on_gpu(self, q, g):
        """``pack.sort_channels_by_group`` through the library's own kernels (gptq_hip_sort_channels)."""
        K, gs = self.infeatures, self.groupsize
        klane = 8 if self.bits == 4 else 32
        if K >= 65536 or K % gs != 0 or gs % klane != 0 or not self._whole_groups():
            return None
        return ops.sort_channels(q, g, self.bits, self.groupsize)

    def prepare_tiled(self):
        """Builds (once per distinct storage of the packed tensors) the layer in the tiled format; returns
        ``(qtile, sz, xsrc, kinv)`` or None when the format does not cover the layer.  ``forward`` calls this
        lazily; loaders may call it up front (the first look at g_idx, for the check of the group sizes, waits for
        the GPU)."""
        if self._compact:
            return self._tiled[1]
        g = self._kernel_g_idx()
        key = tuple((t.data_ptr(), t._version) for t in (self.qweight, self.qzeros, self.scales)) + (
            None if g is None else (g.data_ptr(), g._version),)
        if self._tiled is None or self._tiled[0] != key:
            tensors = None
            if (self.qweight.device.type == "cuda"
                    and tiled_qualifies(self.infeatures, self.outfeatures, self.bits, self.groupsize)
                    and (g is None or self._whole_groups())):
                tensors = ops.tile_prepare(self.qweight, self.qzeros, self.scales, g, self.bits, self.groupsize)
            self._tiled = (key, tensors)
        return self._tiled[1]

    def prepare_transposed(self):
        """Builds (once per distinct storage of the packed tensors) the copy the transposed product runs on;
        returns ``(qtile_t, szt, xsrc)`` or None when the tiled format does not cover the layer.  A compact layer
        keeps the copy it had when it was compacted (its checkpoint tensors are gone)."""
        if self._compact:
            return None if self._tiled_t is None else self._tiled_t[1]
        tiled = self.prepare_tiled()
        if tiled is None:
            return None
        key = self._tiled[0]
        if self._tiled_t is None or self._tiled_t[0] != key:
            xsrc = tiled[2] if self._kernel_g_idx() is not None else None
            qtile_t, szt = ops.tile_prepare_transposed(self.qweight, self.qzeros, self.scales, xsrc, self.bits,
                                                       self.groupsize)
            self._tiled_t = (key, (qtile_t, szt, xsrc))
        return self._tiled_t[1]

    def grad_input(self, grad_out: torch.Tensor) -> torch.Tensor:
        """grad_out[..., outfeatures] @ W^T: below the switch to the library GEMM the fused transposed product
        (gptq_hip_gemm_tiled_transposed), else W from the dequant kernel and the library GEMM."""
        gy = grad_out.reshape(-1, self.outfeatures)
        if gy.dtype != torch.float16:
            gy = gy.half()
        if not gy.is_contiguous():
            gy = gy.contiguous()
        gy = ops.aligned(gy)
        M = gy.size(0)
        # The panel kernel where the library says so; else the matmul kernel's transposed form below the switch.  Measured on
        # MI355X (us, eager, int4 with an activation order; the latter against dequant + library GEMM):
        # 4096 x 11008: 22 / 64 at 16 rows, 37 / 90 at 128; 11008 x 4096: 35 / 66 at 128; 4096 x 4096: 27 / 44 at 128.
        gx = None
        if self.tile_for_prefill and gy.is_cuda and M > 0:
            K, N, bits, gs = self.infeatures, self.outfeatures, self.bits, self.groupsize
            past, asked = False, False
            if self.kernel_switch_threshold and self.grad_switch_threshold:
                for rows, default in ((self.kernel_switch_threshold, self.SWITCH_ROWS),
                                      (self.grad_switch_threshold, self.GRAD_SWITCH_ROWS)):
                    if M >= rows:
                        past, asked = True, asked or rows != default
            plan = (_lib.select_panel(M, K, N, bits, gs, self._kernel_g_idx() is not None, transposed=True)
                    if not asked and tiled_qualifies(K, N, bits, gs) else None)
            if plan is not None or not past:
                t = self.prepare_transposed()
                if t is not None:
                    if plan is None:   # (named here, so that it is not asked for again below)
                        plan = _lib.select_tiled_transposed(M, K, N, bits, gs)
                    gx = ops.gemm_tiled_transposed(gy, t[0], t[1], t[2], K, bits, gs, plan=plan)
        if gx is None:
            if self._compact:
                raise RuntimeError("this layer keeps only its tiled copy (compact()) and has no copy for the gradient "
                                   "of its input: call prepare_transposed() before compact(), or load the model with "
                                   "keep_checkpoint_tensors=True")
            gx = torch.matmul(gy, self.dequantize().t())
        return gx.reshape(grad_out.shape[:-1] + (self.infeatures,))

    def compact(self):
        """Keeps the tiled copy as the layer's ONLY weights: every row count then runs on the tiled kernels and
        the checkpoint's tensors are released (empty buffers stay in their place, so ``state_dict`` no longer
        holds the layer: save before, or reload).  Returns True when the layer is compact afterwards."""
        if self._compact:
            return True
        tensors = self.prepare_tiled()
        if tensors is None:
            return False
        act = self._kernel_g_idx() is not None
        self._tiled = (None, tensors if act else (tensors[0], tensors[1], None, None))
        self._compact = True
        self._sorted = None
        if self._tiled_t is not None:   # a copy for the gradient that exists stays with the layer
            self._tiled_t = (None, self._tiled_t[1])
        dev = self.qweight.device
        self.qweight = torch.empty((0, self.outfeatures), dtype=torch.int32, device=dev)
        self.qzeros = torch.empty((0, self.qzeros.shape[1]), dtype=torch.int32, device=dev)
        self.scales = torch.empty((0, self.outfeatures), dtype=torch.float16, device=dev)
        return True

    def _apply(self, fn, *args, **kwargs):
        # the tiled copy of a compact layer is its weights: it moves with the module (a prepared copy beside
        # the checkpoint tensors is rebuilt instead, when their storage changes)
        super()._apply(fn, *args, **kwargs)
        self._routes.clear()
        if self._compact:
            self._tiled = (None, tuple(None if t is None else fn(t) for t in self._tiled[1]))
            if self._tiled_t is not None and self._tiled_t[1] is not None:
                self._tiled_t = (None, tuple(None if t is None else fn(t) for t in self._tiled_t[1]))
        return self

    # ------------------------------------------------------------------ copying, pickling
    def __getstate__(self):
        """A route holds bound C++ launch objects and closures over this module's tensors: a copy of the module
        (``copy.deepcopy``, ``pickle``, ``torch.save(model)``) gets none of them and decides its routes again.
        Prepared copies beside the checkpoint tensors are rebuilt by the copy as well; the tiled copy of a compact
        layer IS its weights and travels."""
        state = dict(self.__dict__)
        state["_routes"] = {}
        state["_g_state"] = None
        state["_sorted"] = None
        if not self._compact:
            state["_tiled"] = None
            state["_tiled_t"] = None
        return state

    def __setstate__(self, state):
        super().__setstate__(state)

    # ------------------------------------------------------------------ routing
    def __setattr__(self, name, value):
        # any change of a buffer or a switch may change where a row count goes: forget the routes
        if name != "_routes":
            routes = self.__dict__.get("_routes")
            if routes:
                routes.clear()
        super().__setattr__(name, value)

    def _watched(self):
        """The buffers whose contents a route may have baked into a prepared copy."""
        return (self.qweight, self.qzeros, self.scales, self.g_idx)

    def _route(self, M):
        """(what, fn): the product for M rows as one call fn(x2), and the name of the path it takes: "tiled",
        "sorted", "plain" (the checkpoint's own tensors) or "library" (the dequant kernel + library GEMM).  Decided
        once per row count and state of the buffers; the operators are torch.ops.gptq_hip.* (csrc/binding.cpp)."""
        t = torch.ops.gptq_hip
        bits, gs, bias = self.bits, self.groupsize, self.bias

        def bind(kind, a, b, c, d, e):
            if ops.CALL is not None:
                # the operator library binds the layer's constant tensors and the plan for M once: one argument per call
                return ops.CALL.BoundCall(kind, a, b, c, d, e, bias, bits, gs, M, self.infeatures, self.outfeatures)
            if kind == 0:
                return lambda x2: t.gemm.default(x2, a, b, c, d, bias, bits, gs)
            if kind == 1:
                return lambda x2: t.gemm_sorted.default(x2, a, b, c, d, bias, bits, gs)
            return lambda x2: t.gemm_tiled.default(x2, a, b, d, e, bias, bits, gs)

        if self._compact:
            qtile, sz, xsrc, kinv = self._tiled[1]
            return "tiled", bind(2, qtile, sz, None, xsrc, kinv)

        def library(x2):
            # Long prompts (kernel_switch_threshold), 2- and 8-bit layers, or a shape the fused kernels do
            # not cover (activation order with more groups than their LDS table holds): materialise W with
            # the HIP dequant kernel and multiply with the library GEMM, which is what the reference
            # does above its threshold (auto_gptq/nn_modules/qlinear.py:198-245).  Still GPU only.
            out = torch.matmul(x2, self.dequantize())
            return out if bias is None else out + bias

        g = self._kernel_g_idx()
        K, N = self.infeatures, self.outfeatures
        # Which copy the call runs on is the library's decision (gptq_hip_select_route): this module says which
        # copies it may hold and from how many rows it prefers the library GEMM, and builds the copy that was
        # chosen; a copy that the layer's contents do not allow (groups of unequal size) is taken off the offer
        # and the question asked again.
        copies = _lib.COPY_CHECKPOINT
        if self.sort_for_decode and self.bits in self.FUSED_BITS:
            copies |= _lib.COPY_SORTED
        if self.tile_for_prefill:
            copies |= _lib.COPY_TILED | _lib.COPY_TILED_PANEL
        switch_rows = (self.kernel_switch_threshold or 0,
                       self.plain_switch_threshold if self.kernel_switch_threshold else 0,
                       self.act_order_switch_threshold if self.kernel_switch_threshold else 0)
        while True:
            r = _lib.select_route(M, K, N, bits, gs, g is not None, copies, switch_rows)
            if r.copy == _lib.ROUTE_TILED:
                tiled = self.prepare_tiled()
                if tiled is None:
                    copies &= ~(_lib.COPY_TILED | _lib.COPY_TILED_PANEL)
                    continue
                xsrc, kinv = (tiled[2], tiled[3]) if g is not None else (None, None)
                return "tiled", bind(2, tiled[0], tiled[1], None, xsrc, kinv)
            if r.copy == _lib.ROUTE_SORTED:
                srt = self.prepare_decode()
                if srt is None:
                    copies &= ~_lib.COPY_SORTED
                    continue
                return "sorted", bind(1, srt[0], self.qzeros, self.scales, srt[1], None)
            if r.copy == _lib.ROUTE_CHECKPOINT:
                return "plain", bind(0, self.qweight, self.qzeros, self.scales, g, None)
            return "library", library

    def route(self, M: int) -> str:
        """The path a call with M rows takes (see ``_route``); builds the prepared copy it needs."""
        return self._routed(M)[2]

    def _fresh(self, r):
        """Whether a cached route still describes the module: the same buffer objects (code that swaps a buffer
        through ``module._buffers[name] = t`` passes ``__setattr__`` by), not written since."""
        a, b, c, d = r[0]
        buf = self._buffers
        return (a is buf["qweight"] and b is buf["qzeros"] and c is buf["scales"] and d is buf["g_idx"]
                and a._version + b._version + c._version + d._version == r[1])

    def _routed(self, M):
        r = self._routes.get(M)
        if r is not None and self._fresh(r):
            return r
        # (a route is not part of what is being recorded, nor is a copy that it prepares)
        what, fn = self._route(M) if ops.CALL is None else ops.CALL.aside(self._route, M)
        w = self._watched()               # (read after routing: the preparations may have re-made g_idx)
        r = (w, sum(t._version for t in w), what, fn)
        self._routes[M] = r
        return r

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        # (the common case, a contiguous fp16 x whose row count was seen before, does not come here: the call of the module
        # is a C function that runs the bound product itself)
        out_shape = x.shape[:-1] + (self.outfeatures,)
        x2 = x.reshape(-1, x.shape[-1])
        if x2.dtype != torch.float16:
            x2 = x2.half()
        if not x2.is_contiguous():
            x2 = x2.contiguous()
        if x2.requires_grad and torch.is_grad_enabled():
            out = _ProductWithInputGrad.apply(x2, self)   # e.g. adapters trained on top of frozen layers
        else:
            out = self._product(x2)
        return out.reshape(out_shape)

    def _product(self, x2: torch.Tensor) -> torch.Tensor:
        """y[M, N] = x2[M, K] @ W + bias for a contiguous fp16 x2."""
        M = x2.shape[0]
        if M == 0:
            return x2.new_empty((0, self.outfeatures))
        return self._routed(M)[3](x2)

    def dequantize(self) -> torch.Tensor:
        """fp16 [infeatures, outfeatures], the weight the reference materialises on every call."""
        if self._compact:
            # the tiled kernels form the same rounded fp16 weights: the product with the identity is W itself,
            # taken 1024 rows of the identity at a time (a debugging aid: it costs a K-row product)
            qtile, sz, xsrc, kinv = self._tiled[1]
            K, dev = self.infeatures, qtile.device
            w = torch.empty((K, self.outfeatures), dtype=torch.float16, device=dev)
            for k0 in range(0, K, 1024):
                rows = min(1024, K - k0)
                eye = torch.zeros((rows, K), dtype=torch.float16, device=dev)
                eye[torch.arange(rows, device=dev), torch.arange(k0, k0 + rows, device=dev)] = 1
                ops.gemm_tiled(eye, qtile, sz, xsrc, kinv, None, self.bits, self.groupsize, out=w[k0:k0 + rows])
            return w
        return ops.dequant(self.qweight, self.qzeros, self.scales, self._kernel_g_idx(), self.bits, self.groupsize)

    def extra_repr(self) -> str:
        return (f"bits={self.bits}, groupsize={self.groupsize}, infeatures={self.infeatures}, "
                f"outfeatures={self.outfeatures}, bias={self.bias is not None}")


if ops.CALL is not None:
    # the module call of the common case as one C function (csrc/python_call.cpp); it comes back to nn.Module.__call__
    # and forward for everything else
    ops.CALL.install(QuantLinear)


__all__ = ["QuantLinear"]
