"""Thin numpy-facing wrappers over the C ABI: a device `Tensor` (pooled HIP buffer + shape +
dtype) and one function per kernel entry point.  Shapes follow the reference's op judges
(core/source/dopt/core/ops/{basic,math,nnet}.d); all arithmetic happens in libdopthip.so.
"""
import ctypes as C
import functools

import numpy as np

from . import capi

_F32 = np.dtype(np.float32)
_DT = {_F32: capi.F32, np.dtype(np.int32): capi.I32}

# A call of a short kernel takes the host as long as the device, 2.3 us of it the launch itself.  So what follows from shapes
# alone - volumes, ctypes arrays, convolution descriptors - is made once per shape (by value; nothing of a tensor is kept), and
# the common case of a result tensor of the very shape is one comparison.


def _vol(shape):
    v = 1
    for s in shape:
        v *= int(s)
    return v


@functools.lru_cache(maxsize=4096)
def _sizes(shape):
    """capi.sizes of a tuple; shared, so for arguments that the library only reads."""
    return capi.sizes(shape)


class Tensor:
    """A dense row-major device tensor owning a pooled buffer (the HIPBuffer of this backend)."""

    def __init__(self, shape, dtype=np.float32, _ptr=None, _owner=None):
        self.shape = tuple([int(s) for s in shape])
        self.dtype = dtype if dtype is _F32 else np.dtype(dtype)
        self.code = _DT.get(self.dtype)
        if self.code is None:
            raise capi.HipError(3, "Element type not supported.")
        self.size = _vol(self.shape)
        self.nbytes = self.size * 4
        self._owner = _owner
        if _ptr is not None:
            self.ptr = _ptr
        else:
            p = C.c_void_p()
            _run(capi.load().dopt_hip_malloc(C.byref(p), self.nbytes))
            self.ptr = p.value or 0

    def set(self, array):
        a = np.ascontiguousarray(array, dtype=self.dtype)
        if a.nbytes != self.nbytes:
            raise capi.HipError(1, "input buffer is the wrong length.")
        _run(capi.load().dopt_hip_copy_h2d(self.ptr, a.ctypes.data, a.nbytes))
        return self

    def numpy(self):
        out = np.empty(self.shape, self.dtype)
        _run(capi.load().dopt_hip_copy_d2h(out.ctypes.data, self.ptr, self.nbytes))
        return out

    def reshape(self, shape):
        """Aliases the same buffer (the reference's `reshape` has no kernel either)."""
        if _vol(shape) != self.size:
            raise ValueError("reshape changes the volume")
        return Tensor(shape, self.dtype, _ptr=self.ptr, _owner=self)

    def view(self, offset, shape):
        """Sub-buffer starting `offset` elements in (packed batch-norm outputs)."""
        if offset + _vol(shape) > self.size:
            raise ValueError("view out of range")
        return Tensor(shape, self.dtype, _ptr=self.ptr + 4 * offset, _owner=self)

    def free(self):
        if self._owner is None and self.ptr:
            capi.load().dopt_hip_free(self.ptr)
        self.ptr = 0

    def __del__(self):
        try:
            self.free()
        except Exception:
            pass


def _run(rc):
    if rc:
        capi.check(rc)


def tensor(array, dtype=None):
    a = np.ascontiguousarray(array, dtype=dtype)
    if a.dtype == np.float64:
        a = a.astype(np.float32)
    if a.dtype == np.int64:
        a = a.astype(np.int32)
    return Tensor(a.shape, a.dtype).set(a)


def sync():
    _run(capi.load().dopt_hip_sync())


def _out(out, shape, dtype=_F32):
    """The result tensor: a fresh zero-filled pooled buffer, or the caller's (a kernel's `execute`
    is handed its output buffer by the plan, cuda/package.d:68-79)."""
    if out is None:
        return Tensor(shape, dtype)
    if out.shape == shape and out.dtype == dtype:
        return out
    if _vol(out.shape) != _vol(shape) or out.dtype != np.dtype(dtype):
        raise capi.HipError(1, "output buffer has the wrong size or type")
    return out


# ------------------------------------------------------------------------------- pointwise

def pointwise(op, a, b=None, out=None):
    out = _out(out, a.shape, a.dtype)
    if b is not None and (b.shape != a.shape or b.dtype != a.dtype):
        raise capi.HipError(1, "pointwise operands must have the same type")
    _run(capi.load().dopt_hip_pointwise(op.encode(), a.code, a.size, a.ptr, b.ptr if b is not None else None, out.ptr))
    return out


def pointwise_chain(inputs, nodes, out=None, kinds=None, inner=0):
    """One kernel for a DAG of pointwise nodes.  inputs: tensors; a one-element tensor among longer
    ones is broadcast.  kinds (optional, per input): 0 full tensor, 1 one element, 2 one element per
    row, 3 one element per column of the [n / inner, inner] view.  nodes: (op, lhs, rhs-or-None) with
    operand indices counting the inputs first and then the nodes; the last node is the result."""
    n = max(t.size for t in inputs)
    full = next(t for t in inputs if t.size == n)
    if kinds is None:
        kinds = [1 if (t.size == 1 and n != 1) else 0 for t in inputs]
    if any(t.size != n and k == 0 for t, k in zip(inputs, kinds)) or any(t.dtype != full.dtype for t in inputs):
        raise capi.HipError(1, "pointwise operands must have the same type")
    out = _out(out, full.shape, full.dtype)
    k = len(nodes)
    _run(capi.load().dopt_hip_pointwise_chain(
        full.code, n, inner, len(inputs), (C.c_void_p * len(inputs))(*[t.ptr for t in inputs]),
        (C.c_ubyte * len(inputs))(*kinds), k, (C.c_char_p * k)(*[nd[0].encode() for nd in nodes]),
        (C.c_int * k)(*[nd[1] for nd in nodes]), (C.c_int * k)(*[-1 if nd[2] is None else nd[2] for nd in nodes]), out.ptr))
    return out


@functools.lru_cache(maxsize=4096)
def _kept(shape, axes):
    """The axes (all of them where none are named) and the shape of what is left."""
    axes = axes or tuple(range(len(shape)))
    return axes, tuple([s for i, s in enumerate(shape) if i not in axes])


def _axes(axes):
    return tuple([int(x) for x in axes]) if axes else ()


def _reduce(name, a, axes, out=None):
    axes, oshape = _kept(a.shape, _axes(axes))
    out = _out(out, oshape, a.dtype)
    _run(capi.load().dopt_hip_reduce(name, a.code, _sizes(a.shape), len(a.shape), _sizes(axes), len(axes), a.ptr, out.ptr))
    return out


def sum(a, axes=None, out=None):  # noqa: A001 - reference op name
    return _reduce(b"sum", a, axes, out)


def max_element(a, axes=None, out=None):
    return _reduce(b"maxElement", a, axes, out)


def sum_of_squares(a, axes=None, out=None):
    """sum(mul(a, a), axes) without storing the product: same value as the two operations."""
    axes, oshape = _kept(a.shape, _axes(axes))
    out = _out(out, oshape, a.dtype)
    _run(capi.load().dopt_hip_reduce_squares(_sizes(a.shape), len(a.shape), _sizes(axes), len(axes), a.ptr, out.ptr))
    return out


def argmin(a, axis, out=None):
    oshape = list(a.shape)
    oshape[axis] = 1
    out = _out(out, tuple(oshape), np.int32)
    _run(capi.load().dopt_hip_argmin(a.code, _sizes(a.shape), len(a.shape), axis, a.ptr, out.ptr))
    return out


# ------------------------------------------------------------------------------- layout

def slice(a, start, stop, out=None):  # noqa: A001
    oshape = tuple([e - s for s, e in zip(start, stop)])
    out = _out(out, oshape, a.dtype)
    _run(capi.load().dopt_hip_slice(len(a.shape), _sizes(a.shape), _sizes(oshape), _sizes(tuple(start)), a.ptr, out.ptr))
    return out


def pad(a, before, after, out=None):
    oshape = tuple([b + s + e for b, s, e in zip(before, a.shape, after)])
    out = _out(out, oshape, a.dtype)
    _run(capi.load().dopt_hip_pad(len(a.shape), _sizes(a.shape), _sizes(oshape), _sizes(tuple(before)), a.ptr, out.ptr))
    return out


def repeat(a, reps, out=None):
    oshape = tuple([s * r for s, r in zip(a.shape, reps)])
    out = _out(out, oshape, a.dtype)
    _run(capi.load().dopt_hip_repeat(len(a.shape), _sizes(a.shape), _sizes(tuple(reps)), a.ptr, out.ptr))
    return out


def transpose(a, out=None):
    rows, cols = a.shape
    out = _out(out, (cols, rows), a.dtype)
    _run(capi.load().dopt_hip_transpose2d(rows, cols, a.ptr, out.ptr))
    return out


# ------------------------------------------------------------------------------- dense / conv

def matmul(a, b, out=None):
    if a.dtype != np.float32 or b.dtype != np.float32:
        raise capi.HipError(3, "Element type not supported.")
    M, K = a.shape
    K2, N = b.shape
    if K != K2:
        raise capi.HipError(1, "matmul: inner dimensions differ")
    out = _out(out, (M, N))
    _run(capi.load().dopt_hip_sgemm(M, N, K, a.ptr, b.ptr, out.ptr))
    return out


def matmul_t(a, b, trans_a=False, trans_b=False, out=None):
    """op(a) . op(b): trans_a / trans_b read the operand transposed (a stored [K, M], b stored [N, K])."""
    K, M = (a.shape if trans_a else a.shape[::-1])
    N, K2 = (b.shape if trans_b else b.shape[::-1])
    if K != K2:
        raise capi.HipError(1, "matmul: inner dimensions differ")
    out = _out(out, (M, N))
    _run(capi.load().dopt_hip_sgemm_t(int(trans_a), int(trans_b), M, N, K, a.ptr, b.ptr, out.ptr))
    return out


def matmul_rank1(a, b, u, v, relu=False, trans_a=False, trans_b=False, out=None):
    """op(a) . op(b) + u[M,1] . v[1,N], then relu: a dense layer in one kernel (u, v may both be None)."""
    K, M = (a.shape if trans_a else a.shape[::-1])
    N, K2 = (b.shape if trans_b else b.shape[::-1])
    if K != K2:
        raise capi.HipError(1, "matmul: inner dimensions differ")
    out = _out(out, (M, N))
    _run(capi.load().dopt_hip_sgemm_rank1(int(trans_a), int(trans_b), M, N, K, a.ptr, b.ptr,
                                                u.ptr if u is not None else None, v.ptr if v is not None else None,
                                                int(bool(relu)), out.ptr))
    return out


def conv_desc(xshape, wshape, padding=(0, 0), stride=(1, 1)):
    N, Cc, H, W = xshape
    K, C2, R, S = wshape
    if Cc != C2:
        raise capi.HipError(1, "convolution: channel counts differ")
    return capi.ConvDesc(N, Cc, H, W, K, R, S, padding[0], padding[1], stride[0], stride[1])


def conv_out_shape(d):
    return (d.N, d.K, (d.H + 2 * d.padH - d.R) // d.strideH + 1, (d.W + 2 * d.padW - d.S) // d.strideW + 1)


@functools.lru_cache(maxsize=4096)
def _conv(xshape, wshape, padding, stride):
    """(reference to the descriptor, shape of the result); shared, the library only reads it."""
    d = conv_desc(xshape, wshape, padding, stride)
    return C.byref(d), conv_out_shape(d)


def convolution(x, w, padding=(0, 0), stride=(1, 1), out=None):
    d, oshape = _conv(x.shape, w.shape, tuple(padding), tuple(stride))
    y = _out(out, oshape)
    _run(capi.load().dopt_hip_conv_fwd(d, x.ptr, w.ptr, y.ptr))
    return y


def convolution_bias(x, w, bias, padding=(0, 0), stride=(1, 1), out=None):
    """addBias(convolution(x, w), bias) in one pass."""
    d, oshape = _conv(x.shape, w.shape, tuple(padding), tuple(stride))
    y = _out(out, oshape)
    _run(capi.load().dopt_hip_conv_fwd_bias(d, x.ptr, w.ptr, bias.ptr, y.ptr))
    return y


def conv_bwd_data(dy, w, xshape, padding=(0, 0), stride=(1, 1), out=None):
    d, oshape = _conv(tuple(xshape), w.shape, tuple(padding), tuple(stride))
    if dy.shape != oshape:
        raise capi.HipError(1, "convolutionFeaturesGrad: gradient shape does not match")
    dx = _out(out, tuple(xshape))
    _run(capi.load().dopt_hip_conv_bwd_data(d, dy.ptr, w.ptr, dx.ptr))
    return dx


def conv_bwd_filter(dy, x, wshape, padding=(0, 0), stride=(1, 1), out=None):
    d, oshape = _conv(x.shape, tuple(wshape), tuple(padding), tuple(stride))
    if dy.shape != oshape:
        raise capi.HipError(1, "convolutionFiltersGrad: gradient shape does not match")
    dw = _out(out, tuple(wshape))
    _run(capi.load().dopt_hip_conv_bwd_filter(d, dy.ptr, x.ptr, dw.ptr))
    return dw


# ------------------------------------------------------------------------------- NN ops

def _nci(shape):
    inner = _vol(shape[2:]) if len(shape) > 2 else 1
    return shape[0], shape[1], inner


def maxpool(x, dims, out=None):
    N, Cc, H, W = x.shape
    y = _out(out, (N, Cc, H // dims[0], W // dims[1]))
    _run(capi.load().dopt_hip_maxpool_fwd(N, Cc, H, W, dims[0], dims[1], x.ptr, y.ptr))
    return y


def maxpool_grad(dy, x, dims, out=None):
    N, Cc, H, W = x.shape
    dx = _out(out, x.shape)
    _run(capi.load().dopt_hip_maxpool_bwd(N, Cc, H, W, dims[0], dims[1], dy.ptr, x.ptr, dx.ptr))
    return dx


def softmax(x, out=None):
    y = _out(out, x.shape)
    _run(capi.load().dopt_hip_softmax_fwd(*_nci(x.shape), x.ptr, y.ptr))
    return y


def softmax_grad(dy, y, out=None):
    dx = _out(out, y.shape)
    _run(capi.load().dopt_hip_softmax_bwd(*_nci(y.shape), dy.ptr, y.ptr, dx.ptr))
    return dx


def relu(x, out=None):
    y = _out(out, x.shape)
    _run(capi.load().dopt_hip_relu_fwd(x.size, x.ptr, y.ptr))
    return y


def relu_grad(dy, x, out=None):
    dx = _out(out, x.shape)
    _run(capi.load().dopt_hip_relu_bwd(x.size, dy.ptr, x.ptr, dx.ptr))
    return dx


def add_bias(x, b, out=None):
    y = _out(out, x.shape)
    _run(capi.load().dopt_hip_bias_fwd(*_nci(x.shape), x.ptr, b.ptr, y.ptr))
    return y


def add_bias_grad(dy, out=None):
    db = _out(out, (dy.shape[1],))
    _run(capi.load().dopt_hip_bias_bwd(*_nci(dy.shape), dy.ptr, db.ptr))
    return db


def bn_train(x, scale, bias, run_mean, run_var, momentum, out=None):
    N, Cc, inner = _nci(x.shape)
    packed = _out(out, (x.size + 2 * Cc,))
    _run(capi.load().dopt_hip_bn_train(N, Cc, inner, float(momentum), x.ptr, scale.ptr, bias.ptr, run_mean.ptr,
                                             run_var.ptr, packed.ptr))
    return packed


def bn_train_relu(x, scale, bias, run_mean, run_var, momentum, out=None):
    """batchNormTrain whose y part already went through relu."""
    N, Cc, inner = _nci(x.shape)
    packed = _out(out, (x.size + 2 * Cc,))
    _run(capi.load().dopt_hip_bn_train_relu(N, Cc, inner, float(momentum), x.ptr, scale.ptr, bias.ptr,
                                                  run_mean.ptr, run_var.ptr, packed.ptr))
    return packed


def bn_grad_relu(dy, y, x, scale, out=None):
    """batchNormGrad(reluGrad(dy, y, .), x, scale): y is the relu output."""
    N, Cc, inner = _nci(x.shape)
    packed = _out(out, (x.size + 2 * Cc,))
    _run(capi.load().dopt_hip_bn_grad_relu(N, Cc, inner, dy.ptr, y.ptr, x.ptr, scale.ptr, packed.ptr))
    return packed


def bn_train_pool(x, scale, bias, run_mean, run_var, momentum, relu=True, out=None, pooled=None):
    """batchNormTrain (+ relu) and maxpool(y, [2, 2]) in one call: (packed, pooled)."""
    N, Cc, H, W = x.shape
    packed = _out(out, (x.size + 2 * Cc,))
    pooled = _out(pooled, (N, Cc, H // 2, W // 2))
    _run(capi.load().dopt_hip_bn_train_pool(N, Cc, H, W, float(momentum), x.ptr, None, scale.ptr, bias.ptr,
                                                  run_mean.ptr, run_var.ptr, packed.ptr, 1 if relu else 0, pooled.ptr))
    return packed, pooled


def bn_grad_pool(dpooled, y, x, scale, out=None, dx_sum=None):
    """batchNormGrad(reluGrad(maxpoolGrad(dpooled, ., y), y, .), x, scale)."""
    N, Cc, H, W = x.shape
    packed = _out(out, (x.size + 2 * Cc,))
    _run(capi.load().dopt_hip_bn_grad_pool(N, Cc, H, W, dpooled.ptr, y.ptr, x.ptr, scale.ptr, packed.ptr,
                                                 dx_sum.ptr if dx_sum is not None else None))
    return packed


def bn_grad(dy, x, scale, out=None):
    N, Cc, inner = _nci(x.shape)
    packed = _out(out, (x.size + 2 * Cc,))
    _run(capi.load().dopt_hip_bn_grad(N, Cc, inner, dy.ptr, x.ptr, scale.ptr, packed.ptr))
    return packed


def bn_infer(x, scale, bias, mean, var, out=None):
    y = _out(out, x.shape)
    _run(capi.load().dopt_hip_bn_infer(*_nci(x.shape), x.ptr, scale.ptr, bias.ptr, mean.ptr, var.ptr, y.ptr))
    return y


# ------------------------------------------------------------------------------- optimizers

class FusedOptimizer:
    """Multi-tensor in-place updater over fixed parameter / gradient / state tensors."""

    def __init__(self, params, grads, m, v=None, vhat=None, skip=None):
        n = len(params)
        refs = (capi.TensorRef * max(n, 1))()
        for i in range(n):
            refs[i] = capi.TensorRef(params[i].ptr, grads[i].ptr, m[i].ptr, v[i].ptr if v else None,
                                     vhat[i].ptr if vhat else None, params[i].size,
                                     1 if (skip and skip[i]) else 0)
        self._keep = (params, grads, m, v, vhat)
        h = C.c_void_p()
        _run(capi.load().dopt_hip_optim_create(n, refs, C.byref(h)))
        self._h = h
        self.b1 = C.c_float(1.0)   # online/adam.d:44-45: b1, b2 start at 1
        self.b2 = C.c_float(1.0)

    def sgd(self, lr=0.01, mu=0.0, nesterov=False):
        _run(capi.load().dopt_hip_sgd_step(self._h, lr, mu, int(nesterov)))

    def adam(self, alpha=1e-3, beta1=0.9, beta2=0.999, eps=1e-8):
        _run(capi.load().dopt_hip_adam_step(self._h, alpha, beta1, beta2, eps, C.byref(self.b1),
                                                  C.byref(self.b2)))

    def amsgrad(self, alpha=1e-3, beta1=0.9, beta2=0.999, eps=1e-8):
        _run(capi.load().dopt_hip_amsgrad_step(self._h, alpha, beta1, beta2, eps, C.byref(self.b1),
                                                     C.byref(self.b2)))

    def close(self):
        if self._h:
            capi.load().dopt_hip_optim_destroy(self._h)
            self._h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass
