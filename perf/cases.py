"""Measured cases: what a user of this framework has it do, through its public entry points.

A case is one of eight kinds of work, each of them a call or a short sequence of calls as a user's program makes them:

  dot             Tensor product into a tensor the program owns (`gemm`), any transposition
  dense           Dense.forward with bias and relu: inference, and the forward half of training
  dense_backward  the three products of Dense's backward edge: dx = dy.W^T, dW = x^T.dy, db = sum of dy's rows
  conv            Conv2.forward with bias and relu
  conv_backward   Conv2's backward edge: dW = gm^T.im2col(x), dx = col2im(gm.W), gm the gradient as [bs*oh*ow, oc]
  pool            MaxPool2 forward, then its backward in place on a clone of the input
  lenet_infer     LeNet5 logits of a batch, as one launch or layer by layer
  lenet_train     one LeNet5 training step with momentum, replayed from its captured graph

Inputs are seeded and made on the GPU.  bf16 tensors of the framework are raw 16-bit patterns; they are handed out as
torch.bfloat16 views of the same memory.
"""
import ctypes as C
import math

import numpy as np
import torch

import autograph_amd as ag
from autograph_amd._ffi import check, lib

_TORCH = {"f32": torch.float32, "bf16": torch.bfloat16}
_SIZE = {"f32": 4, "bf16": 2}


def listed():
    return [
        # the headline product: a square bf16 product that fills the chip
        {"name": "dot_bf16_8192", "kind": "dot", "dtype": "bf16", "m": 8192, "k": 8192, "n": 8192, "ta": False, "tb": False},
        # an f32 weight-gradient product (transposed left operand)
        {"name": "dot_f32_4096_tn", "kind": "dot", "dtype": "f32", "m": 4096, "k": 4096, "n": 4096, "ta": True, "tb": False},
        # the large Dense layer in bf16, training or bulk inference
        {"name": "dense_bf16_16384x4096x4096", "kind": "dense", "dtype": "bf16", "m": 16384, "k": 4096, "n": 4096, "relu": True},
        # the same layer serving a handful of requests
        {"name": "dense_bf16_16x4096x4096", "kind": "dense", "dtype": "bf16", "m": 16, "k": 4096, "n": 4096, "relu": True},
        # a classifier head of ragged sizes: rows that are no multiple of a 16-byte vector
        {"name": "dense_bf16_1999x2047x1001", "kind": "dense", "dtype": "bf16", "m": 1999, "k": 2047, "n": 1001, "relu": False},
        # training of a mid-sized Dense layer
        {"name": "dense_backward_bf16_4096x2048x1000", "kind": "dense_backward", "dtype": "bf16", "m": 4096, "k": 2048, "n": 1000},
        # a convolution in the body of an image network
        {"name": "conv_bf16_256x64to128_56x56", "kind": "conv", "dtype": "bf16", "bs": 256, "ic": 64, "oc": 128, "h": 56, "w": 56,
         "f": 3, "s": 1, "p": 1, "bias": True, "relu": True},
        # the first convolution of one: three channels, a large filter, stride 2, odd rows
        {"name": "conv_f32_64x3to64_95x95_7x7s2", "kind": "conv", "dtype": "f32", "bs": 64, "ic": 3, "oc": 64, "h": 95, "w": 95,
         "f": 7, "s": 2, "p": 3, "bias": True, "relu": True},
        # training of a convolution in the body
        {"name": "conv_backward_f32_64x64to128_28x28", "kind": "conv_backward", "dtype": "f32", "bs": 64, "ic": 64, "oc": 128, "h": 28,
         "w": 28, "f": 3, "s": 1, "p": 1},
        # the pooling layer behind a large activation, both directions
        {"name": "pool_f32_256x64x56x56", "kind": "pool", "dtype": "f32", "bs": 256, "c": 64, "h": 56, "w": 56, "size": 2},
        # small-network inference at the batch size the benchmark uses
        {"name": "lenet_infer_f32_1000", "kind": "lenet_infer", "dtype": "f32", "bs": 1000, "path": "single"},
        # small-network training at the batch size the benchmark uses
        {"name": "lenet_train_bf16_100", "kind": "lenet_train", "dtype": "bf16", "bs": 100},
    ]


# ---- the ranges: sizes, types and options that the kinds above are used with ----

_KINDS = ("dot", "dense", "dense_backward", "conv", "conv_backward", "pool", "lenet_infer", "lenet_train")


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _log_size(rng, lo, hi):
    """Log-uniform; half of the sizes are whole multiples of 8, the others are left as they fall, odd ones among them."""
    v = _log_int(rng, lo, hi)
    return max(8, v // 8 * 8) if v >= 8 and rng.random() < 0.5 else v


def _draw_one(rng):
    kind = rng.choice(_KINDS)
    case = {"kind": kind, "dtype": rng.choice(("f32", "bf16"))}
    if kind == "dot":
        case.update(m=_log_size(rng, 16, 8192), k=_log_size(rng, 16, 8192), n=_log_size(rng, 16, 8192), ta=rng.random() < 0.5,
                    tb=rng.random() < 0.5)
    elif kind in ("dense", "dense_backward"):
        case.update(m=_log_size(rng, 1 if kind == "dense" else 16, 16384), k=_log_size(rng, 64, 8192), n=_log_size(rng, 10, 8192))
        if kind == "dense":
            case.update(relu=rng.random() < 0.5)
    elif kind in ("conv", "conv_backward"):
        f = rng.choice((1, 3, 3, 5, 7))
        h = _log_int(rng, max(8, 2 * f), 112)
        case.update(bs=_log_int(rng, 1, 256), ic=rng.choice((1, 3, 6, 16, 24, 32, 64, 128, 256)), oc=rng.choice((6, 16, 32, 48, 64, 96, 128, 256)),
                    h=h, w=rng.choice((h, _log_int(rng, max(8, 2 * f), 112))), f=f, s=rng.choice((1, 1, 2)), p=rng.choice((0, f // 2)))
        if kind == "conv":
            case.update(bias=rng.random() < 0.5, relu=rng.random() < 0.5)
    elif kind == "pool":
        h = _log_int(rng, 8, 112)
        case.update(bs=_log_int(rng, 1, 256), c=_log_int(rng, 1, 256), h=h, w=rng.choice((h, _log_int(rng, 8, 112))), size=rng.choice((2, 2, 3)))
    elif kind == "lenet_infer":
        case.update(bs=_log_int(rng, 1, 8192), path=rng.choice(("single", "layers")))
    else:
        case.update(bs=_log_int(rng, 8, 1024))
    return case


def _cost(case):
    """Seconds at everyday rates: the measure by which a drawn case is kept below the largest listed one."""
    w = work(case)
    return max(w["bytes"] / 4e12, w["flops"] / (1.2e14 if case["dtype"] == "f32" else 1.2e15))


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        case = _draw_one(rng)
        # a convolution's patch matrix, where a program has one, stays below 2 GB
        if case["kind"].startswith("conv") and _patch_elements(case) * _SIZE[case["dtype"]] > 2e9:
            continue
        if _cost(case) <= most:
            return case


# ---- helpers ----


class _Memory:
    """A framework tensor's memory as torch reads it; holds the tensor, so the memory lives as long as torch's view."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.__cuda_array_interface__ = {
            "shape": tensor.shape, "typestr": "<f4" if tensor.dtype == "f32" else "<i2",
            "strides": tuple(s * _SIZE[tensor.dtype] for s in tensor.strides), "data": (tensor._data_ptr(), False), "version": 2}


class _Loss(C.c_float * 1):
    """The loss of a training step, complete once the device is idle: one float in pinned host memory that the trainer frees, so
    the view holds the trainer."""


def _torch(tensor):
    view = torch.as_tensor(_Memory(tensor), device="cuda")
    return view if tensor.dtype == "f32" else view.view(torch.bfloat16)


def _tensor(values, dtype):
    """A framework tensor holding torch values (rounded to bf16 if asked for)."""
    values = values.to(_TORCH[dtype]).contiguous()
    out = ag.Tensor.uninit(tuple(values.shape), dtype)
    torch.cuda.synchronize()
    check(lib.agh_memcpy_d2d(out._ptr(), values.data_ptr(), values.numel() * _SIZE[dtype]))
    check(lib.agh_sync())
    return out


class _Random:
    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def normal(self, shape, std, dtype):
        return _tensor(torch.randn(shape, generator=self.gen, device="cuda") * std, dtype)

    def uniform(self, shape, lo, hi, dtype):
        return _tensor(torch.rand(shape, generator=self.gen, device="cuda") * (hi - lo) + lo, dtype)

    def activation(self, shape, dtype):
        """What a layer behind a relu sees: normal values, the negative half zero."""
        return _tensor(torch.randn(shape, generator=self.gen, device="cuda").clamp_(min=0), dtype)


def _out_hw(case):
    return ((case["h"] + 2 * case["p"] - case["f"]) // case["s"] + 1, (case["w"] + 2 * case["p"] - case["f"]) // case["s"] + 1)


def _patch_elements(case):
    oh, ow = _out_hw(case)
    return case["bs"] * oh * ow * case["ic"] * case["f"] ** 2


_LENET = (((6, 1, 5, 5), 25), ((16, 6, 5, 5), 150), ((256, 128), 256), ((128, 84), 128), ((84, 10), 84), ((10,), 84))
_LENET_PARAMS = sum(math.prod(s) for s, _ in _LENET)
_LENET_FLOPS = 2 * (576 * 6 * 25 + 64 * 16 * 150 + 256 * 128 + 128 * 84 + 84 * 10)  # forward, one image


# ---- what a program has in hand before the call ----


def prepare(case, seed):
    ag.Device(0)
    r, dt, kind = _Random(seed), case["dtype"], case["kind"]
    st = {"case": case}
    if kind == "dot":
        m, k, n = case["m"], case["k"], case["n"]
        make = (lambda s: r.uniform(s, -1, 1, dt)) if dt == "f32" else (lambda s: r.normal(s, 0.02, dt))
        a, b = make((k, m) if case["ta"] else (m, k)), make((n, k) if case["tb"] else (k, n))
        st.update(a=a.t() if case["ta"] else a, b=b.t() if case["tb"] else b, c=ag.Tensor.uninit((m, n), dt))
        st["out"] = _torch(st["c"])
    elif kind == "dense":
        k = case["k"]
        st.update(x=r.activation((case["m"], k), dt),
                  layer=ag.Dense(r.normal((k, case["n"]), math.sqrt(2 / k), dt), r.normal((case["n"],), 0.1, dt)))
    elif kind == "dense_backward":
        m, k, n = case["m"], case["k"], case["n"]
        st.update(x=r.activation((m, k), dt), w=r.normal((k, n), math.sqrt(2 / k), dt), dy=r.normal((m, n), 1 / m, dt))
    elif kind in ("conv", "conv_backward"):
        bs, ic, oc, f = case["bs"], case["ic"], case["oc"], case["f"]
        st["x"] = r.activation((bs, ic, case["h"], case["w"]), dt)
        w = r.normal((oc, ic, f, f), math.sqrt(2 / (ic * f * f)), dt)
        if kind == "conv":
            bias = r.normal((oc,), 0.1, dt) if case["bias"] else None
            st["layer"] = ag.Conv2(w, bias, (case["p"],) * 2, (case["s"],) * 2)
        else:
            oh, ow = _out_hw(case)
            opts = {"filter": (f, f), "padding": (case["p"],) * 2, "stride": (case["s"],) * 2}
            st.update(w=w, dy=r.normal((bs, oc, oh, ow), 1 / bs, dt), im2col=ag.Im2ColConv2Options(**opts),
                      col2im=ag.Col2ImConv2Options(shape=(oh, ow), **opts))
    elif kind == "pool":
        size, h, w = case["size"], case["h"], case["w"]
        st.update(x=r.normal((case["bs"], case["c"], h, w), 1, dt), layer=ag.MaxPool2((size, size)), opts=ag.MaxPool2Options((size,) * 2, (size,) * 2),
                  dy=r.normal((case["bs"], case["c"], (h - size) // size + 1, (w - size) // size + 1), 0.1, dt))
    else:
        bs = case["bs"]
        params = [r.uniform(s, -math.sqrt(2 / fan), math.sqrt(2 / fan), dt) for s, fan in _LENET]
        model = ag.LeNet5(*params)
        x = r.uniform((bs, 1, 28, 28), 0, 1, dt)
        st.update(model=model, x=x)
        if kind == "lenet_infer":
            st["out"] = torch.empty((bs, 10), dtype=_TORCH[dt], device="cuda")
        else:
            labels = torch.randint(0, 10, (bs,), generator=r.gen, device="cuda").to(torch.uint8)
            target = ag.Buffer(bs)
            torch.cuda.synchronize()
            check(lib.agh_memcpy_d2d(target.ptr, labels.data_ptr(), bs))
            check(lib.agh_sync())
            trainer = ag.LeNet5Trainer(model, bs, learning_rate=0.01, optimizer=ag.SGD(0.01))
            trainer.capture(x, target)
            check(lib.agh_sync())
            st.update(trainer=trainer, target=target)
            loss = _Loss.from_address(trainer._loss_host.value)
            loss.owner = trainer
            st["out"] = [_torch(t) for t in trainer.params + trainer.grads + trainer.velocities]
            st["out"].append(torch.from_numpy(np.frombuffer(loss, np.float32)))
    return st


# ---- one pass ----


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "dot":
        ag.gemm(1.0, st["a"], st["b"], 0.0, st["c"])
        return st["out"]
    if kind == "dense":
        return _torch(st["layer"].forward(st["x"], relu=case["relu"]))
    if kind == "dense_backward":
        dy = st["dy"]
        return [_torch(t) for t in (dy.dot(st["w"].t()), st["x"].t().dot(dy), dy.sum_axis0())]
    if kind == "conv":
        return _torch(st["layer"].forward(st["x"], relu=case["relu"]))
    if kind == "conv_backward":
        dy, w = st["dy"], st["w"]
        bs, oc, oh, ow = dy.shape
        gm = dy.permuted_axes((0, 2, 3, 1)).as_standard_layout().into_shape((bs * oh * ow, oc))
        dw = gm.t().dot(st["x"].im2col_conv2(st["im2col"]))
        dx = gm.dot(w.into_shape((oc, dw.shape[1]))).col2im_conv2(st["col2im"])
        return [_torch(dw), _torch(dx)]
    if kind == "pool":
        x = st["x"]
        y, dx = st["layer"].forward(x), x.clone()
        dx.max_pool2_backward(st["dy"], st["opts"])
        return [_torch(y), _torch(dx)]
    if kind == "lenet_infer":
        if case["path"] == "layers":
            return _torch(st["model"].forward_fused(st["x"]))
        st["model"].forward_single_launch(st["x"], st["out"].data_ptr())
        return st["out"]
    st["trainer"].replay()
    return st["out"]


# ---- the work a pass cannot do without ----


def work(case):
    es, kind = _SIZE[case["dtype"]], case["kind"]
    if kind in ("dot", "dense", "dense_backward"):
        m, k, n = case["m"], case["k"], case["n"]
        if kind == "dense_backward":  # x, w, dy in; dx, dW, db out
            return {"bytes": es * (2 * m * k + 2 * k * n + m * n + n), "flops": 4.0 * m * k * n + m * n}
        return {"bytes": es * (m * k + k * n + m * n + (n if kind == "dense" else 0)), "flops": 2.0 * m * k * n}
    if kind in ("conv", "conv_backward"):
        oh, ow = _out_hw(case)
        x, y = case["bs"] * case["ic"] * case["h"] * case["w"], case["bs"] * case["oc"] * oh * ow
        w = case["oc"] * case["ic"] * case["f"] ** 2
        flops = 2.0 * case["oc"] * _patch_elements(case)
        if kind == "conv":
            return {"bytes": es * (x + y + w + (case["oc"] if case["bias"] else 0)), "flops": flops}
        return {"bytes": es * (2 * x + y + 2 * w), "flops": 2 * flops}
    if kind == "pool":  # x, dy in; y, dx out
        size = case["size"]
        x, y = case["h"] * case["w"], ((case["h"] - size) // size + 1) * ((case["w"] - size) // size + 1)
        return {"bytes": es * case["bs"] * case["c"] * (2 * x + 2 * y), "flops": float(case["bs"] * case["c"] * x)}
    bs = case["bs"]
    if kind == "lenet_infer":
        return {"bytes": es * (bs * 794 + _LENET_PARAMS), "flops": float(_LENET_FLOPS * bs)}
    # images, labels; parameters and velocities read and written, gradients written
    return {"bytes": es * (bs * 784 + 5 * _LENET_PARAMS) + bs, "flops": float((3 * _LENET_FLOPS - 2 * 576 * 6 * 25) * bs)}


def tolerance(case):
    """About four times what the path differs by from itself in 64 bits (2-norm): 1.2e-6 in f32 at k = 4096; 2.4e-3 in bf16 with
    a bias (two roundings); 4.1e-3 where col2im adds in bf16.  LeNet5: fused against layer by layer, where a relu mask may
    flip: 2e-3 in bf16."""
    if case["kind"] == "pool":
        return "exact"  # copies of input values
    if case["dtype"] == "f32":
        return {"rel": 1e-5 if case["kind"] == "lenet_train" else 5e-6}
    return {"rel": 1.6e-2 if case["kind"] == "conv_backward" else 1e-2}
