"""Python face of the op, mirroring the wrapper TensorFlow generates for the reference's
REGISTER_OP("ApproxConv2DWithMinMaxVars") (tf2/src/approx_nn_ops.cpp:38-54): same argument names,
order and meaning as the call in tf2/test/test_table_approx_conv_2d.py:47-49.

Tensors are torch tensors on a ROCm device (torch is only the owner of device memory and of the
stream); all arithmetic happens in libaxconv_hip.so.
"""
import ctypes
import weakref

import numpy as np

import torch

from . import _lib


class InvalidArgumentError(ValueError):
    """tensorflow::errors::InvalidArgument in the reference."""


class UnimplementedError(NotImplementedError):
    """tensorflow::errors::Unimplemented in the reference."""


def _check(rc):
    if rc == _lib.OK:
        return
    msg = _lib.load().axc_last_error().decode()
    if rc == _lib.INVALID_ARGUMENT:
        raise InvalidArgumentError(msg)
    if rc == _lib.UNIMPLEMENTED:
        raise UnimplementedError(msg)
    raise RuntimeError(msg)


_PADDING = {"VALID": _lib.PAD_VALID, "SAME": _lib.PAD_SAME, "EXPLICIT": _lib.PAD_EXPLICIT}
_FORMAT = {"NHWC": _lib.FORMAT_NHWC, "NCHW": _lib.FORMAT_NCHW}


def make_desc(input_shape, filter_shape, strides, padding, explicit_paddings=(), data_format="NHWC",
              dilations=(1, 1, 1, 1), num_bits=8):
    if len(input_shape) != 4:
        raise InvalidArgumentError("input must be 4-dimensional")
    if len(filter_shape) != 4:
        raise InvalidArgumentError("filter must be 4-dimensional")
    if len(strides) != 4:
        raise InvalidArgumentError("Sliding window strides must specify 4 dimensions")
    if len(dilations) != 4:
        raise InvalidArgumentError("Sliding window dilations field must specify 4 dimensions")
    if isinstance(padding, bytes):
        padding = padding.decode()
    if padding not in _PADDING:
        raise InvalidArgumentError("Invalid padding")
    if data_format not in _FORMAT:
        raise InvalidArgumentError("Invalid data format")
    d = _lib.ConvDesc()
    for i in range(4):
        d.input_shape[i] = int(input_shape[i])
        d.filter_shape[i] = int(filter_shape[i])
        d.strides[i] = int(strides[i])
        d.dilations[i] = int(dilations[i])
    d.padding = _PADDING[padding]
    d.data_format = _FORMAT[data_format]
    d.num_bits = int(num_bits)
    ep = list(explicit_paddings) + [0] * 8
    for i in range(8):
        d.explicit_paddings[i] = int(ep[i])
    return d


def conv2d_geometry(desc):
    dims = _lib.ConvDims()
    _check(_lib.load().axc_conv2d_geometry(ctypes.byref(desc), ctypes.byref(dims)))
    return dims


def quant_props(input_min, input_max, filter_min, filter_max):
    qp = _lib.QuantProps()
    _check(_lib.load().axc_quant_props_compute(float(input_min), float(input_max), float(filter_min),
                                               float(filter_max), ctypes.byref(qp)))
    return qp


class TruthTable:
    """Device-resident 256x256 uint16 truth table (the op's `mul_map_file` attr, loaded once)."""

    def __init__(self, source="", num_bits=8):
        lib = _lib.load()
        handle = ctypes.c_void_p()
        if isinstance(source, (str, bytes)):
            name = source.encode() if isinstance(source, str) else source
            _check(lib.axc_table_create_from_file(name, int(num_bits), ctypes.byref(handle)))
        else:
            import numpy as np
            if int(num_bits) != 8:
                raise InvalidArgumentError("only num_bits = 8 is supported")
            host = np.ascontiguousarray(source, dtype=np.uint16).reshape(-1)
            if host.size != 65536:
                raise InvalidArgumentError("truth table must hold 65536 uint16 entries")
            _check(lib.axc_table_create(host.ctypes.data, ctypes.byref(handle)))
        self.handle = handle

    def __del__(self):
        try:
            if getattr(self, "handle", None):
                _lib.load().axc_table_destroy(self.handle)
                self.handle = None
        except Exception:
            pass


_workspaces = {}


def _workspace(device, stream, nbytes):
    """Scratch memory of a call, cached per (device, current stream): calls issued on one stream run in order and
    may share it; calls on different streams may overlap and must not."""
    key = (device, stream)
    buf = _workspaces.get(key)
    if buf is None or buf.numel() < nbytes:
        buf = torch.empty(max(int(nbytes), 256), dtype=torch.uint8, device=device)
        _workspaces[key] = buf
    return buf


def _scalar(v):
    if type(v) is float:
        return v
    if torch.is_tensor(v):
        return float(v.item())
    return float(v)


# The current stream's handle; the public way makes a Stream object of it first, which takes 2 us.
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def _stream(device):
    return _raw_stream(device.index) if _raw_stream else torch.cuda.current_stream(device).cuda_stream


def _launch(device, fn, *args):
    """fn(*args) with `device` current: entering a device's context takes longer than all else here."""
    if torch.cuda.current_device() == device.index:
        rc = fn(*args)
    else:
        with torch.cuda.device(device):
            rc = fn(*args)
    if rc != _lib.OK:
        _check(rc)


class _Layer:
    """What a call needs to know of its shapes and attributes: made once for each, never changed."""

    def __init__(self, desc, depthwise):
        dims = conv2d_geometry(desc)
        self.desc = desc
        self.ref = ctypes.byref(desc)
        self.columns = dims.in_depth if depthwise else dims.out_depth
        self.out_shape = (dims.batch, int(dims.out_rows), int(dims.out_cols), self.columns)
        self.depthwise = depthwise

    def workspace(self, lib, device, stream):
        """Asked for on every call: what it has to hold depends on the forms that are pinned."""
        nbytes = ctypes.c_size_t()
        fn = lib.axc_depthwise_conv2d_workspace_bytes if self.depthwise else lib.axc_conv2d_workspace_bytes
        _check(fn(self.ref, ctypes.byref(nbytes)))
        return _workspace(device, stream, nbytes.value)


def _require_device_f32(t, what):
    if not torch.is_tensor(t) or not t.is_cuda:
        raise InvalidArgumentError("%s must be a tensor on the GPU" % what)
    if t.dtype != torch.float32:
        raise UnimplementedError("%s: only float32 is registered for this op" % what)
    return t.contiguous()


class ApproxConv2DWithMinMaxVars:
    """One op instance: attrs fixed at construction, like the reference's OpKernel
    (ApproxConv2DOp, tf2/src/approx_nn_conv_ops.cpp:411-468)."""

    def __init__(self, strides, num_bits, mul_map_file, padding, explicit_paddings=(), data_format="NHWC",
                 dilations=(1, 1, 1, 1), depthwise=False):
        self.strides = list(strides)
        self.num_bits = int(num_bits)
        self.padding = padding
        self.explicit_paddings = list(explicit_paddings)
        self.data_format = data_format
        self.dilations = list(dilations)
        self.depthwise = depthwise
        self.table = mul_map_file if isinstance(mul_map_file, TruthTable) else TruthTable(mul_map_file, num_bits)
        self._layers = {}
        # attr checks the reference performs at construction (InitApproxConv2DParameters)
        make_desc((1, 1, 1, 1), (1, 1, 1, 1), self.strides, self.padding, self.explicit_paddings,
                  self.data_format, self.dilations, self.num_bits)

    def _desc(self, input, filter):
        return make_desc(tuple(input.shape), tuple(filter.shape), self.strides, self.padding,
                         self.explicit_paddings, self.data_format, self.dilations, self.num_bits)

    def _out_shape(self, dims):
        depth = dims.in_depth if self.depthwise else dims.out_depth
        return (dims.batch, int(dims.out_rows), int(dims.out_cols), depth)

    def _layer(self, input, filter):
        key = (input.shape, filter.shape, tuple(self.strides), self.num_bits, self.padding, tuple(self.explicit_paddings),
               self.data_format, tuple(self.dilations), self.depthwise)
        layer = self._layers.get(key)
        if layer is None:
            layer = _Layer(self._desc(input, filter), self.depthwise)
            if len(self._layers) >= 256:
                self._layers.clear()
            self._layers[key] = layer
        return layer

    def _run(self, input, filter, mins, acc_i32):
        lib = _lib.load()
        input = _require_device_f32(input, "input")
        filter = _require_device_f32(filter, "filter")
        layer, device = self._layer(input, filter), input.device
        stream = _stream(device)
        ws = layer.workspace(lib, device, stream)
        out = torch.empty(layer.out_shape, dtype=torch.int32 if acc_i32 else torch.float32, device=device)
        if self.depthwise:
            fn = lib.axc_depthwise_conv2d_minmax_acc_i32 if acc_i32 else lib.axc_depthwise_conv2d_minmax
        else:
            fn = lib.axc_conv2d_minmax_acc_i32 if acc_i32 else lib.axc_conv2d_minmax
        _launch(device, fn, self.table.handle, layer.ref, input.data_ptr(), filter.data_ptr(), *[_scalar(m) for m in mins],
                out.data_ptr(), ws.data_ptr(), ws.numel(), stream)
        return out

    def __call__(self, input, filter, input_min, input_max, filter_min, filter_max, bias=None, activation=None):
        """The op.  With `bias` and / or `activation` ("relu"): the op followed by bias_add and the activation, fused
        into its store (the tail of the Keras layer's call, fake_approx_convolutional.py:261)."""
        if bias is None and activation is None:
            return self._run(input, filter, (input_min, input_max, filter_min, filter_max), False)
        if activation not in (None, "relu"):
            raise InvalidArgumentError("activation must be None or 'relu'")
        lib = _lib.load()
        input = _require_device_f32(input, "input")
        filter = _require_device_f32(filter, "filter")
        layer, device = self._layer(input, filter), input.device
        if bias is not None:
            bias = _require_device_f32(bias, "bias")
            if bias.numel() != layer.columns:
                raise InvalidArgumentError("bias must have one value per output channel")
        stream = _stream(device)
        ws = layer.workspace(lib, device, stream)
        out = torch.empty(layer.out_shape, dtype=torch.float32, device=device)
        _launch(device, lib.axc_depthwise_conv2d_minmax_bias_act if self.depthwise else lib.axc_conv2d_minmax_bias_act,
                self.table.handle, layer.ref, input.data_ptr(), filter.data_ptr(),
                _scalar(input_min), _scalar(input_max), _scalar(filter_min), _scalar(filter_max),
                bias.data_ptr() if bias is not None else None, 1 if activation == "relu" else 0,
                out.data_ptr(), ws.data_ptr(), ws.numel(), stream)
        return out

    def output_shape(self, input, filter):
        return self._layer(input, filter).out_shape

    def call_and_add(self, input, filter, input_min, input_max, filter_min, filter_max, addend, activation=None):
        """The op, a tensor like its output added to it, and the activation behind that: as a residual network's sum, which
        needs no pass of its own then.  The activation keeps NaN, as the networks' elementwise pass does."""
        if activation not in (None, "relu"):
            raise InvalidArgumentError("activation must be None or 'relu'")
        if self.depthwise:
            raise UnimplementedError("call_and_add: dense layers only")
        lib = _lib.load()
        input = _require_device_f32(input, "input")
        filter = _require_device_f32(filter, "filter")
        addend = _require_device_f32(addend, "addend")
        layer, device = self._layer(input, filter), input.device
        if tuple(addend.shape) != layer.out_shape:
            raise InvalidArgumentError("addend must have the output's shape %s" % (layer.out_shape,))
        stream = _stream(device)
        ws = layer.workspace(lib, device, stream)
        out = torch.empty(layer.out_shape, dtype=torch.float32, device=device)
        _launch(device, lib.axc_conv2d_minmax_bias_add_act, self.table.handle, layer.ref, input.data_ptr(), filter.data_ptr(),
                _scalar(input_min), _scalar(input_max), _scalar(filter_min), _scalar(filter_max), None, addend.data_ptr(),
                1 if activation == "relu" else 0, out.data_ptr(), ws.data_ptr(), ws.numel(), stream)
        return out

    def accumulators(self, input, filter, input_min, input_max, filter_min, filter_max):
        """int32 sums of table entries before the epilogue (parity entry point)."""
        return self._run(input, filter, (input_min, input_max, filter_min, filter_max), True)


def _version(t):
    """How often torch has seen the tensor's memory written to; None where it does not count."""
    return None if t.is_inference() else t._version


class FakeApproxConv2D:
    """The reference's Keras layer around the op (FakeApproxConv2D.call,
    tf2/python/keras/layers/fake_approx_convolutional.py:223-261) as one device-side call: min/max of the batch
    and of the kernel, fake quantization of both, the op, bias_add, activation.  No host synchronisation."""

    def __init__(self, strides, mul_map_file, padding="SAME", dilation_rate=(1, 1), activation=None, num_bits=8,
                 depthwise=False):
        """depthwise: the layer wraps the depthwise variant (kernel [rows, cols, C, 1], bias one value per channel)."""
        if activation not in (None, "relu"):
            raise UnimplementedError("activation %r: only None and 'relu' are fused" % (activation,))
        self.op = ApproxConv2DWithMinMaxVars([1, strides[0], strides[1], 1], num_bits, mul_map_file, padding.upper(),
                                             dilations=[1, dilation_rate[0], dilation_rate[1], 1], depthwise=depthwise)
        self.depthwise = depthwise
        self.activation = 1 if activation == "relu" else 0

    def __call__(self, inputs, kernel, bias=None):
        return self._run(inputs, kernel, bias, None, False)[0]

    def call_in_turn(self, inputs, kernel, bias=None, input_range=None, want_range=True):
        """The call, for a program that makes one layer's output the next one's input: (output, range).  `range` is what
        the call saw of its outputs' smallest and largest value, for the input_range of a call on that very output, which
        then need not read the tensor to find them; None where the kernel that ran does not report it.

        With any other input, or one that torch knows to have been written to since, the call finds the range itself; so it
        does for outputs made under torch.inference_mode(), whose changes torch does not count.  Writes that torch does not
        see (through data_ptr() or .data) are the caller's to mind."""
        if input_range is not None:
            inputs = _require_device_f32(inputs, "input")
            if not torch.is_tensor(input_range) or input_range.device != inputs.device:
                raise InvalidArgumentError("input_range must be a tensor on the input's GPU")
            if (input_range.dtype != torch.float32 or not input_range.is_contiguous() or
                    input_range.numel() * 4 < _lib.RANGE_BYTES):
                raise InvalidArgumentError("input_range must be what call_in_turn returned")
            of, version = getattr(input_range, "_range_of", (None, None))
            if version is None or of() is not inputs or _version(inputs) != version:
                input_range = None
        out, seen = self._run(inputs, kernel, bias, input_range, want_range)
        if seen is not None:
            seen._range_of = weakref.ref(out), _version(out)
        return out, seen

    def _run(self, inputs, kernel, bias, input_range, want_range):
        """call_in_turn for a caller that knows input_range to be that of `inputs` as they are."""
        lib = _lib.load()
        inputs = _require_device_f32(inputs, "input")
        kernel = _require_device_f32(kernel, "filter")
        if bias is not None:
            bias = _require_device_f32(bias, "bias")
            if bias.numel() != (kernel.shape[2] if self.depthwise else kernel.shape[3]):
                raise InvalidArgumentError("bias must have one value per output channel")
        layer, device = self.op._layer(inputs, kernel), inputs.device
        stream = _stream(device)
        ws = layer.workspace(lib, device, stream)
        out = torch.empty(layer.out_shape, dtype=torch.float32, device=device)
        args = (self.op.table.handle, layer.ref, inputs.data_ptr(), kernel.data_ptr(),
                bias.data_ptr() if bias is not None else None, self.activation, out.data_ptr())
        if input_range is None and not want_range:
            _launch(device, lib.axc_fake_approx_depthwise_conv2d if self.depthwise else lib.axc_fake_approx_conv2d,
                    *args, ws.data_ptr(), ws.numel(), stream)
            return out, None
        seen = torch.empty(_lib.RANGE_BYTES // 4, dtype=torch.float32, device=device) if want_range else None
        ranges = _lib.LayerRanges(None if input_range is None else input_range.data_ptr(),
                                  None if seen is None else seen.data_ptr(), 0)
        _launch(device, lib.axc_fake_approx_depthwise_conv2d_ranged if self.depthwise else lib.axc_fake_approx_conv2d_ranged,
                *args, ctypes.byref(ranges), ws.data_ptr(), ws.numel(), stream)
        return out, seen if ranges.output_written else None


# ---- tf1 AxConv2D (tf1/axqconv/axqconv.cc) ----------------------------------------------------------------------
def float_to_quantized_unclamped_quint8(value, range_min, range_max):
    """FloatToQuantizedUnclamped<quint8> for the value 0.0f (tf1/axqconv/quantization_utils.h:49-64): the zero
    point the reference derives per tensor (tf1/axqconv/axqconv.cc:364-367).  Computed by the library."""
    if float(value) != 0.0:
        raise UnimplementedError("only the code of 0.0f is needed by AxConv2D")
    zp = ctypes.c_int32()
    _check(_lib.load().axc_quint8_zero_point(float(range_min), float(range_max), ctypes.byref(zp)))
    return zp.value


def quantization_range_for_multiplication(min_a, max_a, min_b, max_b):
    """QuantizationRangeForMultiplication<quint8, quint8, qint32> (tf1/axqconv/quantization_utils.h:114-140): the
    float range the qint32 output of AxConv2D stands for (tf1/axqconv/axqconv.cc:427-431)."""
    lo, hi = ctypes.c_float(), ctypes.c_float()
    _check(_lib.load().axc_qint32_range_for_multiplication(float(min_a), float(max_a), float(min_b), float(max_b),
                                                           ctypes.byref(lo), ctypes.byref(hi)))
    return lo.value, hi.value


def tune_table(table):
    """AxTune of the tf1 op (tf1/axqconv/approximate_selector.h:52-85) applied to a uint16[65536] table."""
    lib = _lib.load()
    src = np.ascontiguousarray(table, np.uint16).reshape(-1)
    if src.size != 65536:
        raise InvalidArgumentError("table must hold 65536 entries")
    out = np.zeros(65536, np.uint16)
    _check(lib.axc_table_tune_weights(src.ctypes.data, out.ctypes.data))
    return out


def ax_conv2d(input, filter, min_input, max_input, min_filter, max_filter, strides, padding, table):
    """The tf1 op AxConv2D (registration tf1/axqconv/axqconv.cc:66-94): quint8 codes in (uint8 tensors on the GPU),
    (qint32 output, min_output, max_output) out.  `table` is a TruthTable (AxMult / AxTune already applied)."""
    lib = _lib.load()
    if input.dtype != torch.uint8 or filter.dtype != torch.uint8:
        raise UnimplementedError("AxConv2D: only quint8 input and filter are registered")
    if not input.is_cuda or not filter.is_cuda:
        raise InvalidArgumentError("input and filter must be tensors on the GPU")
    input, filter = input.contiguous(), filter.contiguous()
    layer = _Layer(make_desc(tuple(input.shape), tuple(filter.shape), list(strides), padding, (), "NHWC", (1, 1, 1, 1), 8), False)
    device = input.device
    stream = _stream(device)
    ws = layer.workspace(lib, device, stream)
    out = torch.empty(layer.out_shape, dtype=torch.int32, device=device)
    off_in = float_to_quantized_unclamped_quint8(0.0, min_input, max_input)
    off_f = float_to_quantized_unclamped_quint8(0.0, min_filter, max_filter)
    _launch(device, lib.axc_axconv2d_quint8, table.handle, layer.ref, input.data_ptr(), filter.data_ptr(), off_in, off_f,
            out.data_ptr(), ws.data_ptr(), ws.numel(), stream)
    lo, hi = quantization_range_for_multiplication(min_input, max_input, min_filter, max_filter)
    return out, lo, hi


def conv2d_tile_plan(input_shape, filter_shape, strides=(1, 1, 1, 1), padding="SAME", dilations=(1, 1, 1, 1)):
    """The dense kernel's tile plan for a layer on the current device, as a dict."""
    lib = _lib.load()
    desc = make_desc(tuple(input_shape), tuple(filter_shape), list(strides), padding, (), "NHWC", list(dilations), 8)
    plan = (ctypes.c_int32 * 8)()
    _check(lib.axc_conv2d_tile_plan(ctypes.byref(desc), plan))
    # preexpanded_rows: 0 = rows expanded inside every tile, 1 = pre-expanded rows, 2 = pre-expanded rows read by the
    # kernel without a barrier between fills
    keys = ("columns_per_tile", "rows_per_tile", "row_tiles", "column_tiles", "k_splits", "workgroups",
            "fills_per_split", "preexpanded_rows")
    return dict(zip(keys, [int(v) for v in plan]))


def conv2d_matrix_plan(input_shape, filter_shape, strides=(1, 1, 1, 1), padding="SAME", dilations=(1, 1, 1, 1)):
    """How the kernel whose sums the matrix cores make cuts a layer on the current device, as a dict; None for a layer
    that does not run it.  (Layers that conv2d_direct_plan names run that way instead.)"""
    lib = _lib.load()
    desc = make_desc(tuple(input_shape), tuple(filter_shape), list(strides), padding, (), "NHWC", list(dilations), 8)
    plan = (ctypes.c_int32 * 8)()
    _check(lib.axc_conv2d_matrix_plan(ctypes.byref(desc), plan))
    rows = ctypes.c_int32()
    _check(lib.axc_conv2d_matrix_rows(ctypes.byref(desc), ctypes.byref(rows)))
    if not plan[0]:
        return None
    # own_rows: 0 = reads pre-expanded rows, 1 = makes them itself in every tile, 2 = the same with the operands exchanged
    keys = ("units_per_wavefront", "units_per_tile", "row_tiles", "column_tiles", "k_splits", "workgroups",
            "fills_per_split")
    return dict(zip(keys, [int(v) for v in plan[1:]]), own_rows=rows.value - 1)


def conv2d_direct_plan(input_shape, filter_shape, strides=(1, 1, 1, 1), padding="SAME", dilations=(1, 1, 1, 1), layer=False):
    """How a layer that runs as one launch on the current device is cut, as a dict; None for one that does not.  layer: as
    the layer call runs it, not the op."""
    lib = _lib.load()
    desc = make_desc(tuple(input_shape), tuple(filter_shape), list(strides), padding, (), "NHWC", list(dilations), 8)
    plan = (ctypes.c_int32 * 8)()
    _check(lib.axc_conv2d_direct_plan(ctypes.byref(desc), int(layer), plan))
    if not plan[0]:
        return None
    keys = ("pixels_per_tile", "columns_per_tile", "elements_per_chunk", "chunks", "row_tiles", "column_tiles", "workgroups")
    return dict(zip(keys, [int(v) for v in plan[1:]]))


def set_tile_columns(columns):
    """Pins the dense kernel's tile width (16 / 32 / 64 columns; 0 = the planner's choice) for the whole process."""
    _check(_lib.load().axc_set_tile_columns(int(columns)))


def set_preexpand(mode):
    """Which dense layers run out of pre-expanded rows: 0 = the planner's choice, 1 = all that can, -1 = none."""
    _check(_lib.load().axc_set_preexpand(int(mode)))


def set_matrix_rows(mode):
    """Rows of the kernel whose sums the matrix cores make: 0 = the planner's choice, 1 = pre-expanded ones only, 2 = made
    by the kernel itself wherever it can, 3 = the same with the operands exchanged, 4 = whole layers in one launch wherever
    possible."""
    _check(_lib.load().axc_set_matrix_rows(int(mode)))


def set_merged_launches(mode):
    """Launches that do the work of several (layers that conv2d_direct_plan names; what precedes the lookups of layers given as
    codes): 0 = where the planner says so, except while the timers run, 1 = while they run too, -1 = never."""
    _check(_lib.load().axc_set_merged_launches(int(mode)))


def set_wait_limit(polls):
    """Polls a wavefront of the barrier-free LUT-GEMM kernel makes in one wait before it gives up (tests of the
    report; the default is 2**20)."""
    _check(_lib.load().axc_set_wait_limit(int(polls)))


_table_cache = {}


def _cached_table(mul_map_file, num_bits):
    if isinstance(mul_map_file, TruthTable):
        return mul_map_file
    if not isinstance(mul_map_file, (str, bytes)):
        return TruthTable(mul_map_file, num_bits)
    key = (mul_map_file, int(num_bits))
    if key not in _table_cache:
        _table_cache[key] = TruthTable(mul_map_file, num_bits)
    return _table_cache[key]


def approx_conv2d_with_min_max_vars(input, filter, input_min, input_max, filter_min, filter_max, strides,
                                    num_bits, mul_map_file, padding, explicit_paddings=(), data_format="NHWC",
                                    dilations=(1, 1, 1, 1), name=None):
    """Drop-in for the generated wrapper of the reference op (argument order of
    tf2/test/test_table_approx_conv_2d.py:47-49).  mul_map_file may also be a TruthTable or a
    uint16[65536] array, so seeded synthetic tables need no file."""
    op = ApproxConv2DWithMinMaxVars(strides, num_bits, _cached_table(mul_map_file, num_bits), padding,
                                    explicit_paddings, data_format, dilations)
    return op(input, filter, input_min, input_max, filter_min, filter_max)


def approx_depthwise_conv2d_with_min_max_vars(input, filter, input_min, input_max, filter_min, filter_max,
                                              strides, num_bits, mul_map_file, padding, explicit_paddings=(),
                                              data_format="NHWC", dilations=(1, 1, 1, 1), name=None):
    """Depthwise variant (filter [rows, cols, C, 1]); the reference has no such op."""
    op = ApproxConv2DWithMinMaxVars(strides, num_bits, _cached_table(mul_map_file, num_bits), padding,
                                    explicit_paddings, data_format, dilations, depthwise=True)
    return op(input, filter, input_min, input_max, filter_min, filter_max)


def quantize(values, vmin, vmax):
    """uint8 codes of a float32 device tensor (parity entry point for the quantize expression)."""
    values = _require_device_f32(values, "values")
    codes = torch.empty(values.shape, dtype=torch.uint8, device=values.device)
    with torch.cuda.device(values.device):
        _check(_lib.load().axc_quantize(values.data_ptr(), values.numel(), float(vmin), float(vmax),
                                        codes.data_ptr(), _stream(values.device)))
    return codes


def conv2d_codes_acc_i32(table, input_codes, filter_codes, input_zero_code, strides=(1, 1, 1, 1),
                         padding="SAME", dilations=(1, 1, 1, 1)):
    """int32 LUT-GEMM sums on caller-supplied uint8 codes (NHWC / HWIO device tensors)."""
    lib = _lib.load()
    if input_codes.dtype != torch.uint8 or filter_codes.dtype != torch.uint8:
        raise InvalidArgumentError("codes must be uint8")
    input_codes = input_codes.contiguous()
    filter_codes = filter_codes.contiguous()
    layer = _Layer(make_desc(tuple(input_codes.shape), tuple(filter_codes.shape), strides, padding, (), "NHWC", dilations), False)
    device = input_codes.device
    stream = _stream(device)
    ws = layer.workspace(lib, device, stream)
    out = torch.empty(layer.out_shape, dtype=torch.int32, device=device)
    _launch(device, lib.axc_conv2d_codes_acc_i32, table.handle, layer.ref, input_codes.data_ptr(), filter_codes.data_ptr(),
            int(input_zero_code), out.data_ptr(), ws.data_ptr(), ws.numel(), stream)
    return out


# ---- measurement helpers ---------------------------------------------------------------------

def profile_enable(on=True):
    _check(_lib.load().axc_profile_enable(1 if on else 0))


def profile_reset():
    _check(_lib.load().axc_profile_reset())


def profile_read():
    """{kernel name: (total_ms, launches)} since the last reset."""
    lib = _lib.load()
    out = {}
    i = 0
    while True:
        name = ctypes.create_string_buffer(64)
        ms = ctypes.c_double()
        n = ctypes.c_int64()
        if lib.axc_profile_read(i, name, 64, ctypes.byref(ms), ctypes.byref(n)) != _lib.OK:
            break
        out[name.value.decode()] = (ms.value, n.value)
        i += 1
    return out


def lds_gather_peak():
    v = ctypes.c_double()
    _check(_lib.load().axc_lds_gather_peak(ctypes.byref(v), None))
    return v.value


def lds_read_peak():
    """Streaming ds_read_b128 rate in bytes/s over all CUs (measured)."""
    v = ctypes.c_double()
    _check(_lib.load().axc_lds_read_peak(ctypes.byref(v), None))
    return v.value


def valu_issue_peak():
    """Issue rate of the LUT-GEMM's accumulate instruction mix in lane operations per second (measured)."""
    v = ctypes.c_double()
    _check(_lib.load().axc_valu_issue_peak(ctypes.byref(v), None))
    return v.value


def lookup_mix_peak():
    """Table entries per second of a kernel made of nothing but the LUT-GEMM's per-lookup instructions (address,
    16-byte LDS read, accumulate), in its occupancy (measured)."""
    v = ctypes.c_double()
    _check(_lib.load().axc_lookup_mix_peak(ctypes.byref(v), None))
    return v.value


def dense_accumulate_ops_per_lookup():
    v = ctypes.c_double()
    _check(_lib.load().axc_dense_accumulate_ops_per_lookup(ctypes.byref(v)))
    return v.value


def device_info():
    a, b, c = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    _check(_lib.load().axc_device_info(ctypes.byref(a), ctypes.byref(b), ctypes.byref(c)))
    return {"compute_units": a.value, "lds_bytes_per_workgroup": b.value, "clock_khz": c.value}
