"""torch.Tensor <-> tv.Tensor without copies, and autograd functions around the mask-based sparse
convolution (forward = implicit_gemm2 Forward, backward = BackwardInput + BackwardWeight).

``torch2tensor`` / ``tensor2torch`` stand where the reference's ``PyTorchTools.torch2tensor`` /
``tensor2torch`` do (cumm/bindings.py:53-86 over include/tensorview/torch_utils.h).  torch is
plumbing here: it owns activations, parameters and the stream (allocation, zero fill, making a
tensor contiguous); every computing kernel that runs is this library's, including the ReLU gate
and the bias gradient of the backward pass.  Imported on demand: nothing else in the package
needs torch.
"""
import ctypes
import warnings
from typing import Optional, Sequence, Tuple

import torch

from . import _capi, pairs, tuner
from . import tensorview as tv
from .conv.main import ConvMainUnitTest
from .tensorview.gemm import Activation, ConvOpType, ConvParams

_TORCH_TO_TV = {torch.float32: tv.float32, torch.float16: tv.float16, torch.bfloat16: tv.bfloat16,
                torch.int32: tv.int32, torch.int8: tv.int8, torch.uint8: tv.uint8, torch.int64: tv.int64,
                torch.int16: tv.int16, torch.float64: tv.float64, torch.bool: tv.bool_}
_TV_TO_TORCH = {v: k for k, v in _TORCH_TO_TV.items()}
# torch has no full unsigned support: tensor2torch(cast_uint_to_int=True) views them as signed
_UINT_AS_INT = {tv.uint32: torch.int32, tv.uint16: torch.int16, tv.uint64: torch.int64}
_TYPESTR = {torch.float32: "<f4", torch.float16: "<f2", torch.int32: "<i4", torch.int8: "|i1", torch.uint8: "|u1",
            torch.int64: "<i8", torch.int16: "<i2", torch.float64: "<f8", torch.bool: "|b1"}


def torch2tensor(t: torch.Tensor) -> tv.Tensor:
    """A tv.Tensor over the storage of ``t`` (any strides); ``t`` is kept alive by the view."""
    if t.dtype not in _TORCH_TO_TV:
        raise ValueError("unsupported torch dtype %s" % t.dtype)
    device = t.device.index if t.is_cuda else -1
    if t.is_cuda and device is None:
        device = torch.cuda.current_device()
    return tv.from_blob_strided(t.data_ptr(), list(t.shape), list(t.stride()), _TORCH_TO_TV[t.dtype], device,
                                keepalive=t)


class _DeviceArray:
    """What torch.as_tensor needs to wrap device memory in place."""

    def __init__(self, ten: tv.Tensor, typestr: str, itemsize: int):
        self._keep = ten
        self.__cuda_array_interface__ = {
            "shape": tuple(ten.shape), "typestr": typestr, "data": (ten.byte_pointer(), False), "version": 2,
            "strides": tuple(s * itemsize for s in ten.stride)}


def tensor2torch(ten: tv.Tensor, clone: bool = True, cast_uint_to_int: bool = False) -> torch.Tensor:
    """The reference's signature (clone=True copies; clone=False shares the memory and keeps ``ten``
    alive)."""
    dt = ten.dtype
    if dt in _UINT_AS_INT:
        if not cast_uint_to_int:
            raise ValueError("torch has no such unsigned type: pass cast_uint_to_int=True")
        tdt = _UINT_AS_INT[dt]
    elif dt in _TV_TO_TORCH:
        tdt = _TV_TO_TORCH[dt]
    else:
        raise ValueError("unsupported tv dtype %d" % dt)
    if ten.empty():
        return torch.empty(list(ten.shape), dtype=tdt, device="cuda" if ten.device >= 0 else "cpu")
    if ten.device < 0:
        arr = ten.numpy_view()
        res = torch.from_numpy(arr).view(tdt) if tdt != torch.bfloat16 else torch.from_numpy(arr).view(torch.bfloat16)
    else:
        carrier = torch.int16 if tdt == torch.bfloat16 else tdt
        res = torch.as_tensor(_DeviceArray(ten, _TYPESTR[carrier], ten.itemsize), device="cuda:%d" % ten.device)
        if tdt == torch.bfloat16:
            res = res.view(torch.bfloat16)
    return res.clone() if clone else res


def current_stream() -> int:
    # (what torch.cuda.current_stream() wraps in an object: a tenth of the host time of a small forward pass)
    return torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())


_TUNER = tuner.Tuner(steps=3, warmup=1)


_DESP_LIKE = {}


def _desp_like(dtype, op, parallel=False, dynamic=False):
    """A descriptor of the wanted kind (the tuner then picks the tile); looked up once per kind:
    building the table of all descriptors costs more than a forward launch.  ``dynamic``: several
    mask words per position (kernel volumes above 32)."""
    key = (dtype, op, parallel, dynamic)
    if key not in _DESP_LIKE:
        for d in ConvMainUnitTest.get_all_conv_algo_desp():
            if (d.dtype_a == dtype and d.dtype_c == dtype and ConvOpType(d.op_type) == op and not d.is_int8_inference and
                    bool(d.split_k_parallel) == parallel and d.mask_sparse and bool(d.dynamic_mask) == dynamic):
                _DESP_LIKE[key] = d
                break
        else:
            raise RuntimeError("can't find any suitable algo for your parameters.")
    return _DESP_LIKE[key].copy()


# the fields of the argument block that hold each tensor's address.  By the pass and never by comparing
# addresses: tensors of a call may share their storage (a gradient that is the layer's own input).  D is the
# result itself where no bias is added.
_FIELDS = {
    ConvOpType.Forward: {"input": ("ptr_A",), "weight": ("ptr_B",), "output": ("ptr_C", "ptr_D")},
    ConvOpType.BackwardInput: {"output": ("ptr_A",), "weight": ("ptr_B",), "input": ("ptr_C", "ptr_D")},
    ConvOpType.BackwardWeight: {"output": ("ptr_A",), "input": ("ptr_B",), "weight": ("ptr_C", "ptr_D"), "workspace": ("workspace",)},
}
_WITH_BIAS = dict(_FIELDS[ConvOpType.Forward], output=("ptr_C",), bias=("ptr_D", "bias_pointer"))


class _Launch:
    """The validated argument block of one operator call, replayed with other tensors of the same
    shapes - and on other geometries: the first call of its kind goes through the operator's prelude
    and the tuner (close to a millisecond of Python), a repeat copies the block, patches the pointers
    that change from call to call into it and calls the C entry point.  A copy per call, so that
    threads can share a geometry."""

    __slots__ = ("fn", "cdesc", "args", "fields", "tile_m", "_call")

    def __init__(self, fn, cdesc, args, fields, tile_m):
        self.fn, self.cdesc, self.args, self.fields, self.tile_m = fn, cdesc, args, fields, tile_m
        self._call = ctypes.byref(cdesc)

    @classmethod
    def of(cls, params: ConvParams, roles) -> "_Launch":
        prep = params.__dict__.get("_prepared")
        if prep is None:
            raise RuntimeError("the operator call left no validated argument block")
        args = _copy(prep[5])
        fields = _WITH_BIAS if "bias" in roles else _FIELDS[ConvOpType(params.conv_algo_desp.op_type)]
        for role, t in roles.items():
            if t.numel() and any(getattr(args, f) != t.data_ptr() for f in fields[role]):
                raise RuntimeError("the argument block does not point at the %s tensor" % role)
        return cls(prep[1], prep[4], args, fields, int(params.conv_algo_desp.tile_shape[0]))

    def on(self, n_pos, rows_in, rows_out, indices, mask, argsort, mask_out) -> "_Launch":
        """The same call on another geometry (device addresses)."""
        args = _copy(self.args)
        args.N, args.rows_in, args.rows_out = n_pos, rows_in, rows_out
        args.indice_ptr, args.mask_ptr, args.mask_argsort_ptr, args.mask_out_ptr = indices, mask, argsort, mask_out
        return _Launch(self.fn, self.cdesc, args, self.fields, self.tile_m)

    def __call__(self, stream: int, workspace_bytes: int = 0, **tensors) -> None:
        args = _copy(self.args)
        for role, t in tensors.items():
            ptr = t.data_ptr()
            for f in self.fields[role]:
                setattr(args, f, ptr)
        if workspace_bytes:
            args.workspace_bytes = workspace_bytes
        status = self.fn(self._call, ctypes.byref(args), stream)
        if status:
            _capi.check(status)


def _copy(args: _capi.SparseConvArgs) -> _capi.SparseConvArgs:
    return _capi.SparseConvArgs.from_buffer_copy(args)


# validated calls by kind (pass, types, channels, kernel volume, epilogue, size class): what _Launch.on
# moves to the next geometry.  Bounded by the kinds of layers a program has.
_KINDS = {}


_NATIVE_SYMBOLS = ("sparse_conv_more", "last_error", "relu_backward", "gate_sums", "column_sum_workspace",
                   "query_conv_workspace", "query_wgrad_ordered_workspace", "wgrad_pairs_sums", "wgrad_pairs_workspace", "subm_pairs",
                   "subm_pairs_workspace", "conv_pairs_workspace", "conv_pairs_sites", "conv_pairs_fill", "order_pairs_coarse",
                   "order_pairs_coarse_workspace")
_native_module = None


def _native():
    """The native half of this module (csrc/torch_native.cpp), built first if it is not there or not of these sources
    and this torch; None where that cannot be done - no host compiler, no headers of torch: the functions here make all calls then."""
    global _native_module
    if _native_module is None:
        from . import build
        try:
            build.build_torch_native()
            from . import _torch_native as native
        except (ImportError, OSError, RuntimeError) as e:
            warnings.warn("the native half of the torch bridge is not there, Python makes its calls: %s" % e, RuntimeWarning)
            _native_module = False
        else:
            native.bind({"cumm_hip_" + n: ctypes.cast(getattr(_capi.lib(), "cumm_hip_" + n), ctypes.c_void_p).value
                         for n in _NATIVE_SYMBOLS})
            native.set_backward(_backward)
            _native_module = native
    return _native_module or None


def _remember(g: "SparseConvGeometry", key, kind, launch: "_Launch", op: ConvOpType, features, weight, bias=None) -> None:
    """A validated call of a kind, for the geometries to come - here and in native code."""
    _KINDS[kind] = launch
    if g._native is None:
        return
    relu, tile_m, deterministic = key[5] if key[0] == "fwd" else False, key[3] if key[0] == "wgrad" else 0, key[-1]
    n_pos = g.n_in if op == ConvOpType.BackwardInput else g.n_out
    _native().remember(op.value, features.dtype, weight.dtype, None if bias is None else bias.dtype, int(weight.shape[0]),
                       int(weight.shape[2]), g.kv, g.subm, _size_class(n_pos), g._device.index, bool(relu), tile_m, deterministic,
                       bytes(launch.cdesc), bytes(launch.args), launch.tile_m)


def _size_class(n: int) -> int:
    return max(n - 1, 0).bit_length()      # (the tuner's bucket of the position count)


def _bytes(n: int, device) -> torch.Tensor:
    return torch.empty(max(int(n), 256), dtype=torch.uint8, device=device)


# output channels from which the gradient's gate and sums go by position (torch_native.cpp has the same, and why)
_GATE_FROM = 64


class _HandedOut:
    """What a tv tensor over the block of a geometry keeps alive: its memory goes back to torch's allocator as
    tv's own storage goes back to the driver, when the device has finished with it.  (The operators run
    such a tensor on streams that torch's allocator does not hear of.)"""

    def __init__(self, block: torch.Tensor):
        self.block = block

    def __del__(self):
        try:
            if not torch.cuda.is_current_stream_capturing():
                torch.cuda.synchronize(self.block.device)
        except Exception:
            pass


class SparseConvGeometry:
    """Pair tables, masks and sorts of one convolution geometry, built on the GPU once and shared by
    every layer (and every pass) that uses it.  Kernel volumes up to 32 have one mask word per
    position; above that (up to 128, e.g. 5 x 5 x 5) the masks have ``ceil(kv / 32)`` words, forward
    and backward-input run on the ``dynamic_mask`` descriptors, and backward-weight - which has no
    such kernel, in the reference neither - goes over the pair lists of all offsets.

    All tables lie in one block from torch's caching allocator (a new cloud per iteration then
    allocates nothing from the driver); ``indices_fwd`` and the other tables are views of it."""

    _TABLES = ("indices_fwd", "indices_bwd", "mask_fwd", "order_fwd", "mask_bwd", "order_bwd", "indices_fwd_pos", "indices_bwd_pos")
    _lists = _list_block = None      # (several mask words only)
    _partial = frozenset()           # tables by position that are written only where the launches read them
    _recorded = False                # built while its stream was recorded: every replay writes the tables anew
    _native = None                   # the geometry as native code has it

    def __init__(self, coords: torch.Tensor, spatial_shape: Sequence[int], ksize=(3, 3, 3), stride=None,
                 padding=(1, 1, 1), dilation=(1, 1, 1), batch_size: int = 1):
        if coords.dtype != torch.int32 or not coords.is_cuda or coords.dim() != 2 or coords.shape[1] != 4:
            raise ValueError("coords must be a cuda int32 tensor [N, 4] of (batch, z, y, x)")
        self.subm = stride is None
        if self.subm:
            pairs._check_odd_ksize(ksize)
        three = lambda a: tuple(int(v) for v in a)
        ksize = three(ksize)
        self.kv = kv = ksize[0] * ksize[1] * ksize[2]
        self.words = words = (kv + 31) // 32
        self._stream, self._device, self.n_in = current_stream(), coords.device, int(coords.shape[0])
        # (how far the light end of each sorted order reaches - the hint of the forward and backward-input
        # launches - stays on the device: the sort leaves it in the library's table under the sorted
        # array's address and the launches look it up there; 0 = not given here)
        self.light_fwd = self.light_bwd = 0
        self._reduced, self._reduced_streams, self._written = {}, {}, set()
        self._own_launches = {}      # calls of the layers on this geometry, see _Launch
        self._tensors = {}
        geo = (coords.contiguous(), three(spatial_shape), ksize, None if self.subm else three(stride), three(padding), three(dilation),
               int(batch_size))
        native = _native()
        if native is not None:
            self._native, self.out_coords, self.out_shape, ordered = native.build(*geo)
            self.n_out, self._block = self._native.n_out, self._native.block
        else:
            ordered = self._build(*geo)
        # masks, an order of the positions by them, and the pair tables once more in that order: what
        # forward and backward-input read (a tile's entries for one offset are then consecutive in
        # memory); backward-weight keeps the table by row
        if ordered:
            self._partial = frozenset(("indices_fwd_pos", "indices_bwd_pos"))
            self._recorded = torch.cuda.is_current_stream_capturing()
        else:
            self._order_one_by_one()
        if words > 1:
            self._make_lists()

    def _build(self, coords, spatial_shape, ksize, stride, padding, dilation, batch_size) -> bool:
        """Tables, order and tables by position, where native code does not make them; False: large tables, to be
        ordered by _order_one_by_one."""
        lib, arr3, s, dev, n_in = _capi.lib(), ctypes.c_int32 * 3, self._stream, self._device, self.n_in
        shape, ks, pad, dil = (arr3(*a) for a in (spatial_shape, ksize, padding, dilation))
        if self.subm:
            self.n_out, self.out_coords, self.out_shape = n_in, coords, spatial_shape
            self._allocate()
            ws = _bytes(lib.cumm_hip_subm_pairs_workspace(n_in), dev)
            _capi.check(lib.cumm_hip_subm_pairs(coords.data_ptr(), n_in, shape, ks, dil, self._ptr["indices_fwd"], self._ptr["indices_bwd"],
                                                None, None, ws.data_ptr(), ws.numel(), s))
        else:
            geo = (shape, ks, arr3(*stride), pad, dil)
            need = int(lib.cumm_hip_conv_pairs_workspace(n_in, batch_size, *geo))
            if need == 0:
                raise ValueError("bad geometry (kernel volume 1..128, non-empty output grid) or too many voxels")
            ws = _bytes(need, dev)
            out_shape, found = arr3(), ctypes.c_int32(0)
            _capi.check(lib.cumm_hip_conv_pairs_sites(coords.data_ptr(), n_in, batch_size, *geo, out_shape, ctypes.byref(found),
                                                      ws.data_ptr(), ws.numel(), s))
            self.n_out, self.out_shape = int(found.value), tuple(out_shape)
            self.out_coords = torch.empty((self.n_out, 4), dtype=torch.int32, device=dev)
            self._allocate()
            _capi.check(lib.cumm_hip_conv_pairs_fill(coords.data_ptr(), n_in, batch_size, *geo, self.n_out, self.out_coords.data_ptr(),
                                                     self._ptr["indices_fwd"], self._ptr["indices_bwd"], None, None, ws.data_ptr(),
                                                     ws.numel(), s))
        if 4 * self.kv * max(n_in, self.n_out) >= 1 << 31:
            return False
        sides, p = (_capi.OrderSide * 2)(), self._ptr
        for d, side, n in ((sides[0], "fwd", self.n_out), (sides[1], "bwd", n_in)):
            d.indices, d.n = p["indices_" + side], n
            d.sorted_mask, d.argsort, d.by_position = p["mask_" + side], p["order_" + side], p["indices_%s_pos" % side]
        count = 2
        if self.subm:      # (one order serves both; the backward table is the forward one with its offsets reversed)
            sides[0].by_position_reversed, count = p["indices_bwd_pos"], 1
        ws = _bytes(lib.cumm_hip_order_pairs_coarse_workspace(sides, count, self.kv), dev)
        _capi.check(lib.cumm_hip_order_pairs_coarse(sides, count, ks, ws.data_ptr(), ws.numel(), s))
        return True

    @property
    def _launches(self):
        """The calls of the layers on this geometry; of a pass that native code made alone, its name."""
        calls = dict(self._own_launches)
        if self._native is not None:
            names = ("fwd", "dgrad", "wgrad" if self.words == 1 else "wgrad_pairs")
            own = {key[0] for key in calls}
            calls.update({(name,): None for i, name in enumerate(names) if self._native.made(i) and name not in own})
        return calls

    @_launches.setter
    def _launches(self, calls):
        self._own_launches = calls

    def _order_one_by_one(self) -> None:
        """For tables of 2^31 bytes and more, which cumm_hip_order_pairs and the launches refuse: whoever builds
        one wants the tables (the per-offset convolution walks lists of them)."""
        lib, p, s, kv, words = _capi.lib(), self._ptr, self._stream, self.kv, self.words
        for side, n in (("fwd", self.n_out), ("bwd", self.n_in)):
            if side == "fwd" or not self.subm:
                raw = torch.empty((n, words), dtype=torch.int32, device=self._device)
                _capi.check(lib.cumm_hip_masks_from_pairs(p["indices_" + side], kv, n, raw.data_ptr(), s))
                need = lib.cumm_hip_sort_by_mask_workspace(n) if words == 1 else lib.cumm_hip_sort_by_mask_words_workspace(n)
                ws = _bytes(need, self._device)
                to = (p["mask_" + side], p["order_" + side], ws.data_ptr(), ws.numel(), s)
                if words == 1:
                    bits = (1 << kv) - 1 if kv < 32 else 0xFFFFFFFF
                    _capi.check(lib.cumm_hip_sort_by_mask_ordered(raw.data_ptr(), n, bits, int(kv <= 27), *to))
                else:
                    _capi.check(lib.cumm_hip_sort_by_mask_words(raw.data_ptr(), n, words, *to))
            _capi.check(lib.cumm_hip_pairs_by_position(p["indices_" + side], p["order_" + side], kv, n, p["indices_%s_pos" % side], s))

    def _allocate(self) -> None:
        self._block = _bytes(self._lay_out(0), self._device)
        self._lay_out(self._block.data_ptr())

    def _lay_out(self, base: int) -> int:
        """Where the tables lie in the block (torch_native.cpp has the same); its size."""
        n_out, n_in, kv, words = self.n_out, self.n_in, self.kv, self.words
        mask = [self.n_out] if words == 1 else [n_out, words]
        spec = [("indices_fwd", [kv, n_out], tv.int32), ("indices_bwd", [kv, n_in], tv.int32),
                ("indices_fwd_pos", [kv, n_out], tv.int32), ("indices_bwd_pos", [kv, n_in], tv.int32),
                ("mask_fwd", mask, tv.uint32), ("order_fwd", [n_out], tv.int32)]
        mask = [n_in] if words == 1 else [n_in, words]
        if not self.subm:
            spec += [("mask_bwd", mask, tv.uint32), ("order_bwd", [n_in], tv.int32)]
        self._spec, at = {}, 0
        for name, dims, dtype in spec:
            self._spec[name] = (at, dims, dtype)
            size = 4
            for d in dims:
                size *= d
            at += (size + 255) // 256 * 256
        # the words of tiles of 64 and of 128 positions, rounded up to 256 bytes (see reduced_address)
        reduced_64, reduced_128 = at, at + (n_out // 64 + 64) // 64 * 256
        if words == 1:
            at = reduced_128 + (n_out // 128 + 64) // 64 * 256
        self._ptr = {name: base + v[0] for name, v in self._spec.items()}
        self._reduced_at = {64: base + reduced_64, 128: base + reduced_128} if words == 1 else {}
        if self.subm:      # the forward masks serve the backward-input pass, bit-reversed in the kernel
            for name in ("mask", "order"):
                self._spec[name + "_bwd"], self._ptr[name + "_bwd"] = self._spec[name + "_fwd"], self._ptr[name + "_fwd"]
        return at

    def _make_lists(self) -> None:
        """The per-offset pair lists of backward-weight; their counts come to the host."""
        n, kv, lib = self.n_out, self.kv, _capi.lib()
        lists = torch.empty((2, kv, n), dtype=torch.int32, device=self._device)
        counts = torch.empty(kv, dtype=torch.int32, device=self._device)
        need = int(lib.cumm_hip_pair_lists_workspace(kv, n))
        ws = _bytes(need, self._device)
        _capi.check(lib.cumm_hip_pair_lists(self._ptr["indices_fwd"], kv, n, lists[0].data_ptr(), lists[1].data_ptr(),
                                            counts.data_ptr(), ws.data_ptr(), ws.numel(), self._stream))
        self._list_block = lists
        counts = counts.cpu().numpy()
        self._lists = self._lists_over(lists, counts)
        if self._native is not None:
            self._native.set_lists(lists, counts.clip(0, n).tolist())

    def _lists_over(self, keepalive, counts) -> pairs.DevicePairLists:
        pair_in, pair_out = (tv.from_blob(t.data_ptr(), [self.kv, self.n_out], tv.int32, self._device.index, keepalive=keepalive)
                             for t in self._list_block)
        return pairs.DevicePairLists(pair_in, pair_out, counts)

    def __getattr__(self, name: str):
        if name == "lists":      # (the passes take their own, whose streams are recorded)
            own = self._lists
            self.lists = None if own is None else self._lists_over(_HandedOut(self._list_block), own.counts)
            return self.lists
        if name in ("_spec", "_ptr", "_reduced_at") and self._native is not None:
            self._lay_out(self._block.data_ptr())      # (where somebody asks)
            return self.__dict__[name]
        if name not in SparseConvGeometry._TABLES or self.__dict__.get("_block") is None:
            raise AttributeError(name)
        if name in self._partial:
            self._complete(name)
        return self._view(name)

    def _complete(self, name: str) -> None:
        """Whoever looks at a table by position gets all of it: the entries of runs without a pair are written too (the
        others once more, as they are).  Behind the construction, whatever stream and device the reader is on: it
        needs to be ordered behind that only when it uses the table, as for every other one.  Where a stream is being
        recorded nothing waits: what is there before a graph, torch has waited for when it begins."""
        side, lib = name[8:11], _capi.lib()
        n = self.n_out if side == "fwd" else self.n_in
        with torch.cuda.device(self._device):
            stream, recorded = current_stream(), torch.cuda.is_current_stream_capturing()
            if n:
                if not recorded and stream != self._stream and not lib.cumm_hip_stream_is_capturing(self._stream):
                    _capi.check(lib.cumm_hip_stream_synchronize(self._stream))
                self.used_on(stream)
                _capi.check(lib.cumm_hip_pairs_by_position(self._ptr["indices_" + side], self._ptr["order_" + side], self.kv, n,
                                                           self._ptr[name], stream))
            if not recorded:
                torch.cuda.current_stream().synchronize()      # (it may be read on any stream)
                if not self._recorded:
                    self._partial = self._partial - {name}

    def _view(self, name: str) -> tv.Tensor:
        t = self._tensors.get(name)
        if t is None:
            _, dims, dtype = self._spec[name]
            t = self._tensors[name] = tv.from_blob(self._ptr[name], dims, dtype, self._device.index,
                                                    keepalive=_HandedOut(self._block))
        return t

    def used_on(self, stream: int) -> None:
        """Tell torch's allocator that ``stream`` - the current one - reads the tables."""
        if stream != self._stream:
            current = torch.cuda.current_stream()
            self._block.record_stream(current)
            if self._lists is not None:
                self._list_block.record_stream(current)
        for width, own in self._reduced_streams.items():
            if stream != own:
                self._reduced[width].record_stream(torch.cuda.current_stream())

    def reduced_address(self, width: int) -> int:
        """One word per run of ``width`` sorted output positions: the forward launch writes (all of) the
        OR of the run's masks here (its ``mask_output``), and backward-weight reads it.  The words of the
        kernels' tile heights lie in the block of the tables: memory that the first forward pass took from
        its own stream's pool could be in use there still when another stream writes it, and again while
        another stream reads it."""
        self._written.add(width)
        if width in self._reduced_at:
            return self._reduced_at[width]
        buf = self._reduced.get(width)
        if buf is None:
            buf = torch.empty(max((self.n_out + width - 1) // width, 1), dtype=torch.int32, device=self._device)
            self._reduced[width], self._reduced_streams[width] = buf, current_stream()
        return buf.data_ptr()

    def reduced_mask_buffer(self, width: int) -> tv.Tensor:
        """Those words as a tv tensor; zeros until a forward pass with tiles of that height has run."""
        fresh = width not in self._written and not (self._native is not None and self._native.written(width))
        at, count = self.reduced_address(width), max((self.n_out + width - 1) // width, 1)
        owner = self._reduced.get(width, self._block)
        if fresh:
            first = at - owner.data_ptr()
            (owner[first:first + 4 * count] if owner is self._block else owner).zero_()
        return tv.from_blob(at, [count], tv.uint32, self._device.index, keepalive=owner)


class _SparseConvFunction(torch.autograd.Function):

    @staticmethod
    def forward(ctx, features, weight, bias, geometry: SparseConvGeometry, relu: bool):
        features, weight = features.contiguous(), weight.contiguous()
        if features.dim() != 2 or features.shape[0] != geometry.n_in:
            raise ValueError("features must be [%d, C]: one row per input site of the geometry" % geometry.n_in)
        if weight.dim() != 3 or weight.shape[1] != geometry.kv or weight.shape[2] != features.shape[1]:
            raise ValueError("weight must be [K, %d, %d]" % (geometry.kv, features.shape[1]))
        _check_device(geometry, features, weight, bias)      # (a remembered call takes addresses)
        out = torch.empty((geometry.n_out, weight.shape[0]), dtype=features.dtype, device=features.device)
        roles = {"input": features, "weight": weight, "output": out}
        if bias is not None:
            roles["bias"] = bias = bias.contiguous()
        stream = current_stream()
        geometry.used_on(stream)
        key = ("fwd", features.dtype, weight.dtype, weight.shape, None if bias is None else (bias.dtype, bias.shape), relu, _deterministic())
        launch = geometry._own_launches.get(key)
        if launch is None:
            launch = _forward_launch(geometry, key, roles, relu, stream)
        launch(stream, **roles)
        ctx.geometry, ctx.relu, ctx.has_bias, ctx.tile_m = geometry, relu, bias is not None, launch.tile_m
        ctx.save_for_backward(features, weight, out if relu else None)
        return out

    @staticmethod
    def backward(ctx, grad_out):
        features, weight, out = ctx.saved_tensors
        return _backward(ctx.geometry, features, weight, out, grad_out, ctx.needs_input_grad, ctx.relu, ctx.has_bias, ctx.tile_m) + (None, None)


def _backward(g: SparseConvGeometry, features, weight, out, grad_out, needed, relu: bool, has_bias: bool, tile_m: int):
    """The gradients of features, weight and bias (None where not ``needed``)."""
    _check_device(g, features, weight, out, grad_out)      # (saved-tensor hooks may have moved them)
    grad_out = grad_out.contiguous()
    dtype = _TORCH_TO_TV[features.dtype]
    stream = current_stream()
    g.used_on(stream)
    lib = _capi.lib()
    grad_in = grad_w = grad_b = None
    # the gradient passes where the fused ReLU let the output through; its column sums are the
    # bias gradient (one pass over the gradient for both)
    rows, k_out = int(grad_out.shape[0]), int(grad_out.shape[1])
    if has_bias and needed[2]:
        grad_b = torch.empty(k_out, dtype=grad_out.dtype, device=grad_out.device)
        need = int(lib.cumm_hip_column_sum_workspace(rows, k_out))
        ws = _bytes(need, grad_out.device)
        if relu:
            gated = torch.empty_like(grad_out)
            sums = _capi.GateSums(gated.data_ptr(), grad_b.data_ptr(), grad_out.data_ptr(), out.data_ptr(), rows, k_out,
                                  ws.data_ptr(), ws.numel(), None, g._ptr["order_fwd"] if k_out >= _GATE_FROM else None)
            _capi.check(lib.cumm_hip_gate_sums(ctypes.byref(sums), dtype, stream))
            grad_out = gated
        else:
            _capi.check(lib.cumm_hip_column_sum(grad_b.data_ptr(), grad_out.data_ptr(), rows, k_out, dtype,
                                                ws.data_ptr(), ws.numel(), stream))
    elif relu:
        gated = torch.empty_like(grad_out)
        _capi.check(lib.cumm_hip_relu_backward(gated.data_ptr(), grad_out.data_ptr(), out.data_ptr(),
                                               grad_out.numel(), dtype, stream))
        grad_out = gated
    if needed[0]:
        # inputs that feed no output site sit in tiles the kernel skips (mask 0): zero them
        grad_in = torch.empty_like(features) if g.subm else torch.zeros_like(features)
        roles = {"input": grad_in, "weight": weight, "output": grad_out}
        key = ("dgrad", dtype, weight.shape, _deterministic())
        launch = g._own_launches.get(key)
        if launch is None:
            launch = _backward_input_launch(g, key, roles, dtype, stream)
        launch(stream, **roles)
    if needed[1] and g.words > 1:
        # no mask kernel for this pass: the products of all kernel offsets over their pair lists, in
        # one call (an offset without pairs writes zeros)
        from .conv import native
        grad_w = torch.empty_like(weight)
        key = ("wgrad_pairs", dtype, weight.shape)
        plan = g._own_launches.get(key)
        if plan is None:
            plan = native.WeightPlan(torch2tensor(grad_out), torch2tensor(features), torch2tensor(grad_w), g._lists, stream)
            plan.release()      # (every call brings its own tensors)
            g._own_launches[key] = plan
        ws = _bytes(plan.workspace_bytes, grad_out.device)
        plan.rebind(grad_out.data_ptr(), features.data_ptr(), grad_w.data_ptr(), stream, ws.data_ptr())
    elif needed[1]:
        grad_w = torch.empty_like(weight)
        key = ("wgrad", dtype, weight.shape, tile_m, _deterministic())
        hit = g._own_launches.get(key)
        if hit is None:
            hit = g._own_launches[key] = _backward_weight_launch(g, key, features, weight, grad_w, grad_out, dtype, stream)
        launch, need = hit
        # the workspace comes from torch's caching allocator (the prelude's own would be a
        # device allocation per call)
        ws = _bytes(need, grad_out.device)
        launch(stream, need, input=features, weight=grad_w, output=grad_out, workspace=ws)
    return grad_in, grad_w, grad_b


def _deterministic() -> bool:
    """torch's switch for reproducible results: rows added up in one order whatever tile the tuner has picked, weight
    gradients by the fixed-order sum of the partial blocks."""
    return bool(torch.are_deterministic_algorithms_enabled())


def _check_device(g: SparseConvGeometry, *tensors) -> None:
    if any(t is not None and t.device != g._device for t in tensors):
        raise ValueError("all tensors must be on the same device")


def _kind(g: SparseConvGeometry, key, n_pos: int, *tensors):
    """The key of a call in _KINDS; the tensors of a first call are checked here for what the operator's
    prelude checks and a moved call does not: one device, that of the tables (types and shapes are in the
    key)."""
    _check_device(g, *tensors)
    return key + (g.kv, g.subm, _size_class(n_pos), g._device.index)


def _forward_launch(g: SparseConvGeometry, key, roles, relu, stream) -> _Launch:
    features, weight, out, bias = roles["input"], roles["weight"], roles["output"], roles.get("bias")
    kind = _kind(g, key, g.n_out, *roles.values())
    known = _KINDS.get(kind)
    if known is not None and features.numel() and out.numel():
        launch = known.on(g.n_out, g.n_in, g.n_out, g._ptr["indices_fwd_pos"], g._ptr["mask_fwd"], g._ptr["order_fwd"],
                          g.reduced_address(known.tile_m) if g.words == 1 else None)
        g._own_launches[key] = launch
        _remember(g, key, kind, known, ConvOpType.Forward, features, weight, bias)
        return launch
    p = ConvParams(3, ConvOpType.Forward)
    dtype = _TORCH_TO_TV[features.dtype]
    p.conv_algo_desp = _desp_like(dtype, ConvOpType.Forward, dynamic=g.words > 1)
    p.input, p.weight, p.output = torch2tensor(features), torch2tensor(weight), torch2tensor(out)
    p.indices, p.mask, p.mask_argsort = g._view("indices_fwd_pos"), g.mask_fwd, g.order_fwd
    p.indices_by_position = True
    p.mask_int_count = g.words
    p.light_prefix = g.light_fwd
    if bias is not None:
        p.bias, p.beta = torch2tensor(bias), 1.0
    if relu:
        p.act_type = Activation.ReLU
    p.deterministic = key[-1]
    p.stream = stream
    _TUNER.tune_conv(p)
    # the tile masks the forward launch computes anyway are what backward-weight needs
    # (not for several mask words: that backward-weight walks the pair lists)
    if g.words == 1:
        p.mask_output = g.reduced_mask_buffer(int(p.conv_algo_desp.tile_shape[0]))
    ConvMainUnitTest.implicit_gemm2(p)
    launch = g._own_launches[key] = _Launch.of(p, roles)
    _remember(g, key, kind, launch, ConvOpType.Forward, features, weight, bias)
    return launch


def _backward_input_launch(g: SparseConvGeometry, key, roles, dtype, stream) -> _Launch:
    grad_in, weight, grad_out = roles["input"], roles["weight"], roles["output"]
    kind = _kind(g, key, g.n_in, *roles.values())
    known = _KINDS.get(kind)
    if known is not None and grad_in.numel() and grad_out.numel():
        launch = known.on(g.n_in, g.n_in, g.n_out, g._ptr["indices_bwd_pos"], g._ptr["mask_bwd"], g._ptr["order_bwd"], None)
        g._own_launches[key] = launch
        _remember(g, key, kind, known, ConvOpType.BackwardInput, grad_in, weight)
        return launch
    p = ConvParams(3, ConvOpType.BackwardInput)
    p.conv_algo_desp = _desp_like(dtype, ConvOpType.BackwardInput, dynamic=g.words > 1)
    p.input, p.weight, p.output = torch2tensor(grad_in), torch2tensor(weight), torch2tensor(grad_out)
    p.indices, p.mask, p.mask_argsort = g._view("indices_bwd_pos"), g.mask_bwd, g.order_bwd
    p.indices_by_position = True
    p.mask_int_count = g.words
    p.reverse_mask = g.subm
    p.light_prefix = g.light_bwd
    p.deterministic = key[-1]
    p.stream = stream
    _TUNER.tune_conv(p)
    ConvMainUnitTest.implicit_gemm2(p)
    launch = g._own_launches[key] = _Launch.of(p, roles)
    _remember(g, key, kind, launch, ConvOpType.BackwardInput, grad_in, weight)
    return launch


def _backward_weight_launch(g: SparseConvGeometry, key, features, weight, grad_w, grad_out, dtype, stream):
    """(call, bytes of workspace)"""
    tile_m, deterministic = key[3], key[4]
    n_pos, k_out, kv, c_in = int(grad_out.shape[0]), int(weight.shape[0]), int(weight.shape[1]), int(weight.shape[2])
    desp = _desp_like(dtype, ConvOpType.BackwardWeight, parallel=True)
    slices = 32
    need = desp.query_conv_workspace_size(k_out, kv * c_in, n_pos, slices, kv)
    if deterministic:
        need = max(need, int(_capi.lib().cumm_hip_query_wgrad_ordered_workspace(n_pos, c_in, k_out, kv, tile_m)))
    need = max(int(need), 256)
    kind = _kind(g, key, n_pos, grad_out, features, grad_w)
    known = _KINDS.get(kind)
    if known is not None and features.numel() and grad_out.numel():
        return known.on(n_pos, g.n_in, g.n_out, g._ptr["indices_fwd"], g.reduced_address(tile_m), g._ptr["order_fwd"],
                        None), need
    p = ConvParams(3, ConvOpType.BackwardWeight)
    p.conv_algo_desp = desp
    p.input, p.weight, p.output = torch2tensor(features), torch2tensor(grad_w), torch2tensor(grad_out)
    p.indices, p.mask, p.mask_argsort = g.indices_fwd, g.reduced_mask_buffer(tile_m), g.order_fwd
    p.mask_width, p.split_k_slices = tile_m, slices
    p.deterministic = deterministic
    ws = _bytes(need, grad_out.device)
    p.workspace = torch2tensor(ws)
    p.stream = stream
    ConvMainUnitTest.implicit_gemm2(p)
    launch = _Launch.of(p, {"input": features, "weight": grad_w, "output": grad_out, "workspace": ws})
    _remember(g, key, kind, launch, ConvOpType.BackwardWeight, features, grad_w)
    return launch, need


def sparse_conv(features: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor],
                geometry: SparseConvGeometry, relu: bool = False) -> torch.Tensor:
    """features [N_in, C], weight [K, kv, C] (f16 / bf16, cuda) -> [N_out, K]; differentiable in
    features, weight and bias."""
    native = geometry._native
    if native is not None and not torch._C._are_functorch_transforms_active() and not torch.compiler.is_compiling():
        out = _native_module.forward(features, weight, bias, geometry, native, bool(relu))
        if out is not None:
            return out
    return _SparseConvFunction.apply(features, weight, bias, geometry, relu)


class SparseConv3d(torch.nn.Module):
    """A layer over :func:`sparse_conv`: submanifold when its geometry was built without a stride."""

    def __init__(self, in_channels: int, out_channels: int, ksize=(3, 3, 3), bias: bool = True, relu: bool = False,
                 dtype=torch.float16, device="cuda"):
        super().__init__()
        kv = int(ksize[0]) * int(ksize[1]) * int(ksize[2])
        w = torch.randn(out_channels, kv, in_channels, device=device) * (2.0 / (kv * in_channels)) ** 0.5
        self.weight = torch.nn.Parameter(w.to(dtype))
        self.bias = torch.nn.Parameter(torch.zeros(out_channels, dtype=dtype, device=device)) if bias else None
        self.relu = relu

    def forward(self, features: torch.Tensor, geometry: SparseConvGeometry) -> torch.Tensor:
        return sparse_conv(features, self.weight, self.bias, geometry, self.relu)
