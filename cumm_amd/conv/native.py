"""Per-offset ("native") sparse convolution: one gather-GEMM-scatter per kernel offset.

``SparseConvAlgo.Native`` of the reference (include/tensorview/gemm/core/constants.h:34-38): what
its callers fall back to when the mask-based kernels do not apply; kernel volumes above 32 take the
``dynamic_mask`` descriptors forward and backward-input, and this path for their weight gradient.  The
pattern is the reference's own check of its kernels, cumm/conv/main_real_spconv.py:309-403:

    forward          out[pair_out[k]]  += inp[pair_in[k]]   @ W[:, k, :].T     (matmul2, ShuffleAC)
    backward-input   dinp[pair_in[k]]  += dout[pair_out[k]] @ W[:, k, :]       (matmul2, ShuffleAC)
    backward-weight  dW[:, k, :]        = dout[pair_out[k]].T @ inp[pair_in[k]] (all offsets in one call)

Forward and backward-input accumulate all offsets in an fp32 image (the f16 / bf16 -> f32 kernels)
and round once at the end (``cumm_hip_finish_rows``, with bias and activation): one rounding, as
the mask-based kernels make, instead of one per offset.
"""
import ctypes
import threading
from typing import Optional

import numpy as np

from .. import _capi
from .. import tensorview as tv
from ..gemm.main import GemmMainUnitTest, _check_device, _check_dtype, _Slots, desp_to_c
from ..tensorview.gemm import Activation, GemmParams, ShuffleStrideType


_FOUND = {}


def _find(dtype: int, dtype_c: int, shuffle: ShuffleStrideType, tile_m: int, tile_n: int, trans_a: bool,
          trans_b: bool):
    key = (dtype, dtype_c, shuffle, tile_m, tile_n, trans_a, trans_b)
    if key not in _FOUND:
        for d in _descs():
            if (d.dtype_a == dtype and d.dtype_c == dtype_c and d.shuffle_type == shuffle and
                    d.tile_shape[0] == tile_m and d.tile_shape[1] == tile_n and d.trans_a == trans_a and
                    d.trans_b == trans_b and not d.trans_c):
                _FOUND[key] = d
                break
        else:
            raise RuntimeError("can't find any suitable algo for your parameters.")
    return _FOUND[key]


_DESCS = None


def _descs():
    global _DESCS
    if _DESCS is None:
        _DESCS = GemmMainUnitTest.get_all_algo_desp()
    return _DESCS


def _check(inp, weight, lists, n_rows_out):
    if inp.ndim != 2 or weight.ndim != 3:
        raise RuntimeError("error")
    if inp.dtype != weight.dtype or inp.dtype not in (tv.float16, tv.bfloat16):
        raise RuntimeError("the native path takes f16 or bf16 features and weights of one type")
    kv = weight.dim(1)
    if lists.pair_in.dim(0) != kv or lists.pair_out.dim(0) != kv or len(lists.counts) != kv:
        raise RuntimeError("pair lists and weight disagree on the kernel volume")
    if inp.dim(1) % 8 or weight.dim(0) % 8 or weight.dim(2) % 8:
        raise RuntimeError("channel counts must be multiples of 8")
    return kv


def _accumulate_steps(a, a_inds_all, c_inds_all, counts, weight, acc, trans_b, stream):
    """One validated ``GemmParams`` per offset with pairs: acc[c_inds[k]] += a[a_inds[k]] @ op(W[:, k, :])."""
    kv = weight.dim(1)
    n_ch = acc.dim(1)
    steps = []
    for k in range(kv):
        cnt = int(counts[k])
        if cnt == 0:
            continue
        p = GemmParams()
        tile_m = 128 if cnt >= 16384 else 64
        tile_n = 128 if n_ch >= 128 else 64
        p.algo_desp = _find(a.dtype, tv.float32, ShuffleStrideType.ShuffleAC, tile_m, tile_n, False, trans_b).copy()
        p.a, p.b, p.c = a, weight.select(1, k), acc
        p.a_inds = a_inds_all.select(0, k).slice_first_axis(0, cnt)
        p.c_inds = c_inds_all.select(0, k).slice_first_axis(0, cnt)
        p.alpha, p.beta = 1.0, 1.0
        p.stream = stream
        steps.append(p)
    return steps


def _finish(out, acc, bias, act_type, act_alpha, stream):
    _capi.check(_capi.lib().cumm_hip_finish_rows(
        out.byte_pointer(), out.dtype, acc.byte_pointer(), None if bias is None or bias.empty() else bias.byte_pointer(),
        out.dim(0), out.dim(1), 1.0, 1.0, act_type.value if hasattr(act_type, "value") else int(act_type),
        float(act_alpha), stream))


def _fp32_image(rows, channels, acc):
    if acc is None or acc.empty():
        acc = tv.empty([rows, channels], tv.float32, 0)
    elif acc.dtype != tv.float32 or acc.shape != [rows, channels] or acc.device < 0:
        raise RuntimeError("acc must be a device float32 tensor [%d, %d]" % (rows, channels))
    return acc


class _Plan:
    """The launches of one pass over fixed tensors and pair lists: built (and validated) once, run
    any number of times - a repeat run goes straight to the C entry points with the argument blocks
    of the first one.  The plan keeps its tensors alive."""

    def __init__(self, out, acc, steps, bias, act_type, act_alpha, stream):
        self.out, self.acc, self.steps = out, acc, steps
        self.bias, self.act_type, self.act_alpha, self.stream = bias, act_type, act_alpha, stream
        self._ctx = tv.Context()
        self._ctx.set_cuda_stream(stream)

    def __call__(self) -> None:
        self.acc.zero_(self._ctx)
        for p in self.steps:
            GemmMainUnitTest.matmul2(p)
        _finish(self.out, self.acc, self.bias, self.act_type, self.act_alpha, self.stream)

    @property
    def launches(self) -> int:
        return len(self.steps) + 2


def plan_forward(inp: tv.Tensor, weight: tv.Tensor, output: tv.Tensor, lists, *, bias: Optional[tv.Tensor] = None,
                 act_type=Activation.None_, act_alpha: float = 0.0, stream: int = 0,
                 acc: Optional[tv.Tensor] = None) -> _Plan:
    """The forward pass as a reusable plan (``plan()`` runs it): for a layer whose tensors and
    geometry stay in place from call to call."""
    _check(inp, weight, lists, output.dim(0))
    if output.ndim != 2 or output.dim(1) != weight.dim(0) or output.dtype != inp.dtype or weight.dim(2) != inp.dim(1):
        raise RuntimeError("error")
    acc = _fp32_image(output.dim(0), output.dim(1), acc)
    # W[:, k, :] is [K, C]: B stored [n, k]
    steps = _accumulate_steps(inp, lists.pair_in, lists.pair_out, lists.counts, weight, acc, True, stream)
    return _Plan(output, acc, steps, bias, act_type, act_alpha, stream)


def plan_backward_input(dout: tv.Tensor, weight: tv.Tensor, dinp: tv.Tensor, lists, *, stream: int = 0,
                        acc: Optional[tv.Tensor] = None) -> _Plan:
    _check(dout, weight, lists, dinp.dim(0))
    if dinp.ndim != 2 or dinp.dim(1) != weight.dim(2) or dout.dim(1) != weight.dim(0) or dinp.dtype != dout.dtype:
        raise RuntimeError("error")
    acc = _fp32_image(dinp.dim(0), dinp.dim(1), acc)
    # W[:, k, :] is [K, C] with K the contraction: B stored [k, n]
    steps = _accumulate_steps(dout, lists.pair_out, lists.pair_in, lists.counts, weight, acc, False, stream)
    return _Plan(dinp, acc, steps, None, Activation.None_, 0.0, stream)


def forward(inp: tv.Tensor, weight: tv.Tensor, output: tv.Tensor, lists, *, bias: Optional[tv.Tensor] = None,
            act_type=Activation.None_, act_alpha: float = 0.0, stream: int = 0, acc: Optional[tv.Tensor] = None) -> None:
    """output [N_out, K] = act(sum over offsets + bias); ``lists`` from ``pairs.pair_lists_device``
    on the forward table; ``acc``: an fp32 [N_out, K] device tensor to reuse as the image."""
    plan_forward(inp, weight, output, lists, bias=bias, act_type=act_type, act_alpha=act_alpha, stream=stream,
                 acc=acc)()


def backward_input(dout: tv.Tensor, weight: tv.Tensor, dinp: tv.Tensor, lists, *, stream: int = 0,
                   acc: Optional[tv.Tensor] = None) -> None:
    """dinp [N_in, C] = sum over offsets of dout[pair_out[k]] @ W[:, k, :] scattered to pair_in[k]."""
    plan_backward_input(dout, weight, dinp, lists, stream=stream, acc=acc)()


class WeightPlan:
    """Backward-weight of all kernel offsets in one call of the library (``cumm_hip_wgrad_pairs``),
    validated once: run on the tensors it was made for, or through ``rebind`` on others of the same
    shapes and types by address.

    A run that is recorded into a graph does without a workspace of the plan's own - nothing may be
    allocated then, and the graph may outlive the plan, whose workspace other calls get afterwards -
    and makes one product per offset instead."""

    def __init__(self, dout, inp, dweight, lists, stream):
        self._tensors, self._lists, self._stream = (dout, inp, dweight), lists, stream
        self._slots, self._forms = None, _forms(dout, inp, dweight)
        lib = _capi.lib()
        kv, k_out, c_in = dweight.dim(1), dweight.dim(0), dweight.dim(2)
        self._fn = lib.cumm_hip_wgrad_pairs
        self._counts = _counts(lists)
        counts = self._counts.ctypes.data
        self._pairs = (lists.pair_out.byte_pointer(), lists.pair_in.byte_pointer(), counts, kv, lists.pair_in.dim(1))
        self._sizes = (dout.dim(0), inp.dim(0), k_out, c_in, dweight.dtype)
        #: bytes of workspace that a run needs
        self.workspace_bytes = _wgrad_workspace(self._counts, dweight)
        if self.workspace_bytes < 0:
            raise RuntimeError("at most 128 kernel offsets, channel counts multiples of 8")

    def __call__(self) -> None:
        if self._tensors is None:
            raise RuntimeError("the plan has released its tensors: use rebind")
        dout, inp, dweight = self._tensors
        self.rebind(dout.byte_pointer(), inp.byte_pointer(), dweight.byte_pointer(), self._stream)

    def rebind(self, dout_ptr: int, inp_ptr: int, dweight_ptr: int, stream: int, workspace_ptr: Optional[int] = None) -> None:
        """Run on other tensors of the same shapes (device addresses), on ``stream``.  Without a
        workspace (``workspace_bytes`` bytes) the plan's own is used: one run at a time then."""
        if workspace_ptr is None:
            if _capi.lib().cumm_hip_stream_is_capturing(stream):
                WeightSteps(*_views(self._forms, dout_ptr, inp_ptr, dweight_ptr), self._lists, stream)()
                return
            slots = self._slots
            if slots is None or slots.stream != stream:
                slots = self._slots = _Slots(_Slots._device(), stream, max(self.workspace_bytes, 16), id(self))
            workspace_ptr = slots.tensor.byte_pointer()
        status = self._fn(dweight_ptr, dout_ptr, inp_ptr, *self._pairs, *self._sizes, workspace_ptr, self.workspace_bytes, stream)
        if status:
            _capi.check(status)

    def release(self) -> None:
        """Forget the tensors of the first run (a caller that goes on through ``rebind`` with its own);
        the pair lists stay."""
        self._tensors = None

    @property
    def launches(self) -> int:
        """Products the plan makes: one per kernel offset (they share the launches of one call)."""
        return self._pairs[3]


def _forms(*tensors):
    """What a tensor is beside its address."""
    return [(list(t.shape), list(t.stride), t.dtype, t.device) for t in tensors]


def _views(forms, *addresses):
    return [tv.from_blob_strided(at, *form) for at, form in zip(addresses, forms)]


def plan_backward_weight(dout: tv.Tensor, inp: tv.Tensor, dweight: tv.Tensor, lists, *, stream: int = 0):
    """Backward-weight as a reusable plan: dweight[:, k, :] of every kernel offset (zeros for an
    offset without pairs)."""
    _check(inp, dweight, lists, dout.dim(0))
    if dout.ndim != 2 or dout.dim(1) != dweight.dim(0) or dout.dtype != inp.dtype or dweight.dim(2) != inp.dim(1):
        raise RuntimeError("error")
    _check_device(dout, inp, dweight, lists.pair_in, lists.pair_out)
    _check_dtype(lists.pair_in, tv.int32, "pair_in")
    _check_dtype(lists.pair_out, tv.int32, "pair_out")
    if not _in_one_call(dout, inp, dweight, lists):
        return WeightSteps(dout, inp, dweight, lists, stream)
    if (np.asarray(lists.counts) <= 0).any() and not _capi.lib().cumm_hip_stream_is_capturing(stream):
        WeightSteps.no_pair(inp.device)      # (for runs that are recorded)
    return WeightPlan(dout, inp, dweight, lists, stream)


def _in_one_call(dout, inp, dweight, lists) -> bool:
    """What ``cumm_hip_wgrad_pairs`` takes: whole tensors at 16-byte addresses, up to 128 offsets - and lists
    and channels below its limits (-1 for those above), which single products do not have."""
    return (all(t.is_contiguous() and t.byte_pointer() % 16 == 0 for t in (dout, inp, dweight)) and
            lists.pair_in.is_contiguous() and lists.pair_out.is_contiguous() and lists.pair_in.shape == lists.pair_out.shape and
            dweight.dim(1) <= 128 and _wgrad_workspace(_counts(lists), dweight) >= 0)


def _counts(lists) -> np.ndarray:
    """(A count beyond its list ends with the list, as a slice of it does.)"""
    return np.ascontiguousarray(np.clip(lists.counts, 0, lists.pair_in.dim(1)), np.int32)


def _wgrad_workspace(counts: np.ndarray, dweight) -> int:
    return int(_capi.lib().cumm_hip_wgrad_pairs_workspace(counts.ctypes.data, dweight.dim(1), dweight.dim(0), dweight.dim(2)))


class WeightSteps:
    """Backward-weight as one gathered product per kernel offset: rows with a stride of their own, more
    offsets than one call takes, runs that are recorded into a graph.  The first run validates each
    product; runs after it, and ``rebind`` on other tensors of the same shapes, go straight to the C entry
    points.  The products run one after the other on one stream and share a workspace."""

    _NO_PAIR = {}

    @classmethod
    def no_pair(cls, dev: int) -> tv.Tensor:
        """The pairs of an offset without any: absent rows, whose product is zero."""
        if dev not in cls._NO_PAIR:
            cls._NO_PAIR[dev] = tv.from_numpy(np.full(32, -1, np.int32)).cuda()
        return cls._NO_PAIR[dev]

    def __init__(self, dout, inp, dweight, lists, stream):
        self.steps, self._tensors, self._lists, self._stream = [], (dout, inp, dweight), lists, stream
        self._forms, self._launches, self._ran = _forms(dout, inp, dweight), dweight.dim(1), False
        self._blocks, self._slots, self._lock = None, None, threading.Lock()
        self._workspace_bytes = 0
        for k in range(dweight.dim(1)):
            cnt = min(int(lists.counts[k]), lists.pair_in.dim(1))
            p = GemmParams()
            p.algo_desp = _find(inp.dtype, inp.dtype, ShuffleStrideType.ShuffleAB, 64, 64, True, False).copy()
            p.a, p.b, p.c = dout, inp, dweight.select(1, k)
            if cnt > 0:
                p.a_inds = lists.pair_out.select(0, k).slice_first_axis(0, cnt)
                p.b_inds = lists.pair_in.select(0, k).slice_first_axis(0, cnt)
            else:      # one step of absent rows writes the zeros
                p.a_inds = p.b_inds = self.no_pair(inp.device)
            p.stream = stream
            self._workspace_bytes = max(self._workspace_bytes, self._optional(p))
            self.steps.append(p)

    @staticmethod
    def _optional(p) -> int:
        return int(_capi.lib().cumm_hip_query_gemm_optional_workspace(
            ctypes.byref(desp_to_c(p.algo_desp)), p.a.dim(1), p.b.dim(1), p.a_inds.dim(0)))

    def split(self, slices: int, workspace: Optional[tv.Tensor]) -> None:
        """Cut the products that are not spread over the device in any case into ``slices`` where they have
        pairs enough."""
        for p in self.steps:
            if self._optional(p) <= 0 and p.a_inds.dim(0) >= 4096 * slices:
                p.split_k_slices = slices
            if workspace is not None:
                p.workspace = workspace

    def _share(self, stream: int) -> None:
        # (the products of a recorded run use none)
        if (self._workspace_bytes > 0 and (self._slots is None or self._slots.stream != stream) and
                not _capi.lib().cumm_hip_stream_is_capturing(stream)):
            self._slots = _Slots(_Slots._device(), stream, self._workspace_bytes, None)

    def __call__(self) -> None:
        if self._tensors is None:
            raise RuntimeError("the plan has released its tensors: use rebind")
        with self._lock:      # (a product's two launches and the next one's use the same workspace)
            if self._blocks is not None:
                self._run(*(t.byte_pointer() for t in self._tensors), self._stream)
                return
            self._share(self._stream)
            for p in self.steps:
                p.__dict__["_slots"] = self._slots
                GemmMainUnitTest.matmul2(p)
            self._ran = True
            blocks = []
            base = self._tensors[2].byte_pointer()
            for p in self.steps:
                prep = p.__dict__.get("_prepared")
                if prep is None:      # (recorded into a graph: validated again by the next run)
                    return
                args = prep[5]
                blocks.append((prep[1], prep[2], prep[3], args, args.ptr_C - base, bool(args.workspace) and args.split_k_slices == 1,
                               prep[4], prep[6]))
            self._blocks = blocks

    def _run(self, dout_ptr: int, inp_ptr: int, dweight_ptr: int, stream: int) -> None:
        self._share(stream)
        for fn, cdesc_ref, args_ref, args, delta, shares, _, _ in self._blocks:
            args.ptr_A, args.ptr_B = dout_ptr, inp_ptr
            args.ptr_C = args.ptr_D = dweight_ptr + delta
            if shares:
                args.workspace, args.workspace_bytes = self._slots.tensor.byte_pointer(), self._slots.tensor.nbytes
            status = fn(cdesc_ref, args_ref, stream)
            if status:
                _capi.check(status)

    def rebind(self, dout_ptr: int, inp_ptr: int, dweight_ptr: int, stream: int) -> None:
        """Run on other tensors of the same shapes and strides (device addresses), on ``stream``."""
        with self._lock:
            if not self._ran:
                raise RuntimeError("the plan has not run yet")
            if self._blocks is None:      # (recorded so far, which validates nothing for good)
                again = WeightSteps(*_views(self._forms, dout_ptr, inp_ptr, dweight_ptr), self._lists, stream)
                again()
                self._blocks, self._slots = again._blocks, again._slots
            else:
                self._run(dout_ptr, inp_ptr, dweight_ptr, stream)

    def release(self) -> None:
        """Forget the tensors of the first run (a caller that goes on through ``rebind`` with its own): the
        argument blocks hold addresses only, the pair lists belong to their owner."""
        if not self._ran:
            raise RuntimeError("the plan has not run yet")
        self.steps, self._tensors = [], None

    @property
    def launches(self) -> int:
        return self._launches


def backward_weight(dout: tv.Tensor, inp: tv.Tensor, dweight: tv.Tensor, lists, *, split_k_slices: int = 1,
                    stream: int = 0, workspace: Optional[tv.Tensor] = None) -> None:
    """dweight[:, k, :] = dout[pair_out[k]].T @ inp[pair_in[k]] for every offset (zero without pairs).
    ``split_k_slices`` is what a caller of the per-offset products would pass; the pairs are spread
    over the device in any case.  ``workspace`` is used when it is large enough."""
    plan = plan_backward_weight(dout, inp, dweight, lists, stream=stream)
    if isinstance(plan, WeightSteps):
        plan.split(split_k_slices, workspace)
        plan()
    elif (workspace is not None and not workspace.empty() and workspace.nbytes >= plan.workspace_bytes and
          workspace.byte_pointer() % 16 == 0):
        plan.rebind(dout.byte_pointer(), inp.byte_pointer(), dweight.byte_pointer(), stream, workspace.byte_pointer())
    else:
        plan()
