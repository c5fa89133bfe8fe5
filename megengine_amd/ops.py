"""Host-side Python mirror of the two operators, over torch device tensors.

PyTorch is plumbing only here: it owns device memory and the stream.  All arithmetic happens in
the HIP kernels behind the C ABI; a missing library or a non-GPU tensor raises.

The calls mirror megdnn::ConvBiasForward (dnn/include/megdnn/oprs/nn.h:358-536):
    deduce_layout            -> conv_bias_deduce_layout(desc)
    get_workspace_in_bytes   -> conv_bias_workspace(desc, algo)
    get_algorithm_heuristic  -> conv_bias_query(desc)
    exec(src, filter, bias, z, dst, workspace) -> conv_bias_exec(...)
and megdnn::RelayoutFormat (dnn/include/megdnn/oprs/general.h:1348-1373); requant_exec is the unfused
epilogue (the reference's post-process pass; unary ElemwiseMultiType quantized modes and TypeCvt s32 -> s8).

The operators that launch on every call live in the extension module _native (csrc/native.cpp): through ctypes a call cost
the host more than twice its kernel launch.
"""
import ctypes as C

import torch

from . import _abi
from .lib import check, lib

try:
    from ._native import (conv_bias_bind, conv_bias_exec, conv_bias_exec_preprocessed, elemwise_q_exec, pooling_exec,
                          relayout_exec, requant_exec, typecvt_exec)
except ImportError as e:
    raise RuntimeError("the extension module megengine_amd._native is missing or stale: build it with "
                       "`python -m megengine_amd.build` (there is no fallback path)") from e


def _ptr(t):
    if t is None:
        return None
    if not t.is_cuda:
        raise RuntimeError("mi355 operators take GPU tensors only (got %s)" % t.device)
    if not t.is_contiguous():
        raise RuntimeError("tensor must be contiguous")
    return C.c_void_p(t.data_ptr())


def _stream():
    return C.c_void_p(torch._C._cuda_getCurrentRawStream(torch.cuda.current_device()))


def conv_bias_deduce_layout(desc):
    oh, ow = C.c_uint32(), C.c_uint32()
    check(lib().mi355_convbias_deduce_out(C.byref(desc), C.byref(oh), C.byref(ow)))
    return _abi.conv_shapes(desc)[3]


def conv_bias_query(desc, algo=_abi.ALGO_HEURISTIC):
    """-> (Algo, workspace_bytes)"""
    a = _abi.Algo()
    ws = C.c_size_t()
    check(lib().mi355_convbias_s8_query(C.byref(desc), algo, C.byref(a), C.byref(ws)))
    return a, ws.value


def conv_bias_workspace(desc, algo=_abi.ALGO_HEURISTIC):
    return conv_bias_query(desc, algo)[1]


def conv_bias_preprocess(desc, flt, algo):
    """exec_preprocess: the filter re-tiled for `algo` (a torch uint8 tensor), or None when the algorithm reads the
    reference layout only (deduce_preprocessed_filter_layout returns nothing for it)."""
    n = C.c_size_t()
    check(lib().mi355_convbias_s8_preprocess_size(C.byref(desc), C.byref(algo), C.byref(n)))
    if n.value == 0:
        return None
    out = torch.empty(n.value, dtype=torch.uint8, device=flt.device)
    check(lib().mi355_convbias_s8_preprocess(_stream(), C.byref(desc), C.byref(algo), _ptr(flt), _ptr(out), n.value))
    return out


def conv_bias_profile(desc, src, flt, bias, z, dst, algo, warmup=2, iters=10, workspace=None):
    """Average time in microseconds of one launch of `algo` (synchronises the current stream, overwrites dst)."""
    us = C.c_float()
    wsn = workspace.numel() if workspace is not None else 0
    check(lib().mi355_convbias_s8_profile(_stream(), C.byref(desc), C.byref(algo), _ptr(src), _ptr(flt), _ptr(bias),
                                         _ptr(z), _ptr(dst), _ptr(workspace), wsn, warmup, iters, C.byref(us)))
    return us.value


def relayout_desc(mode, shape, group=1, oc=0, elem_bytes=1, scale_src=1.0, scale_dst=1.0):
    d = _abi.RelayoutDesc(mode=mode, ndim=len(shape), group=group, oc=oc, elem_bytes=elem_bytes,
                          scale_src=scale_src, scale_dst=scale_dst)
    for i, s in enumerate(shape):
        d.shape[i] = s
    return d


def relayout_deduce_layout(d):
    nd = C.c_uint32()
    shp = (C.c_uint32 * 7)()
    check(lib().mi355_relayout_deduce(C.byref(d), C.byref(nd), shp))
    return tuple(shp[i] for i in range(nd.value))


def pooling_deduce_layout(d):
    """Output shape of megdnn::PoolingForward for the descriptor (dnn/src/common/pooling.cpp:7-125)."""
    oh, ow = C.c_uint32(), C.c_uint32()
    check(lib().mi355_pooling_deduce_out(C.byref(d), C.byref(oh), C.byref(ow)))
    return _abi.packed_shape(d.format, d.n, d.c, oh.value, ow.value)
