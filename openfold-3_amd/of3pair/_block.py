"""Whole blocks and stacks through one call of the C ABI (of3_pair_block_fwd, of3_pairformer_block_fwd,
of3_pairformer_stack_fwd).

A block issued module by module costs some 200 us of Python (parameter lookups, views, stream and device
queries for each of its seven modules) beside 50 us of launches, more than its kernels take below about 200
tokens.  Here the parameters are gathered in one sweep and the arguments are prepared once per block.

A block is served when it is built of this package's own modules as their constructors left them: anything a
caller may have changed (a replaced or subclassed submodule, a hook on one, a method replaced on one or on its class,
parameters of another dtype than the activations, layouts or widths that need a conversion) makes run_* return None,
and the block then runs module by module.
"""
from __future__ import annotations

import ctypes
import math
import operator
import weakref
from array import array as _array

import torch
from torch.nn.modules import module as _nn_module

from . import _lib, layers
from . import functional as F3

_scan = _lib.load_scan()

_TRI_MUL = ("linear_a_p", "linear_a_g", "linear_b_p", "linear_b_g")
_NORM = (torch.nn.LayerNorm,)
_MULS = {
    layers.TriangleMultiplicationOutgoing: True, layers.TriangleMultiplicationIncoming: False,
    layers.FusedTriangleMultiplicationOutgoing: True, layers.FusedTriangleMultiplicationIncoming: False,
}


class _Refused(Exception):
    """The block is not one that the single call serves."""


# Everything that a block run module by module calls by name: (class or module, name, what this package put there).
_written = []


def written(owner, *names):
    _written.extend((owner, name, getattr(owner, name)) for name in names)


def _as_written():
    """Whether a block's modules still do what the single call does in their place: no method replaced on a class (also
    nn.Module's own __call__, as tracers do), no function of this package replaced by a caller's."""
    for owner, name, value in _written:
        if getattr(owner, name, None) is not value:
            return False
    return True


written(torch.nn.Module, "__call__", "_call_impl", "__getattr__")
written(F3, "triangle_multiplicative_update", "triangle_attention", "swiglu_transition", "pair_bias", "attention_pair_bias")
written(layers.SwiGLUTransition, "__call__", "forward")
written(layers.AttentionPairBias, "__call__", "forward")
for _mul in _MULS:
    written(_mul, "_weights")
# what a pair block calls on itself
PAIR_METHODS = ("tri_mul_out_in", "tri_att_start_end", "_modules_forward", "_mul", "_att")
_CALL = ("forward", "_compiled_call_impl")


class _Params:
    """The parameters of a block in the order of the C ABI, looked up anew in every call: a parameter or a
    submodule that was replaced since, or moved by .to(), is seen.  What the search looks at is noted before it is
    judged, so that a block that was refused is searched again once that has changed."""

    def __init__(self):
        self.owners, self.names, self.held = [], [], []  # children or parameters of a module, name, what they held, or None
        self.refs = []     # (parameters of a module, name, number of values)
        self.shapes = []   # what refs must have; None where a parameter may be absent
        self.entries = []  # (index into refs, first row): the pointers handed over
        self.called = []   # submodules that the block calls as modules
        self.kinds = []    # (a module whose methods the block calls, its type)
        self.own = []      # (attributes of such a module, a name it may not have of its own)
        self.attrs = []    # (attributes of a module, name, the value that a call uses)
        self.noted = []    # the same of values that the search alone looks at
        self.last = (b"", None, None)  # pointers of refs, dtype and pointer array of the last call
        self.lists = None  # refs as _scan takes them

    def link(self, owner, name, held):
        self.owners.append(owner)
        self.names.append(name)
        self.held.append(held)

    def child(self, parent, name, kinds=None):
        children = parent._modules
        sub = children.get(name)
        self.link(children, name, sub)
        if sub is None or (kinds is not None and type(sub) not in kinds):
            raise _Refused
        return sub

    def attr(self, module, *names):
        for name in names:
            self.attrs.append((module.__dict__, name, getattr(module, name)))

    def note(self, module, *names):
        for name in names:
            self.noted.append((module.__dict__, name, getattr(module, name)))

    def no_own(self, module, names):
        attributes = module.__dict__
        for name in names:
            self.own.append((attributes, name))

    def uses(self, module, names):
        """Of a submodule.  Nothing here may hold the block itself: the plans are kept for as long as it lives."""
        self.kinds.append((module, type(module)))
        self.no_own(module, names)

    def calls(self, module):
        self.called.append(module)
        self.uses(module, _CALL)

    def sealed(self, dims):
        """The plan of a finished search; dims None: the block is refused, and the types of what was looked at count too (a
        module may change its own, as one under a parametrization does)."""
        if dims is None:
            self.attrs += self.noted
            self.kinds += [(held, type(held)) for held in self.held if held is not None]
        return self, dims

    def current(self):
        """Whether the block still holds the submodules and attributes that it held."""
        if any(map(operator.is_not, map(dict.get, self.owners, self.names), self.held)):
            return False
        for attributes, name, value in self.attrs:
            if attributes.get(name) != value:
                return False
        for m, kind in self.kinds:
            if type(m) is not kind:
                return False
        return True

    def param(self, module, name, shape, optional=False):
        if name not in module._parameters:
            self.link(module._parameters, name, None)
            raise _Refused
        self.entries.append((len(self.refs), 0))
        self.refs.append((module._parameters, name, math.prod(shape)))
        self.shapes.append((shape, optional))

    def norm(self, module, name, c, optional_bias=False):
        ln = self.child(module, name, _NORM)
        self.param(ln, "weight", (c,))
        self.param(ln, "bias", (c,), optional_bias)

    def linears(self, module, names, shape, bias=False):
        """Of several layers of one shape, written out: they are most of a block."""
        children, entries, refs, shapes = module._modules, self.entries, self.refs, self.shapes
        want, count = (shape, False), math.prod(shape)
        found = [children.get(name) for name in names]
        self.owners += [children] * len(found)
        self.names += names
        self.held += found
        for lin in found:
            if type(lin) is not torch.nn.Linear:
                raise _Refused
            own = lin._parameters
            if "weight" not in own:
                self.link(own, "weight", None)
                raise _Refused
            entries.append((len(refs), 0))
            refs.append((own, "weight", count))
            shapes.append(want)
            if bias:
                self.param(lin, "bias", shape[:1])

    def gather(self, dtype, device=None):
        """The pointer array, or None when a parameter is not a plain contiguous tensor of `dtype` on the GPU `device` (None: anywhere)."""
        seen, seen_dtype, array = self.last
        if self.lists is None:
            self.lists = ([ref[0] for ref in self.refs], [ref[1] for ref in self.refs], _array("q", [ref[2] for ref in self.refs]))
        gpu = -1 if device is None or device.index is None else device.index  # of activations on the host _pair_args has its say
        found = _scan(*self.lists, dtype, seen, gpu) if _scan is not None else None
        if found is None:
            found = self._scan_in_python(dtype, device)
        if found is False:
            return None
        if (found is not True and found != seen) or seen_dtype is not dtype:
            ptrs = _array("Q", seen if found is True else found)
            for (owner, name, _), (shape, optional) in zip(self.refs, self.shapes):
                p = owner.get(name)
                if not optional if p is None else p.shape != shape:
                    return None
            size = dtype.itemsize
            at = [ptrs[ref] + (row * self.shapes[ref][0][1] * size if row else 0) or None for ref, row in self.entries]
            array = (ctypes.c_void_p * len(at))(*at)
            self.last = (ptrs.tobytes(), dtype, array)
        return array

    def _scan_in_python(self, dtype, device):
        """What csrc/host_params.cpp does, for parameters of other types and where it is not built."""
        ptrs = _array("Q")
        for owner, name, count in self.refs:
            p = owner.get(name)
            if p is None:
                ptrs.append(0)
            elif p.numel() == count and p.dtype is dtype and p.is_contiguous() and (device is None or p.device == device):
                ptrs.append(p.data_ptr())
            else:
                return False
        return ptrs.tobytes()


def _pair_params(q, block):
    """Appends what of3_pair_block_fwd takes; returns (C, CH, H, D, HID, inf)."""
    q.no_own(block, PAIR_METHODS)
    mul_out, mul_in = q.child(block, "tri_mul_out", _MULS), q.child(block, "tri_mul_in", _MULS)
    c, ch = mul_out.c_z, mul_out.c_hidden
    for m, outgoing in ((mul_out, True), (mul_in, False)):
        q.attr(m, "c_z", "c_hidden", "_outgoing")
        if _MULS[type(m)] is not outgoing or m._outgoing is not outgoing or (m.c_z, m.c_hidden) != (c, ch):
            raise _Refused
        q.uses(m, ("_weights",))
        q.norm(m, "layer_norm_in", c)
        q.norm(m, "layer_norm_out", ch)
        if isinstance(m, layers.FusedTriangleMultiplicativeUpdate):
            # the a and b matrices are the two halves of each stacked weight: a_p, a_g, b_p, b_g
            n = len(q.refs)
            for name in ("linear_ab_p", "linear_ab_g"):
                lin = q.child(m, name, (torch.nn.Linear,))
                q.param(lin, "weight", (2 * ch, c))
            q.entries[-2:] = [(n, 0), (n + 1, 0), (n, ch), (n + 1, ch)]
        else:
            q.linears(m, _TRI_MUL, (ch, c))
        q.linears(m, ("linear_g",), (c, c))
        q.linears(m, ("linear_z",), (c, ch))
    start, end = (q.child(block, n, (layers.TriangleAttention,)) for n in ("tri_att_start", "tri_att_end"))
    h, d, inf = start.no_heads, q.child(start, "mha", (layers._GatedAttentionParams,)).c_hidden, start.inf
    for m in (start, end):
        mha = q.child(m, "mha", (layers._GatedAttentionParams,))
        q.attr(m, "no_heads", "inf")
        q.note(m, "c_in")
        q.note(mha, "c_hidden")
        if (m.c_in, m.no_heads, mha.c_hidden, m.inf) != (c, h, d, inf):
            raise _Refused
        q.norm(m, "layer_norm", c)
        q.linears(m, ("linear_z",), (h, c))
        q.linears(mha, ("linear_q", "linear_k", "linear_v", "linear_g"), (h * d, c))
        q.linears(mha, ("linear_o",), (c, h * d))
    hid = 0
    if "pair_transition" in block._modules:
        hid = _transition_params(q, block, "pair_transition", c)
    return c, ch, h, d, hid, inf


def _transition_params(q, block, name, c):
    t = q.child(block, name, (layers.SwiGLUTransition,))
    q.calls(t)
    q.note(t, "n")
    hid = t.n * c
    q.norm(t, "layer_norm", c)
    sw = q.child(t, "swiglu", (layers._SwiGLUParams,))
    q.linears(sw, ("linear_a", "linear_b"), (hid, c))
    q.linears(t, ("linear_out",), (c, hid))
    return hid


def _pairformer_params(q, block, pair_block_type):
    pair = q.child(block, "pair_stack", (pair_block_type,))
    q.calls(pair)
    dims = _pair_params(q, pair)
    a = q.child(block, "attn_pair_bias", (layers.AttentionPairBias,))
    q.calls(a)
    mha = q.child(a, "mha", (layers._PairBiasAttentionParams,))
    q.attr(a, "no_heads", "inf")
    q.note(a, "c_q", "c_z")
    c_s, c_z, h = a.c_q, dims[0], a.no_heads
    lin = q.child(mha, "linear_q", (torch.nn.Linear,))
    weight = lin._parameters.get("weight")
    if weight is None or a.c_z != c_z or h < 1 or weight.shape[0] % h:
        q.link(lin._parameters, "weight", weight)
        raise _Refused
    hd = weight.shape[0]
    q.norm(a, "layer_norm_z", c_z, optional_bias=True)
    q.linears(a, ("linear_z",), (h, c_z))
    q.norm(a, "layer_norm_a", c_s)
    q.linears(mha, ("linear_q",), (hd, c_s), bias=True)
    q.linears(mha, ("linear_k", "linear_v", "linear_g"), (hd, c_s))
    q.linears(mha, ("linear_o",), (c_s, hd))
    hid_s = _transition_params(q, block, "single_transition", c_s)
    return dims, (c_s, h, hd // h, hid_s, a.inf)


# block -> (parameters, dimensions, or None where the block is not served), or None: called once
_plans = weakref.WeakKeyDictionary()
# Token count from which a block's first call goes module by module and the parameters are looked for in the second: the
# search takes 100 us or more before the first launch, and from here on issuing the modules keeps ahead of the GPU.
# First pass of new weights, us, searched first / module by module: two trunk blocks at N = 384 1530 / 1330, four updates at
# 768 2110 / 2020, one block at 929 4470 / 4260.
_LATE_FROM = 300


def _first_call(block, z):
    """Whether this is the block's first call and starts without the search for its parameters."""
    if z.dim() < 3 or z.shape[-2] < _LATE_FROM or block in _plans:
        return False
    _plans[block] = None
    return True


def _plan(block, build):
    plan = _plans.get(block)
    if plan is None or not plan[0].current():
        q = _Params()
        try:
            plan = q.sealed(build(q))
        except _Refused:
            plan = q.sealed(None)
        except (AttributeError, TypeError):  # not what the search expects of a module of its type: looked at again next time
            _plans[block] = None
            return q, None
        _plans[block] = plan
    return plan


def _gather(block, build, dtype, device=None):
    """(pointer array, dimensions) of the block's parameters, or None."""
    q, dims = _plan(block, build)
    if dims is None:
        return None
    array = q.gather(dtype, device)
    if array is None:
        return None
    for m in q.called:  # modules that the block would call: their hooks, their mode and a forward of their own are theirs
        if m.training or m._forward_hooks or m._forward_pre_hooks:
            return None
    for attributes, name in q.own:
        if name in attributes:
            return None
    if _nn_module._global_forward_hooks or _nn_module._global_forward_pre_hooks:
        return None
    return array, dims


def _pair_args(z, mask):
    """(z as [B, N, N, C] without a copy, mask as fp32 [B, N, N] or None), or None."""
    if not z.is_cuda or z.dtype not in (torch.bfloat16, torch.float32) or z.dim() < 3:
        return None
    z4, lead = F3._flatten_pair(z)
    if z4.data_ptr() != z.data_ptr():  # a layout that is copied first
        return None
    return z4, F3._mask_arg(mask, lead, z4.shape[0], z4.shape[1], z.device)


def _call(fn, what, device, *args):
    if torch.cuda.current_device() == device.index:
        st = fn(*args)
    else:
        with torch.cuda.device(device):
            st = fn(*args)
    _lib.check(st, what)


def run_pair_block(block, z, mask, inplace, attention_first=False, mask_trans=True):
    """z after the block's modules, or None when the single call does not serve it."""
    if _first_call(block, z) or not _as_written():
        return None
    found = _gather(block, lambda q: _pair_params(q, block), z.dtype, z.device)
    args = found and _pair_args(z, mask)
    if not args:
        return None
    array, (c, ch, h, d, hid, inf) = found
    z4, (m, mptr, mstr) = args
    B, N, _, C = z4.shape
    if C != c:
        return None
    lib = _lib.load()
    code = _lib.OF3_DTYPE_BF16 if z.dtype is torch.bfloat16 else _lib.OF3_DTYPE_F32
    need = lib.of3_pair_block_workspace_bytes(code, B, N, C, ch, h, d, hid)
    if need < 0:
        return None
    out4 = z4 if inplace else F3._out_like(z4)
    stream = F3._stream(z)
    ws = F3._workspace(z.device, need, stream)
    flags = (_lib.OF3_BLOCK_ATTENTION_FIRST if attention_first else 0) | (0 if mask_trans else _lib.OF3_BLOCK_TRANSITION_UNMASKED)
    _call(lib.of3_pair_block_fwd, "of3_pair_block_fwd", z.device, array, z4.data_ptr(), _lib.strides3(z4.stride()[:3]),
          mptr, mstr, out4.data_ptr(), B, N, C, ch, h, d, hid, float(inf), flags, ws.data_ptr(), ws.numel(), code, stream)
    return z if inplace else out4.view(z.shape)


def _pairformer_args(s, z, single_mask, pair_mask, c, c_s):
    """The tensors of a block's or a stack's call: (z4, mask arguments, single mask as fp32), or None."""
    if s.device != z.device or s.dtype is not z.dtype or not s.is_contiguous() or not F3._is_single(s):
        return None
    args = _pair_args(z, pair_mask)
    if not args or s.shape[:-1] != z.shape[:-2] or args[0].shape[-1] != c or s.shape[-1] != c_s:
        return None
    sm = None
    if single_mask is not None:
        F3._require_device(single_mask, s.device, "single_mask")
        sm = single_mask.to(torch.float32).expand(s.shape[:-1]).contiguous()
    return args + (sm,)


def run_pairformer_block(block, pair_block_type, s, z, single_mask, pair_mask, inplace, mask_trans=True):
    """(s, z) after the block, or None when the single call does not serve it."""
    if _first_call(block, z) or not _as_written():
        return None
    found = _gather(block, lambda q: _pairformer_params(q, block, pair_block_type), z.dtype, z.device)
    if not found:
        return None
    array, ((c, ch, h, d, hid, inf), (c_s, h_s, d_s, hid_s, inf_s)) = found
    args = _pairformer_args(s, z, single_mask, pair_mask, c, c_s)
    if not args:
        return None
    z4, (m, mptr, mstr), sm = args
    B, N = z4.shape[:2]
    lib = _lib.load()
    code = _lib.OF3_DTYPE_BF16 if z.dtype is torch.bfloat16 else _lib.OF3_DTYPE_F32
    need = lib.of3_pairformer_block_workspace_bytes(code, B, N, c, ch, h, d, hid, c_s, h_s, d_s, hid_s)
    if need < 0:
        return None
    z_out = z4 if inplace else F3._out_like(z4)
    s_out = s if inplace else torch.empty_like(s)
    stream = F3._stream(z)
    ws = F3._workspace(z.device, need, stream)
    _call(lib.of3_pairformer_block_fwd, "of3_pairformer_block_fwd", z.device, array, s.data_ptr(), z4.data_ptr(),
          _lib.strides3(z4.stride()[:3]), None if sm is None else sm.data_ptr(), mptr, mstr, s_out.data_ptr(),
          z_out.data_ptr(), B, N, c, ch, h, d, hid, c_s, h_s, d_s, hid_s, float(inf), float(inf_s),
          0 if mask_trans else _lib.OF3_BLOCK_TRANSITION_UNMASKED, ws.data_ptr(), ws.numel(), code, stream)
    return s_out, z if inplace else z_out.view(z.shape)


def run_pairformer_stack(blocks, block_type, pair_block_type, s, z, single_mask, pair_mask, inplace, mask_trans=True):
    """(s, z) after all blocks, or None when the single call does not serve them."""
    if not _as_written():
        return None
    if any(_plans.get(block) is None for block in blocks):
        # First calls: finding the parameters takes some 100 us per block.  Block by block that passes beside the kernels of
        # the blocks before (4 blocks at N = 200: 1350 us in place of 1640).
        return None
    arrays, dims = [], None
    for block in blocks:
        if type(block) is not block_type or block.training or block._forward_hooks or block._forward_pre_hooks or any(name in block.__dict__ for name in _CALL):
            return None
        found = _gather(block, lambda q: _pairformer_params(q, block, pair_block_type), z.dtype, z.device)
        if not found or (dims is not None and found[1] != dims):
            return None
        arrays.append(found[0])
        dims = found[1]
    if not arrays:
        return None
    (c, ch, h, d, hid, inf), (c_s, h_s, d_s, hid_s, inf_s) = dims
    args = _pairformer_args(s, z, single_mask, pair_mask, c, c_s)
    if not args:
        return None
    z4, (m, mptr, mstr), sm = args
    B, N = z4.shape[:2]
    lib = _lib.load()
    code = _lib.OF3_DTYPE_BF16 if z.dtype is torch.bfloat16 else _lib.OF3_DTYPE_F32
    need = lib.of3_pairformer_stack_workspace_bytes(code, len(arrays), B, N, c, ch, h, d, hid, c_s, h_s, d_s, hid_s)
    if need < 0:
        return None
    table = (ctypes.POINTER(ctypes.c_void_p) * len(arrays))(*[ctypes.cast(a, ctypes.POINTER(ctypes.c_void_p)) for a in arrays])
    z_out = z4 if inplace else F3._out_like(z4)
    s_out = s if inplace else torch.empty_like(s)
    stream = F3._stream(z)
    ws = F3._workspace(z.device, need, stream)
    _call(lib.of3_pairformer_stack_fwd, "of3_pairformer_stack_fwd", z.device, table, len(arrays), s.data_ptr(), z4.data_ptr(),
          _lib.strides3(z4.stride()[:3]), None if sm is None else sm.data_ptr(), mptr, mstr, s_out.data_ptr(),
          z_out.data_ptr(), B, N, c, ch, h, d, hid, c_s, h_s, d_s, hid_s, float(inf), float(inf_s),
          0 if mask_trans else _lib.OF3_BLOCK_TRANSITION_UNMASKED, ws.data_ptr(), ws.numel(), code, stream,
          F3._side_stream(z.device, stream))
    return s_out, z if inplace else z_out.view(z.shape)
