"""
Sequences of library calls recorded once per set of sizes and replayed by one call.

The forward of a layer is a fixed sequence of launches for given shapes, types and options; between calls only addresses
differ.  Made one by one from Python - a buffer and a foreign call each - the launches of a block of ordinary size cost the
host more than they cost the GPU.  :func:`call` runs a layer's own code on placeholders (:class:`_Place`: a shape, a
type and a place in a buffer), notes the calls it makes, and from then on makes them with ``mi8_run_plan``: one
buffer for everything temporary, one for what a backward takes, and the outputs.

Nothing of an input is kept: a plan belongs to sizes and options, holds no address and no tensor, and is the same for
every stream and thread.  Sizes are recorded when they are met for the third time (``_RECORD_AT``): those that never come back
cost a lookup, unless three or more layers of a model have them.  us of a call among others, call by call / replayed: feed-forward block of 1999 tokens, 1024 / 2816, forward
and backward 391 / 194 (the GPU 182); four attention projections of 1537 tokens x 2048 535 / 306; generation of 23 tokens at
4096 / 11008 69 / 55, of one token at 768 / 2048 40 / 27; 64 experts of 2048 x 1024, 48 tokens x top-8 92 / 70.
"""

from __future__ import annotations

import ctypes
import logging
import operator
import types
from typing import Callable, Optional, Sequence

import torch

from .. import _C
from . import ops

_log = logging.getLogger(__name__)

_OFFSET = (1 << 48) - 1
_STREAM, _IGNORED = -1, -2
_ALIGN = 256

# Sizes above which a sequence is not planned: its launches are long enough, and a buffer for all temporaries holds more than
# they do one by one.  Forward and backward of a block, MiB of the two plans, us call by call / replayed, peak MiB: 67 + 57 418 / 202,
# 68 / 78; 121 + 99 419 / 273, 130 / 150; 221 + 178 464 / 468, 260 / 286; 322 + 233 652 / 650, 404 / 399; 385 + 417 (float32 weights)
# 805 / 802 (on other boxes 771 / 759, 786 / 777), 378 / 444; 434 + 313 837 / 834, 532 / 542; 463 + 420 1008 / 1010, 365 / 408; 520 + 426
# 1055 / 1056, 539 / 626.  Of three projections 154 + 155 484 / 432, 220 / 223; 283 + 286 842 / 840, 460 / 434; 357 + 358 1127 / 1128.
_MOST_BYTES = 448 << 20
_MOST_PLANS, _MOST_SEEN = 512, 4096

# The time a set of sizes is met at which it is recorded.  Recording against what each later call saves, us: forward and
# backward of a block of 1999 tokens, 1024 / 2816, 586 against 200; a linear of 100 tokens, 1024 x 1024, 103 against 19; a block
# generating 23 tokens, 4096 / 11008, 163 against 28, one token, 768 / 2048, 90 against 8.  It pays after 3 to 11 more calls, so not
# for sizes that two layers meet once in a forward of their own.
_RECORD_AT = 3

_QUERIES = {
    "mi8_gemm_splitk_suggest", "mi8_gemm_splitk_workspace_bytes", "mi8_gemm_fp8_batch_pays", "mi8_amax_slots_for",
    "mi8_colamax_workspace_slots", "mi8_two_cast_workspace_words", "mi8_gemm_fp8_swiglu_matches_separate", "mi8_gemm_fp8_swiglu_pays",
    "mi8_gemm_fp8_codes_supported", "mi8_rowseg_code_count", "mi8_swiglu_amax_state_words", "mi8_gemm_fp8_swiglu_slots",
}


class Unplannable(Exception):
    """The recorded code did something other than calls of the library on its buffers."""


class _Device:
    """Stands where a placeholder's device is asked for; :func:`ops._empty` takes places from it."""

    __slots__ = ("index", "recorder")
    type = "cuda"

    def __init__(self, index: int, recorder: "_Recorder"):
        self.index, self.recorder = index, recorder

    def place(self, shape, dtype) -> "_Place":
        return self.recorder.place(shape, dtype)


class _Place:
    """What a recorded function sees of a contiguous GPU tensor."""

    __slots__ = ("device", "dtype", "shape", "address")
    is_cuda, requires_grad, is_meta = True, False, False

    def __init__(self, device: _Device, shape, dtype: torch.dtype, address: int):
        self.device, self.dtype, self.address = device, dtype, address
        self.shape = (int(shape),) if isinstance(shape, int) else tuple(shape)

    def data_ptr(self) -> int:
        return self.address

    def dim(self) -> int:
        return len(self.shape)

    def numel(self) -> int:
        n = 1
        for s in self.shape:
            n *= s
        return n

    def stride(self, d: int) -> int:
        n = 1
        for s in self.shape[d + 1 if d >= 0 else len(self.shape) + d + 1:]:
            n *= s
        return n

    def is_contiguous(self) -> bool:
        return True

    def contiguous(self) -> "_Place":
        return self

    def is_inference(self) -> bool:  # (no version counter to move)
        return True

    def to(self, *args, **kwargs) -> "_Place":
        if kwargs or len(args) != 1 or args[0] != self.dtype:
            raise Unplannable("a conversion")
        return self

    def __getattr__(self, name: str):
        raise Unplannable(f"tensor.{name}")

    def reshape(self, *shape) -> "_Place":
        out = _Place(self.device, shape[0] if len(shape) == 1 and not isinstance(shape[0], int) else shape, self.dtype, self.address)
        if out.numel() != self.numel():
            raise Unplannable("a reshape")
        return out

    def new_empty(self, shape) -> "_Place":
        return self.device.place(shape, self.dtype)

    def __getitem__(self, i) -> "_Place":
        if not isinstance(i, slice) or i.step not in (None, 1) or len(self.shape) != 1 or not i.stop:
            raise Unplannable("an index")
        start = i.start or 0
        return _Place(self.device, i.stop - start, self.dtype, self.address + start * self.dtype.itemsize)


class _Recorder:
    """Stands in for the library: notes calls that enqueue work, answers questions about sizes."""

    def __init__(self, index: int, n_inputs: int):
        self.device = _Device(index, self)
        self.real = _C.lib()
        self.words: list = []
        self.addresses: list = []  # positions of addresses in words, and the number of their call
        self.calls = 0
        self.sizes: list = []      # bytes of the places, numbered after the inputs
        self.n_inputs = n_inputs

    def place(self, shape, dtype) -> _Place:
        p = _Place(self.device, shape, dtype, (self.n_inputs + len(self.sizes) + 1) << 48)
        self.sizes.append(p.numel() * dtype.itemsize)
        return p

    def __getattr__(self, name: str):
        fn = getattr(self.real, name)
        if name in _QUERIES:
            return fn
        number = self.real.mi8_plan_function(name.encode())
        if number < 0:
            raise Unplannable(name)
        return lambda *args: self._note(name, number, fn.argtypes, args)

    def _word(self, value, kind) -> None:
        if kind is ctypes.c_void_p:
            value = int(value or 0)
            if value:
                self.addresses.append((len(self.words), self.calls))
        self.words.append(int(value))

    def _note(self, name: str, number: int, kinds, args) -> int:
        if len(args) != len(kinds):
            raise Unplannable(name)
        self.words.append(number)
        for kind, a in zip(kinds[:-1], args):
            item = getattr(kind, "_type_", None)
            if item is ctypes.c_int32 and kind is not ctypes.c_int32:
                a.value = self._slots(name, args)
                self.words.append(_IGNORED)
            elif isinstance(item, type) and issubclass(item, ctypes.Structure):
                self.words.append(len(a))
                for it in a:
                    for field, fkind in item._fields_:
                        self._word(getattr(it, field), fkind)
            else:
                self._word(a, kind)
        self.words.append(_STREAM)
        self.calls += 1
        return 0

    def _slots(self, name: str, args) -> int:
        if name == "mi8_amax_partials":
            return self.real.mi8_amax_slots_for(args[2])
        if name == "mi8_few_rows_swiglu":
            return self.real.mi8_few_rows_swiglu_slots(*args[7:10], args[1])
        if name == "mi8_gemm_fp8_swiglu":
            return self.real.mi8_gemm_fp8_swiglu_slots(*args[7:10])
        raise Unplannable(name)


def _places(tree):
    if isinstance(tree, _Place):
        yield tree
    elif isinstance(tree, (tuple, list)):
        for t in tree:
            yield from _places(t)


def _pack(temporaries: dict):
    """``(offsets, bytes)`` of temporaries ``{name: (bytes, first call, last call)}`` in one buffer.  Two that no call has in common
    may share bytes, as they do where the allocator is given each back after its last use (the calls of a plan follow one
    another on one stream).  The largest first, each at the lowest offset that is free.

    Bytes are shared where that saves a quarter of them, else every temporary has its own, which is up to 1 % faster.  us of
    forward and backward, shared / of their own, MiB of the backward's temporaries: block of 4096 tokens, 2048 / 8192, float32 weights
    766 / 759, 192 / 209, bfloat16 707 / 701; of 6000 tokens, 1024 / 2816 353 / 351, 12000 623 / 625, 194 / 350; three projections of
    8192 x 2048 410 / 413, 16384 x 2048 807 / 811, 192 / 288."""
    rounded = {name: (size + _ALIGN - 1) // _ALIGN * _ALIGN for name, (size, _, _) in temporaries.items()}
    live: dict = {}
    for name, (_, first, last) in temporaries.items():
        for c in range(first, last + 1):
            live[c] = live.get(c, 0) + rounded[name]
    offsets, end, placed = {}, 0, []
    if 4 * max(live.values(), default=0) > 3 * sum(rounded.values()):
        for name, size in rounded.items():
            offsets[name], end = end, end + size
        return offsets, end
    for name, size in sorted(rounded.items(), key=lambda t: -t[1]):
        _, first, last = temporaries[name]
        at = 0
        for lo, hi in sorted((lo, hi) for lo, hi, f, l in placed if f <= last and first <= l):
            if lo - at >= size:
                break
            at = max(at, hi)
        offsets[name] = at
        placed.append((at, at + size, first, last))
        end = max(end, at + size)
    return offsets, end


class Plan:
    """A recorded sequence.  Buffers in order: the inputs, the temporaries, what is kept for a backward, the outputs."""

    def __init__(self, fn: Callable, specs: Sequence, index: int):
        n = len(specs)
        rec = _Recorder(index, n)
        inputs = [None if s is None else _Place(rec.device, s[0], s[1], (i + 1) << 48) for i, s in enumerate(specs)]
        _C._recording.recorder = rec
        try:
            outs, saved = fn(*inputs)
        finally:
            _C._recording.recorder = None
        where = {}  # place number -> (buffer, offset)
        self.outs = []
        for k, o in enumerate(outs):
            number = (o.address >> 48) - 1
            if number < n or o.address & _OFFSET or number in where:
                raise Unplannable("an output that is no buffer of its own")
            where[number] = (n + 2 + k, 0)
            self.outs.append((o.shape, o.dtype))
        self.kept = 0
        for p in _places(saved):
            self._keep(where, (p.address >> 48) - 1, n, rec.sizes)
        words = list(rec.words)
        calls: dict = {number: [] for number in range(n, n + len(rec.sizes)) if number not in where}  # of the temporaries
        for at, number_of_call in rec.addresses:
            calls.get((words[at] >> 48) - 1, []).append(number_of_call)
        offsets, self.temporary = _pack({number: (rec.sizes[number - n], c[0] if c else -1, c[-1] if c else -1) for number, c in calls.items()})
        if self.temporary + self.kept + sum(rec.sizes[k - n] for k, (b, _) in where.items() if b >= n + 2) > _MOST_BYTES:
            raise Unplannable("more than _MOST_BYTES")
        where.update((number, (n, at)) for number, at in offsets.items())
        for at, _ in rec.addresses:
            number = (words[at] >> 48) - 1
            if number >= n:
                b, off = where[number]
                words[at] = (b + 1) << 48 | (off + (words[at] & _OFFSET))
        self.n_inputs, self.n_words = n, len(words)
        self.words = (ctypes.c_int64 * len(words))(*words)
        self.n_buffers = n + 2 + len(self.outs)
        self._buffers = ctypes.c_void_p * self.n_buffers
        self._saved = self._rebase(saved, where)
        self.then: dict = {}  # plans of the backward, which depend on where this one keeps what it keeps
        self.used = False  # replayed since its table was last full

    def _keep(self, where, number, n, sizes) -> None:
        if number < n:
            raise Unplannable("an input is kept")
        if number not in where:
            where[number] = (n + 1, self.kept)
            self.kept += (sizes[number - n] + _ALIGN - 1) // _ALIGN * _ALIGN
        elif where[number][0] != n + 1:
            raise Unplannable("an output is kept")

    def _rebase(self, tree, where):
        if isinstance(tree, _Place):
            return (tree.shape, tree.dtype, where[(tree.address >> 48) - 1][1] + (tree.address & _OFFSET))
        if isinstance(tree, (tuple, list)):
            return [self._rebase(t, where) for t in tree]
        return tree

    def saved_places(self, slab: _Place):
        """What the recorded function returned to be kept, as places in ``slab``."""

        def build(tree):
            if isinstance(tree, tuple):
                return _Place(slab.device, tree[0], tree[1], slab.address + tree[2])
            return [build(t) for t in tree] if isinstance(tree, list) else tree

        return build(self._saved)

    def saved_tensors(self, kept: Optional[torch.Tensor]):
        """The same as tensors in the buffer ``kept``."""

        def build(tree):
            if isinstance(tree, tuple):
                shape, dtype, at = tree
                n = dtype.itemsize
                for d in shape:
                    n *= d
                return kept[at:at + n].view(dtype).view(shape)
            return [build(t) for t in tree] if isinstance(tree, list) else tree

        return build(self._saved)

    def run(self, inputs):
        """``(outputs, kept)``: the outputs in order and the buffer of what is kept (or ``None``)."""
        buffers = self._buffers(*[None if t is None else t.data_ptr() for t in inputs])
        dev, n = inputs[0].device, self.n_inputs
        temporary = kept = None
        if self.temporary:
            temporary = torch.empty(self.temporary, dtype=torch.uint8, device=dev)
            buffers[n] = temporary.data_ptr()
        if self.kept:
            kept = torch.empty(self.kept, dtype=torch.uint8, device=dev)
            buffers[n + 1] = kept.data_ptr()
        outs = []
        for k, (shape, dtype) in enumerate(self.outs):
            o = torch.empty(shape, dtype=dtype, device=dev)
            buffers[n + 2 + k] = o.data_ptr()
            outs.append(o)
        status = _C.lib().mi8_run_plan(self.words, self.n_words, buffers, self.n_buffers, ops._stream(inputs[0]))
        if status:
            _C.check(status, "mi8_run_plan")
        return outs, kept


class _NoPlan:
    """Stands in the table for a sequence that cannot be recorded, with the reason."""

    used = False

    def __init__(self, reason: str):
        self.reason = reason


_plans: dict = {}
_seen: dict = {}

# The hooks that saved tensors go through on this thread (activation checkpointing, offloading), or None.
_saved_tensor_hooks = torch._C._autograd._top_saved_tensors_default_hooks


def _plannable(inputs) -> bool:
    for t in inputs:
        if t is not None and (type(t) not in (torch.Tensor, torch.nn.Parameter) or not t.is_contiguous() or t.data_ptr() % 16 or not t.is_cuda):
            return False
    return True


_OPS = ops.__dict__
_operations = operator.itemgetter(*(name for name, f in _OPS.items()
                                    if isinstance(f, types.FunctionType) and f.__module__ == ops.__name__ and name[0] != "_"))
_ORIGINALS = _operations(_OPS)


def _observed() -> bool:
    """Someone watches single launches (measurement hooks) or has put a function of theirs in the place of an operation of
    :mod:`ops`, any of which a recorded sequence may have called (0.9 us for the 43 of them)."""
    return ops.GEMM_EVENT_SINK is not None or ops.FORCE_SW_CVT or _operations(_OPS) != _ORIGINALS


def _remember(plans: dict, key: tuple, plan) -> None:
    """A full table gives up what was not replayed since it was last full, or else its older half: sizes that come back stay
    where others come once."""
    if len(plans) >= _MOST_PLANS:
        for k, p in list(plans.items()):
            if not p.used:
                plans.pop(k, None)
            p.used = False
        for k in list(plans)[:len(plans) - _MOST_PLANS // 2] if len(plans) >= _MOST_PLANS else ():
            plans.pop(k, None)
    plans[key] = plan


def call(fn: Callable, inputs: Sequence[Optional[torch.Tensor]], options: tuple, within: Optional[Plan] = None,
         own: int = 0):
    """``(outputs, kept, plan)`` of ``fn(*inputs)`` replayed from its plan, or ``None`` where it has none (yet): then the
    caller runs ``fn`` itself.  ``fn`` returns the tensors to be returned and a tree of those to be kept; what it does must
    follow from the shapes and types of ``inputs`` and from ``options`` (hashable, ``fn`` named in it) alone.  ``within``: the
    plan that this one continues.  ``own``: how many of the last inputs are this package's own tensors (contiguous, aligned).

    A forward under saved-tensor hooks has no plan: it would save one buffer where ``fn`` itself saves the tensors, and
    which of the two runs depends on how often the sizes were met.  Hooks see every saved tensor, and checkpointing refuses a
    re-run that saves other tensors than the first run did."""
    if (within is None and _saved_tensor_hooks(True) is not None) or _observed() or not _plannable(inputs[:-own] if own else inputs):
        return None
    index = inputs[0].get_device()
    key = [options, index]
    for t in inputs:
        if t is None:
            key.append(None)
        elif t.get_device() != index:
            return None  # (a plan launches on one GPU; the calls one by one refuse what they quantise together)
        else:
            key += (t.shape, t.dtype)
    key = tuple(key)
    plans = _plans if within is None else within.then
    plan = plans.get(key)
    if plan is None:
        if within is None:
            met = _seen.get(key, 0) + 1
            if met < _RECORD_AT:
                if len(_seen) >= _MOST_SEEN:
                    _seen.clear()
                _seen[key] = met
                return None
        try:
            plan = Plan(fn, [(tuple(t.shape), t.dtype) if t is not None else None for t in inputs], index)
        except Unplannable as e:
            plan = _NoPlan(str(e))
        except Exception as e:  # of a call that the caller's own run refuses as well, or of this file
            plan = _NoPlan(f"{type(e).__name__}: {e}")
            _log.warning("%s: not recorded, its calls are made one by one (%s)", options[0], plan.reason)
        _remember(plans, key, plan)
    else:
        plan.used = True
    if type(plan) is _NoPlan:
        return None
    return (*plan.run(inputs), plan)
