"""A minimal stand-in for flax.linen.Module: hyper-parameters are constructor
keyword arguments with class-level defaults, parameters live in a nested dict
``{'params': {...}}`` with the reference's names, ``init(seed, *inputs)``
creates them and ``apply(variables, *inputs)`` runs the module."""
from __future__ import annotations

from typing import Any, Dict

import weakref

import torch


class Module:
  _fields: Dict[str, Any] = {}

  def __init__(self, **kwargs):
    fields = {}
    for cls in reversed(type(self).__mro__):
      fields.update(getattr(cls, "_fields", {}))
    self.name = kwargs.pop("name", None)
    unknown = set(kwargs) - set(fields)
    if unknown:
      raise TypeError(f"{type(self).__name__} got unexpected arguments {sorted(unknown)}")
    missing = [k for k, v in fields.items() if v is _REQUIRED and k not in kwargs]
    if missing:
      raise TypeError(f"{type(self).__name__} missing required arguments {missing}")
    for k, v in fields.items():
      setattr(self, k, kwargs.get(k, v))

  def init(self, rng, *inputs):
    raise NotImplementedError

  def apply(self, variables, *inputs, **kwargs):
    raise NotImplementedError

  def __call__(self, variables, *inputs, **kwargs):
    return self.apply(variables, *inputs, **kwargs)


class _Required:
  def __repr__(self):
    return "<required>"


_REQUIRED = _Required()


def generator(rng, device="cpu") -> torch.Generator:
  if isinstance(rng, torch.Generator):
    return rng
  g = torch.Generator(device=device)
  g.manual_seed(int(rng))
  return g


def lecun_normal(gen: torch.Generator, shape, fan_in: int, dtype=torch.float32, device=None):
  """jax.nn.initializers.lecun_normal: truncated normal with variance 1/fan_in."""
  t = torch.empty(shape, dtype=torch.float32)
  torch.nn.init.trunc_normal_(t, mean=0.0, std=1.0, a=-2.0, b=2.0, generator=gen)
  t = t * (1.0 / 0.87962566103423978) / (fan_in ** 0.5)
  return t.to(dtype).to(device) if device is not None else t.to(dtype)


def require_no_grad(what: str, *tensors) -> None:
  """The gating, routing and expert kernels are forward-only (inference).  Called with
  the parameters and inputs of such a module: raises instead of silently cutting the
  graph when autograd is recording and one of them requires a gradient."""
  if not torch.is_grad_enabled():
    return
  for t in tensors:
    if isinstance(t, torch.Tensor) and t.requires_grad:
      raise NotImplementedError(
          f"{what} has no backward pass (inference path): call it under torch.no_grad() or "
          "detach its parameters and inputs.")


def is_plain(*tensors) -> bool:
  """Whether torch operations on these tensors may be replaced by a kernel that sees nothing but their memory:
  ordinary tensors on the GPU, no gradient recorded, and no transform, mode, trace or autocast at work."""
  if torch.is_grad_enabled() and any(t.requires_grad for t in tensors):
    return False
  return is_plain_but_for_gradients(*tensors)


def is_plain_but_for_gradients(*tensors) -> bool:
  """is_plain for an operation that autograd may record."""
  for t in tensors:
    if type(t) not in (torch.Tensor, torch.nn.Parameter) or not t.is_cuda:
      return False
  return not (torch._C._functorch.peek_interpreter_stack() is not None
              or torch.autograd.forward_ad._current_level >= 0 or torch._C._len_torch_dispatch_stack()
              or torch._C._len_torch_function_stack() or torch._C._get_tracing_state() is not None
              or torch.compiler.is_compiling() or torch.is_autocast_enabled())


def make_rngs(rngs, device):
  """``rngs={'gating': seed or torch.Generator}`` (flax's ``rngs=`` argument of apply)
  with every seed turned into a generator on ``device``, so that modules that draw
  one after the other get different numbers.  None stays None."""
  if rngs is None:
    return None
  out = {}
  for name, rng in rngs.items():
    out[name] = rng if isinstance(rng, torch.Generator) else generator(rng, device=device)
  return out


class ParamCache:
  """Derived copies of parameter tensors (casts, packed layouts).

  An entry is valid while the very tensors it was built from are alive and
  unmodified: they are identified by object (views by their base tensor, offset,
  shape and strides), held weakly, and their version counters, addresses and layouts
  are compared (``t.data = other`` changes those without a new version).  An
  address alone does not identify a tensor: the allocator hands a freed block
  to the next tensor of that size."""

  def __init__(self, limit: int = 16):
    self._entries = {}
    self._limit = limit
    self._latest = {}       # tag -> (weak references to the tensors, their states, to the entry) last asked for

  class _Entry:
    __slots__ = ("bases", "states", "value", "__weakref__")

  def get(self, tensors, tag, build):
    tensors = tuple(tensors)
    # The tensors of the last call with this tag, unmodified: what a layer that runs over and over
    # finds (0.7 us per tensor, twice that with the bases and keys below).  An address belongs to one device.
    latest = self._latest.get(tag)
    if latest is not None and len(latest[0]) == len(tensors):
      for t, ref, (version, address, shape, stride, dtype) in zip(tensors, latest[0], latest[1]):
        if (ref() is not t or t._version != version or t.data_ptr() != address or t.dtype is not dtype
            or t.shape != shape or t.stride() != stride):
          break
      else:
        entry = latest[2]()
        if entry is not None:
          return entry.value
    states = [(t._version, t.data_ptr(), t.shape, t.stride(), t.dtype) for t in tensors]
    bases = [t._base if t._base is not None else t for t in tensors]
    key = (tuple((id(b), t.storage_offset()) + s[2:] for b, t, s in zip(bases, tensors, states)), tag)
    entry = self._entries.get(key)
    if entry is None or entry.states != states or not all(r() is b for r, b in zip(entry.bases, bases)):
      entry = self._Entry()
      entry.bases, entry.states, entry.value = tuple(map(weakref.ref, bases)), states, build()
      if len(self._entries) >= self._limit:
        self._entries.clear()
      self._entries[key] = entry
    self._latest[tag] = (tuple(map(weakref.ref, tensors)), states, weakref.ref(entry))
    return entry.value
