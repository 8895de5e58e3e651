"""Host-side logic of the drop-in surface that needs no GPU: name resolution of routers
(vmoe/utils.py:59-109, vmoe/nn/vit_moe.py:76-88), capacity arithmetic, the public
factories, and the refusal to run forward-only kernels under autograd."""
import threading
import time
import weakref

import numpy as np
import pytest
import torch

from vmoe_amd import _hip, kernels, moe, utils
from vmoe_amd.nn import module, routing, vit_moe
from vmoe_amd.projects.soft_moe import router as soft_router


def test_parse_call_forms():
  fn, args, kwargs = utils.parse_call("NoisyTopExpertsPerItemRouter", default_module=routing)
  assert fn is routing.NoisyTopExpertsPerItemRouter and args == () and kwargs == {}
  fn, args, kwargs = utils.parse_call("vmoe_amd.projects.soft_moe.router.SoftRouter", routing)
  assert fn is soft_router.SoftRouter
  fn, args, kwargs = utils.parse_call("NoisyTopItemsPerExpertRouter(noise_std=0.5)", routing)
  assert fn is routing.NoisyTopItemsPerExpertRouter and kwargs == {"noise_std": 0.5}
  fn, args, kwargs = utils.parse_call("compute_capacity(128, 32, 2.0)", moe)
  assert fn(*args, **kwargs) == 8
  with pytest.raises(AttributeError):
    utils.parse_call("NoSuchRouter", routing)
  with pytest.raises(ValueError):
    utils.parse_call("f()()", routing)


@pytest.mark.parametrize("spec,cls", [
    ({}, routing.NoisyTopExpertsPerItemRouter),
    ({"name": "NoisyTopExpertsPerItemRouter"}, routing.NoisyTopExpertsPerItemRouter),
    ({"name": "NoisyTopItemsPerExpertRouter"}, routing.NoisyTopItemsPerExpertRouter),
    ({"name": "vmoe_amd.projects.soft_moe.router.SoftRouter", "num_slots": 2}, soft_router.SoftRouter),
])
def test_create_router_by_name(spec, cls):
  """vmoe/nn/vit_moe.py:76-88: `name` picks the class, `deterministic` is inherited from the
  block unless the router's own arguments set it, dtype and the module name are passed on."""
  block = vit_moe.MlpMoeBlock(mlp_dim=8, num_experts=4, group_size=16, deterministic=True,
                              router=spec, dtype=torch.bfloat16)
  router = block.create_router()
  assert type(router) is cls
  assert router.num_experts == 4 and router.deterministic is True
  assert router.dtype == torch.bfloat16 and router.name == "Router"
  override = vit_moe.MlpMoeBlock(mlp_dim=8, num_experts=4, group_size=16, deterministic=True,
                                 router=dict(spec, deterministic=False))
  assert override.create_router().deterministic is False


def test_create_split_rngs():
  """vmoe/nn/vit_moe.py:90-99."""
  mk = lambda v: vit_moe.MlpMoeBlock(mlp_dim=8, num_experts=4, group_size=16, split_rngs=v)
  assert mk(False).create_split_rngs() == {"params": False, "dropout": False}
  assert mk(True).create_split_rngs() == {"params": True, "dropout": True}
  assert mk(("dropout",)).create_split_rngs() == {"params": False, "dropout": True}


def test_compute_capacity_values(goldens):
  for case in goldens["compute_capacity"]["cases"]:
    case = dict(case)
    expected = case.pop("expected")
    assert moe.compute_capacity(**case) == expected
  with pytest.raises(ValueError, match="must be greater than or equal to 1"):
    moe.compute_capacity(128, 32, -1.0)
  # Python's round() rounds halves to even (vmoe/moe.py:240)
  assert moe.compute_capacity(20, 8, 1.0, ceil_or_round="round", multiple_of=1) == 2
  assert moe.compute_capacity(28, 8, 1.0, ceil_or_round="round", multiple_of=1) == 4


def test_get_dense_einsum_dispatcher():
  """vmoe/moe.py:260-264: the gates are the combine weights, keyword arguments pass through."""
  gates = torch.rand((2, 6, 3))
  d = moe.get_dense_einsum_dispatcher(gates, partition_spec=("a",))
  assert isinstance(d, moe.DenseEinsumDispatcher)
  assert d.combine_weights is gates and d.partition_spec == ("a",)


def test_forward_only_modules_refuse_autograd():
  """The gating, routing and expert kernels have no backward pass: with a parameter or an
  input that requires a gradient they raise instead of returning a result cut out of the
  graph.  (The check comes before any device call, so CPU tensors do here.)"""
  x = torch.zeros((2, 8, 16))
  w = torch.zeros((16, 4), requires_grad=True)
  for layer in (routing.NoisyTopExpertsPerItemRouter(num_experts=4, deterministic=True),
                routing.NoisyTopItemsPerExpertRouter(num_experts=4, deterministic=True,
                                                     dispatcher=dict(name="einsum", capacity=2))):
    with pytest.raises(NotImplementedError, match="no backward pass"):
      layer.apply({"params": {"dense": {"kernel": w}}}, x)
  soft = soft_router.SoftRouter(num_experts=4, num_slots=1)
  mu = torch.zeros((16, 4, 1), requires_grad=True)
  with pytest.raises(NotImplementedError, match="no backward pass"):
    soft.apply({"params": {"mu": mu, "scale": torch.ones(())}}, x)
  mlp = vit_moe.MlpBlock(mlp_dim=8)
  params = {"Dense_0": {"kernel": torch.zeros((1, 16, 8), requires_grad=True), "bias": torch.zeros((1, 8))},
            "Dense_1": {"kernel": torch.zeros((1, 8, 16)), "bias": torch.zeros((1, 16))}}
  with pytest.raises(NotImplementedError, match="no backward pass"):
    mlp.apply_experts({"params": params}, torch.zeros((1, 4, 16)))
  with pytest.raises(NotImplementedError, match="no backward pass"):
    mlp.apply_experts_gathered({"params": params}, torch.zeros((4, 16)),
                               torch.zeros((1, 4), dtype=torch.int32),
                               torch.zeros((1,), dtype=torch.int32))
  # without autograd recording the same calls reach the device layer (and fail there on CPU tensors)
  with torch.no_grad():
    with pytest.raises(Exception) as info:
      mlp.apply_experts({"params": params}, torch.zeros((1, 4, 16)))
    assert not isinstance(info.value, NotImplementedError)


@pytest.mark.parametrize("other", [
    lambda t: torch.full((2, 3), 5.0),                       # same shape
    lambda t: torch.full((4, 5), 5.0),
    lambda t: t.data.to(torch.bfloat16),
    lambda t: t.data.t(),                                    # same address, other strides
    lambda t: t.data.view(3, 2),
], ids=["same-shape", "shape", "dtype", "transposed", "reshaped"])
def test_param_cache_sees_data_assignment(other):
  """``p.data = other`` raises no version counter: the address and the layout tell."""
  p = torch.nn.Parameter(torch.arange(6.0).view(2, 3))
  cache = module.ParamCache()
  derive = lambda: cache.get((p,), "t", lambda: p.detach().clone())
  for _ in range(2):
    assert torch.equal(derive(), p)
  p.data = other(p)
  for _ in range(2):
    got = derive()
    assert got.dtype == p.dtype and torch.equal(got, p)


def test_param_cache_holds_what_its_limit_allows():
  """Derived values live as long as their entries; in-place edits and other tensors are noticed."""
  cache = module.ParamCache(limit=1)
  p, q = torch.zeros(3), torch.ones(3)
  derive = lambda t, tag: cache.get((t,), tag, lambda: t + 1)
  first = weakref.ref(derive(p, "a"))
  assert first() is derive(p, "a")
  derive(q, "b")                                             # the limit of one: the first entry goes
  assert first() is None
  assert derive(p, "a").tolist() == [1, 1, 1]
  p.add_(1)
  assert derive(p, "a").tolist() == [2, 2, 2]
  assert derive(q, "a").tolist() == [2, 2, 2]
  with pytest.raises(ZeroDivisionError):                     # a build that fails leaves nothing behind
    cache.get((p,), "c", lambda: 1 // 0)
  assert cache.get((p,), "c", lambda: 7) == 7


def _on_cpu(monkeypatch, **more):
  """The kernels that the modules below call, as plain torch."""
  packed = []
  fakes = dict(cast=lambda t, dtype: t.to(dtype),
               pack_expert_weights=lambda w: packed.append(w) or w.transpose(1, 2).contiguous(),
               expert_mlp=lambda x, **kw: kw, **more)
  for name, fn in fakes.items():
    monkeypatch.setattr(kernels, name, fn)
  return packed


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("param_dtype", [torch.bfloat16, torch.float32])
def test_mlp_block_biases_follow_edits_without_a_version(monkeypatch, dtype, param_dtype):
  """Biases are read on every call (``b.data.add_`` raises no version counter), and one that changed
  leaves the packed kernels alone."""
  packed = _on_cpu(monkeypatch)
  block = vit_moe.MlpBlock(mlp_dim=8, deterministic=True, dtype=dtype)
  params = {f"Dense_{i}": {"kernel": torch.randn((2, 8, 8)).to(param_dtype),
                           "bias": torch.zeros((2, 8), dtype=param_dtype)} for i in range(2)}
  x = torch.zeros((2, 4, 8), dtype=dtype)
  for step in range(3):
    kw = block.apply_experts({"params": params}, x)
    for name, layer in (("b0", "Dense_0"), ("b1", "Dense_1")):
      assert kw[name].dtype == dtype and torch.equal(kw[name], params[layer]["bias"].to(dtype))
      params[layer]["bias"].data.add_(step + 1)
  assert len(packed) == (2 if dtype == torch.bfloat16 else 0)
  first = weakref.ref(params["Dense_0"]["bias"])
  del kw, params
  assert first() is None                                     # nothing of the block holds them


def test_experts_choice_router_kernel_follows_edits_without_a_version(monkeypatch):
  seen = []
  _on_cpu(monkeypatch, gate_topk=lambda x, w, k, **kw: (seen.append(w) or (x, None, None)))
  monkeypatch.setattr(routing.NoisyTopItemsPerExpertRouter, "_create_dispatcher_and_metrics",
                      lambda self, gates: (gates, {}))
  router = routing.NoisyTopItemsPerExpertRouter(num_experts=4, deterministic=True, dtype=torch.bfloat16,
                                                dispatcher=dict(name="einsum", capacity=2))
  kernel = torch.zeros((16, 4))
  for step in range(3):
    router.apply({"params": {"dense": {"kernel": kernel}}}, torch.zeros((1, 8, 16)))
    assert torch.equal(seen[-1], kernel.to(torch.bfloat16))
    kernel.data.add_(1)


def _bad_calls():
  """(name, call): every tensor of a call with an axis too many or too few, then with too few values or
  the wrong width; shapes that one another's wrapper accepts are in `good`."""
  i32, f32 = (lambda *s: torch.zeros(s, dtype=torch.int32)), (lambda *s: torch.zeros(s))
  mlp = dict(x=f32(2, 6, 8), w0=f32(2, 8, 16), b0=f32(2, 16), w1=f32(2, 16, 8), b1=f32(2, 8))
  packed = dict(x=f32(2, 6, 8), w0=None, b0=f32(2, 16), w1=None, b1=f32(2, 8), w0t=f32(2, 16, 8), w1t=f32(2, 8, 16))
  gathered = dict(mlp, x=f32(12, 8), x_rows=i32(2, 6), rows_per_expert=i32(2))
  good = [
      ("gate_topk", dict(x=f32(2, 6, 8), w=f32(8, 4), num_selected_experts=2, logit_bias=f32(4)),
       dict(x=[(12, 8), (1, 2, 6, 8)], w=[(8, 4, 1), (4, 4)], logit_bias=[(3,)])),
      ("route_assign", dict(topk_val=f32(2, 6, 2), topk_idx=i32(2, 6, 2), num_experts=4, capacity=3, batch_priority=True),
       dict(topk_idx=[(12, 2), (1, 2, 6, 2)], topk_val=[(2, 6, 1)])),
      ("top_items_metrics", dict(gates=f32(2, 6, 4), capacity=3), dict(gates=[(12, 4), (2, 6, 2, 2)])),
      ("dispatch", dict(x=f32(6, 8), token_slot=i32(6, 2), slot_token=i32(9)),
       dict(x=[(6,), (6, 2, 8), (7, 8)], token_slot=[(), (5, 2)], out=[(9, 7)])),
      ("combine", dict(y=f32(9, 8), token_slot=i32(6, 2), weights=f32(6, 2)),
       dict(y=[(9,), (9, 2, 8)], token_slot=[(12,), (2, 3, 2)], weights=[(6, 1)], out=[(6, 7)])),
      ("einsum_dispatch", dict(w=f32(2, 6, 3, 2), data=f32(2, 6, 8), out_dtype=torch.float32),
       dict(w=[(2, 6, 6), (2, 6, 3, 2, 1)], data=[(), (2, 5, 8)])),
      ("einsum_combine", dict(w=f32(2, 6, 3, 2), data=f32(12, 8), out_dtype=torch.float32),
       dict(w=[(2, 6, 6), (2, 6, 3, 2, 1)], data=[(), (11, 8)])),
      ("combine_backward_data", dict(dout=f32(6, 8), token_slot=i32(6, 2), weights=f32(6, 2), slot_token=i32(9), num_slots=9),
       dict(dout=[(6,), (6, 2, 8)], token_slot=[(), (5, 2)], weights=[(5, 2)], slot_token=[(8,)])),
      ("combine_backward_weights", dict(dout=f32(6, 8), y=f32(9, 8), token_slot=i32(6, 2)),
       dict(dout=[(6,), (6, 2, 8)], y=[(9,), (9, 2, 4), (9, 7)], token_slot=[(), (5, 2)])),
      ("combine_backward", dict(dout=f32(6, 8), y=f32(9, 8), token_slot=i32(6, 2), weights=f32(6, 2), slot_token=i32(9)),
       dict(dout=[(6,), (6, 2, 8)], y=[(9,), (9, 7)], token_slot=[(), (5, 2)], weights=[(5, 2)], slot_token=[(8,)])),
      ("dispatch_backward", dict(dbuf=f32(9, 8), token_slot=i32(6, 2)), dict(dbuf=[(9,), (9, 2, 8)], token_slot=[(12,), (2, 3, 2)])),
      ("indices_to_slots", dict(indices=i32(2, 6, 2, 2), num_experts=4, capacity=3), dict(indices=[(12, 2), (2, 6, 2, 1)])),
      ("add_layer_norm", dict(residual=f32(6, 8), branch=f32(6, 8), scale=f32(8), bias=f32(8), eps=1e-6, out_dtype=torch.float32),
       dict(residual=[()], branch=[(6, 4)], scale=[(7,)], bias=[(7,)])),
      ("attention", dict(q=f32(2, 5, 3, 64), k=f32(2, 7, 3, 64), v=f32(2, 7, 3, 64), scale=0.125),
       dict(q=[(2, 5, 192), (1, 2, 5, 3, 64)], k=[(2, 7, 192), (1, 7, 3, 64), (2, 7, 2, 64)],
            v=[(2, 7, 192), (1, 7, 3, 64), (2, 6, 3, 64)])),
      ("soft_route", dict(x=f32(2, 6, 8), mu=f32(8, 4), scale=1.0, with_stats=True),
       dict(x=[(12, 8), (1, 2, 6, 8)], mu=[(8, 2, 2), (7, 4)])),
      ("expert_mlp", mlp, dict(x=[(12, 8), (2, 3, 2, 8), (2, 6, 4)], w0=[(8, 16), (1, 8, 16), (2, 4, 16)],
                               w1=[(16, 8), (1, 16, 8), (2, 8, 8), (2, 16, 4)], b0=[(16,)], b1=[(8,)], out=[(2, 6, 7)])),
      ("expert_mlp", packed, dict(x=[(2, 3, 2, 8)], w0t=[(16, 8), (2, 16, 4), (1, 16, 8)], w1t=[(8, 16), (2, 4, 16), (2, 8, 8)])),
      ("expert_mlp", gathered, dict(x=[(1, 12, 8), (12,)], x_rows=[(12,), (1, 2, 6)], rows_per_expert=[(1,)])),
  ]
  for name, args, bad in good:
    for arg, shapes in bad.items():
      like = args.get(arg)
      for shape in shapes:
        t = torch.zeros(shape, dtype=torch.float32 if like is None else like.dtype)
        yield pytest.param(name, dict(args, **{arg: t}), id=f"{name}-{arg}-{'x'.join(map(str, shape)) or 'scalar'}")
  for what, compact in (("fill-axes", (i32(2), i32(1, 6, 2), 3)), ("slot-axes", (i32(1, 2), i32(6, 2), 3)),
                        ("groups", (i32(2, 2), i32(1, 6, 2), 3))):
    yield pytest.param("expert_mlp", dict(mlp, x=f32(12, 8), compact=compact), id=f"expert_mlp-compact-{what}")


@pytest.mark.parametrize("name,args", _bad_calls())
def test_entry_points_refuse_tensors_of_the_wrong_shape(monkeypatch, name, args):
  """The C ABI is told addresses and sizes: what they are taken from is checked on the host.  (Shapes are
  looked at before anything else, so CPU tensors do here.)"""
  monkeypatch.setattr(_hip, "raw_stream", lambda: 0)
  with pytest.raises(ValueError):
    getattr(kernels, name)(**args)


@pytest.mark.parametrize("name", ["combine_backward", "combine_backward_weights"])
@pytest.mark.parametrize("types", [(torch.float32, torch.bfloat16), (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("timed", [False, True])
def test_gradients_of_combine_refuse_rows_of_another_type(monkeypatch, name, types, timed):
  """The kernels read y with the width of dout's type: bfloat16 rows under a float32 gradient would be
  read past their end."""
  monkeypatch.setattr(_hip, "raw_stream", lambda: 0)
  monkeypatch.setattr(_hip, "timed", lambda call: timed)
  slots = torch.zeros((6, 2), dtype=torch.int32)
  more = (torch.zeros((6, 2)), None) if name == "combine_backward" else ()
  with pytest.raises(TypeError, match="dout"):
    getattr(kernels, name)(torch.zeros((6, 8), dtype=types[0]), torch.zeros((9, 8), dtype=types[1]), slots, *more)


@pytest.mark.parametrize("dtype", [_hip.F32, _hip.BF16])
@pytest.mark.parametrize("D", [8, 40, 144])
def test_gathered_rows_of_broken_k_tiles_are_refused(dtype, D):
  """x_rows asks for whole 32-wide k tiles at every size; refused before anything is launched."""
  p = _hip.ExpertMlpParams(16, 16, None, 16, None, 16, 16, 16, 16, 1 << 40, 2, 6, D, 64, dtype, _hip.GELU_TANH, 16, 16, 12)
  assert _hip.lib().vmoe_expert_mlp(_hip.ctypes.byref(p), None) == kernels._E_UNSUPPORTED


@pytest.mark.parametrize("name", ["vmoe_combine_backward", "vmoe_combine_backward_data", "vmoe_combine_backward_weights",
                                  "vmoe_dispatch", "vmoe_combine", "vmoe_dispatch_backward"])
def test_row_movers_refuse_more_rows_than_a_launch_has_waves(name):
  """A wave per row: 2^32 - 1 threads are 2^26 - 1 rows.  (Rows and slots of eight bfloat16 values; dispatch and
  combine take such a kernel where the rows are too wide for their others.)"""
  n, D = (1 << 26, 8) if "backward" in name and name != "vmoe_dispatch_backward" else (1 << 26, 1 << 17)
  if name == "vmoe_dispatch":
    p = _hip.DispatchParams(16, 16, 16, 16, n // 2, n // 2 + 1, 2, D, _hip.BF16)
  elif "backward_" in name or name == "vmoe_combine_backward":
    slots = 8 if name.endswith("weights") else n // 2 + 1
    p = _hip.CombineBackwardParams(16, 16, 16, 16, 16, 16, 16, n + 1 - slots if slots > 8 else n, slots, 2, D, _hip.BF16)
  else:
    p = _hip.CombineParams(16, 16, 16, 16, n, 8, 2, D, _hip.BF16)
  assert getattr(_hip.lib(), name)(_hip.ctypes.byref(p), None) == -5      # VMOE_E_OVERFLOW


def test_dispatch_needs_a_number_of_slots(monkeypatch):
  monkeypatch.setattr(_hip, "raw_stream", lambda: 0)
  with pytest.raises(TypeError):
    kernels.dispatch(torch.zeros((6, 8)), torch.zeros((6, 2), dtype=torch.int32), None)


@pytest.mark.parametrize("num_slots", [9, 9.0, np.float32(9)])
def test_dispatch_takes_any_number_that_is_an_integer(monkeypatch, num_slots):
  """int(num_slots), as a capacity computed in floating point asks for: the call gets as far as the device."""
  monkeypatch.setattr(_hip, "raw_stream", lambda: 0)
  with pytest.raises(_hip.VmoeError, match="ROCm device"):
    kernels.dispatch(torch.zeros((6, 8)), torch.zeros((6, 2), dtype=torch.int32), None, num_slots=num_slots)


@pytest.mark.parametrize("shape", [(3, 0), (0,), (0, 0)])
def test_add_layer_norm_refuses_an_empty_last_axis(monkeypatch, shape):
  """The number of rows is a quotient: ZeroDivisionError, not a trap."""
  monkeypatch.setattr(_hip, "raw_stream", lambda: 0)
  for branch in (None, torch.zeros(shape)):
    with pytest.raises(ZeroDivisionError):
      kernels.add_layer_norm(torch.zeros(shape), branch, None, None, 1e-6, torch.float32)


def test_native_host_side_releases_the_interpreter():
  """Other Python threads run while a native call does its work (here: a copy of a transposed tensor,
  before the call finds that it is not on the GPU)."""
  x = torch.zeros((6000, 6000)).t()
  started, done, ticks = threading.Event(), threading.Event(), []

  def tick():
    started.set()
    while not done.wait(0.002):
      ticks.append(time.perf_counter())

  thread = threading.Thread(target=tick)
  threads = torch.get_num_threads()
  torch.set_num_threads(1)
  try:
    thread.start()
    started.wait()
    begin = time.perf_counter()
    with pytest.raises(_hip.VmoeError, match="no CPU fallback"):
      _hip.host().cast(0, x, torch.bfloat16)
    end = time.perf_counter()
  finally:
    torch.set_num_threads(threads)
    done.set()
    thread.join()
  assert sum(begin < t < end for t in ticks) >= 3, (len(ticks), end - begin)


def test_expert_mlp_sizes_come_from_the_operands(monkeypatch):
  """The parameter block of a call takes its sizes from the items, not from a caller's output buffer,
  which may be larger or flat."""
  from vmoe_amd import _hip as H
  monkeypatch.setattr(H, "ptr", lambda t: None if t is None else t.data_ptr())
  E, R, D, M = 3, 5, 16, 32
  w0t, w1t = torch.zeros(E, M, D), torch.zeros(E, D, M)
  for out in (torch.zeros(E, R, D), torch.zeros(E + 1, R + 2, D), torch.zeros(E * R, D)):
    for x, x_rows in ((torch.zeros(E, R, D), None), (torch.zeros(7, D), torch.zeros(E, R, dtype=torch.int32))):
      p = kernels._expert_mlp_params(x, None, None, None, None, w0t, w1t, True, out, None, x_rows)
      assert (p.E, p.R, p.D, p.M, p.num_items) == (E, R, D, M, 0 if x_rows is None else 7)
  with pytest.raises(ValueError):      # gathered items have two axes
    kernels._expert_mlp_params(torch.zeros(7, D, 2), None, None, None, None, w0t, w1t, True, torch.zeros(E, R, D),
                         None, torch.zeros(E, R, dtype=torch.int32))


def _ragged_mlp_bytes(E, R, D, M):
  """Workspace of a bfloat16 call with row counts: a product that takes the large tiles keeps a plan in it."""
  one = _hip.c_void_p(16)
  p = _hip.ExpertMlpParams(one, None, None, None, None, one, one, one, None, 0, E, R, D, M, _hip.BF16, 0, one, None, 0)
  return _hip.lib().vmoe_expert_mlp_workspace_bytes(_hip.ctypes.byref(p))


@pytest.mark.parametrize("E,R,D,M,small", [
    (1, 10482, 224, 832, False), (1, 10770, 288, 1088, False), (1, 12229, 288, 1152, False),
    (3, 3411, 352, 1408, False),                              # two to six (batch, column tile) pairs
    (1, 196, 768, 3072, True), (8, 52, 768, 3072, True)])
def test_small_tiles_are_not_taken_where_they_would_run_on_few_dies(monkeypatch, E, R, D, M, small):
  """gemm_bf16_rows_kernel gives all row tiles of a (batch, column tile) pair to one die: over many rows of a
  narrow layer most dies have nothing to do, and the large tiles are the faster ones."""
  monkeypatch.delenv("VMOE_SECOND_PRODUCT", raising=False)
  monkeypatch.delenv("VMOE_ROW_TILES", raising=False)
  chosen = _ragged_mlp_bytes(E, R, D, M)
  monkeypatch.setenv("VMOE_ROW_TILES", "off")
  assert (chosen < _ragged_mlp_bytes(E, R, D, M)) == small


@pytest.mark.parametrize("E,R,D,M", [(51, 729, 640, 2560), (20, 1571, 640, 2560), (28, 381, 576, 2304)])
def test_medium_tiles_are_chosen_by_the_rounds_that_a_plan_makes_of_them(monkeypatch, E, R, D, M):
  """A launch plan deals whole row tiles to the dies: shapes whose medium tiles would fill the chip's rounds one by one, and
  do not as rows of column tiles, keep the large ones."""
  monkeypatch.delenv("VMOE_SECOND_PRODUCT", raising=False)
  monkeypatch.delenv("VMOE_ROW_TILES", raising=False)
  chosen = _ragged_mlp_bytes(E, R, D, M)
  monkeypatch.setenv("VMOE_ROW_TILES", "off")
  assert chosen == _ragged_mlp_bytes(E, R, D, M)


@pytest.mark.parametrize("packed", [True, False])
@pytest.mark.parametrize("has_aux,inputs", [(True, 1), (False, 2)])
def test_only_dispatchers_without_packed_rows_ask_for_float32_products(packed, has_aux, inputs):
  """A layer behind a bfloat16 dispatcher with packed rows takes the same float32 products with auxiliary
  outputs or several inputs, where its rows are not packed, as without them."""
  class Inner:
    supports_packed = lambda self: packed
    dispatch = combine = lambda self, data: data

  class Experts:
    def apply_experts(self, variables, *dispatched, float32_products=False):
      asked.append(float32_products)
      return (dispatched[0], None) if has_aux else dispatched[0]

    apply_experts.takes_float32_products = True

  asked = []
  layer = moe.sparse_moe_spmd(Experts, has_aux=has_aux)()
  items = [torch.zeros((2, 3), dtype=torch.int32)] * inputs       # (integers pass the dispatcher uncast)
  layer.apply({}, moe.Bfloat16Dispatcher(Inner()), *items)
  assert asked == [not packed]


def test_negative_indices_are_refused_in_every_thread(monkeypatch):
  """Two threads dispatch by the same new maps before the counters of invalid indices arrive: one waits for them
  first and raises, and so does the other."""
  monkeypatch.setattr(moe.K, "indices_to_slots", lambda *args: (None, None, torch.tensor([0, 1])))
  event = type("Event", (), {"record": lambda self: None, "synchronize": lambda self: None})
  monkeypatch.setattr(torch.cuda, "Event", event)
  dispatcher = moe.ExpertIndicesDispatcher(torch.zeros((1, 2, 1, 2), dtype=torch.int32), torch.ones((1, 2, 1)), 2, 2)
  dispatcher._maps(settle=False)
  for _ in range(2):
    with pytest.raises(ValueError, match="negative indices"):
      dispatcher._settle()
  with pytest.raises(ValueError, match="negative indices"):
    dispatcher._maps()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("same", [True, False])
def test_library_projections_get_weights_in_their_own_layout(monkeypatch, dtype, same):
  """Where the library multiplies, it is handed contiguous (out, in) weights in every type, not transposed views;
  the result is the projections' in the reference's order."""
  linear, seen = torch.nn.functional.linear, []
  monkeypatch.setattr(torch.nn.functional, "linear", lambda x, w, b: seen.append(w) or linear(x, w, b))
  attn = vit_moe.MultiHeadDotProductAttention(num_heads=2, dtype=dtype)
  x = torch.randn(2, 5, 16, generator=torch.Generator().manual_seed(0))
  kv = x if same else x[:, :3].contiguous()
  p = attn.init(0, x, kv)["params"]
  out = attn.apply({"params": p}, x, kv)
  assert len(seen) == (2 if same else 3) and all(w.is_contiguous() for w in seen)
  q, k, v = (torch.einsum("bsd,dhe->bhse", t, p[n]["kernel"]) for n, t in (("query", x), ("key", kv), ("value", kv)))
  want = torch.einsum("bhse,hed->bsd", torch.nn.functional.scaled_dot_product_attention(q, k, v), p["out"]["kernel"])
  assert torch.allclose(out.float(), want, rtol=0, atol=1e-5 if dtype == torch.float32 else 5e-2)


@pytest.mark.parametrize("x,w,b", [
    ((6, 4), (4, 8), (16,)),            # a bias longer than the row
    ((6, 4), (4, 8), (1,)),
    ((6, 4), (4, 8), (6, 8)),
    ((6, 4), (8, 8), (8,)),
    ((6, 0), (0, 8), (8,)),
])
@pytest.mark.parametrize("timed", [False, True])
def test_dense_refuses_what_its_sizes_do_not_cover(monkeypatch, x, w, b, timed):
  """Widths that differ, an empty one, and biases of other sizes than a row."""
  if timed:
    monkeypatch.setattr(_hip, "_timing_sink", {})
  else:
    monkeypatch.setattr(_hip, "raw_stream", lambda: 0)
  with pytest.raises(ValueError):
    kernels.dense(torch.zeros(x), torch.zeros(w), torch.zeros(b))


@pytest.mark.parametrize("bias", [(8,), (1, 8), (6, 8), (6, 1), (1,), ()])
def test_dense_layers_spread_biases_as_the_library_does(monkeypatch, bias):
  """A bias that is not one row of the output takes the library's product, which spreads it; one that is goes to
  the package's."""
  asked = []
  monkeypatch.setattr(kernels, "dense_pays", lambda *args: True)
  monkeypatch.setattr(kernels, "dense_takes", lambda *args: True)
  monkeypatch.setattr(module, "is_plain", lambda *args: True)
  monkeypatch.setattr(kernels, "dense", lambda x, w, b: asked.append(b.shape) or x @ w + b)
  x, w, b = torch.randn(6, 4), torch.randn(4, 8), torch.randn(bias)
  assert torch.allclose(vit_moe._affine(x, w, b), torch.addmm(b, x, w))
  assert asked == ([(8,)] if bias == (8,) else [])
  if bias in [(8,), (1,), ()]:
    assert torch.allclose(vit_moe.MultiHeadDotProductAttention._project(x, w, b), x @ w + b)
    assert len(asked) == (2 if bias == (8,) else 0)
  with pytest.raises(RuntimeError):
    vit_moe._affine(torch.randn(6, 8), w, b)


@pytest.mark.parametrize("full", [True, False])
@pytest.mark.parametrize("gathers,takes", [(True, True), (False, True), (True, False)])
def test_experts_hear_that_every_packed_row_is_live(full, gathers, takes):
  """What experts choice knows about its rows reaches experts that ask for it, and only those."""
  class Dispatcher(moe.ExpertIndicesDispatcher):
    dispatch_packed = lambda self, data: (data, self.packed_rows()[1])
    combine_packed = lambda self, data: data

  class Experts:
    supports_packed_rows = True
    can_gather = lambda self, items: gathers

    def apply_experts_gathered(self, variables, items, row_token, rows_per_expert, **hints):
      asked.append(hints)
      return items

    def apply_experts(self, variables, dispatched, rows_per_expert=None, **hints):
      asked.append(hints)
      return dispatched

    apply_experts.takes_full_rows = apply_experts_gathered.takes_full_rows = takes

  asked = []
  maps = (torch.zeros((2, 3, 1), dtype=torch.int32), torch.full((2,), 4), torch.zeros((2, 4), dtype=torch.int32))
  dispatcher = Dispatcher(torch.zeros((2, 3, 1, 2), dtype=torch.int32), torch.ones((2, 3, 1)), 2, 2)
  dispatcher.set_packed_maps(maps, full_rows=full)
  wrapped = moe._SparseEinsumDispatcher(dispatcher, torch.float32)
  for d in (dispatcher, wrapped):
    moe.sparse_moe_spmd(Experts)().apply({}, d, torch.zeros((2, 3, 8)))
  assert asked == [{"full_rows": True} if full and takes else {}] * 2


@pytest.mark.parametrize("rows,D,M,pays", [
    (1568, 768, 2304, True),                                    # either side of where multiples of 256 stop
    (4521, 768, 2304, True), (4522, 768, 2304, False),
    (40690, 256, 768, True), (40691, 256, 768, False),
    (50176, 704, 2112, True), (50176, 1024, 1024, False),        # other widths do not
    (2089, 1152, 1160, True), (2096, 1152, 1160, False),
    (100, 1020, 768, False), (100, 768, 1020, False), (0, 768, 768, False),
    (1 << 20, 960, 960, True), (1 << 21, 960, 960, False),       # byte offsets of 31 bits
])
def test_where_bfloat16_dense_layers_take_the_kernel(rows, D, M, pays):
  assert kernels.dense_pays(rows, D, M, torch.bfloat16) == pays


def test_kept_launch_plans_are_those_of_the_shapes_that_ask(monkeypatch):
  """A thread keeps what it worked out for its last shapes: more of them, in any order, get their own."""
  monkeypatch.delenv("VMOE_ROW_TILES", raising=False)
  shapes = [(1, 1568, 768, 3072), (8, 412, 768, 3072), (32, 1600, 768, 3072), (5, 800, 832, 3328), (47, 140, 576, 2304),
            (20, 1571, 640, 2560)]
  monkeypatch.setenv("VMOE_SECOND_PRODUCT", "")           # (worked out anew on every call)
  want = [_ragged_mlp_bytes(*s) for s in shapes]
  monkeypatch.delenv("VMOE_SECOND_PRODUCT")
  rng = np.random.default_rng(0)
  for i in rng.integers(0, len(shapes), 200):
    assert _ragged_mlp_bytes(*shapes[i]) == want[i]
