"""What this framework is asked to do, as cases that can be timed.

Five kinds of call, all through the public entry points:

* ``sparse``: one sparse MoE layer (``MlpMoeBlock`` with the default router: top-K experts per
  item, capacity-bounded buffers, with or without batch priority routing);
* ``choice``: the same layer with the experts-choice router;
* ``soft``: the same layer with the Soft MoE router;
* ``model``: a whole V-MoE vision transformer, images to logits;
* ``grad``: dispatch and combine with their gradients, around experts of the caller's own.

``listed()`` names cases from a single image to the largest batch, ``draw()`` gives others of the
same ranges: odd group sizes, widths between the usual ones, expert counts that are no power of
two, capacity factors on both sides of one.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from vmoe_amd import moe
from vmoe_amd.nn import vit_moe

_SOFT_ROUTER = "vmoe_amd.projects.soft_moe.router.SoftRouter"


def listed():
  return [
      # One 224 px image at 16 x 16 patches through one layer of the B/16 model (8 experts): what an
      # on-line server waits for.  Launches, latency and reading the weights.
      dict(name="sparse_one_image", kind="sparse", images=1, tokens=196, group=1, d=768, m=3072,
           experts=8, k=2, cf=1.05, bpr=True, skew=0.0, dtype="bfloat16"),
      # The S/32-style layer in float32: 32 images of 49 tokens, every image a group.
      dict(name="sparse_s32_f32", kind="sparse", images=32, tokens=49, group=1, d=512, m=2048,
           experts=8, k=2, cf=1.05, bpr=False, skew=0.0, dtype="float32"),
      # One group of the 32-expert layer: a small serving batch, 300 MB of expert weights for 1 568
      # tokens.
      dict(name="sparse_b16_one_group", kind="sparse", images=8, tokens=196, group=8, d=768, m=3072,
           experts=32, k=2, cf=1.0, bpr=True, skew=0.0, dtype="bfloat16"),
      # The headline layer: 256 images, 32 experts, batch priority routing.
      dict(name="sparse_b16", kind="sparse", images=256, tokens=196, group=8, d=768, m=3072,
           experts=32, k=2, cf=1.0, bpr=True, skew=0.0, dtype="bfloat16"),
      # The L/16 layer at 384 px with half the capacity and an unbalanced router.
      dict(name="sparse_l16_half_capacity", kind="sparse", images=64, tokens=576, group=4, d=1024,
           m=4096, experts=32, k=2, cf=0.5, bpr=True, skew=2.0, dtype="bfloat16"),
      # Experts choose their items: B/16 layer, 64 images.
      dict(name="choice_b16", kind="choice", images=64, tokens=196, group=8, d=768, m=3072,
           experts=32, cf=2.0, dtype="bfloat16"),
      # Soft MoE as benchmarked: 128 experts of one slot, 256 images.
      dict(name="soft_b16_one_slot", kind="soft", images=256, tokens=196, d=768, m=3072,
           experts=128, slots=1, dtype="bfloat16"),
      # Soft MoE with as many slots as the router's default capacity factor of 1 gives: 196 tokens,
      # 128 experts, two slots each.
      dict(name="soft_b16_default_slots", kind="soft", images=64, tokens=196, d=768, m=3072,
           experts=128, slots=2, dtype="bfloat16"),
      # A small Soft MoE layer in float32 (S/32: 49 tokens per image, as many slots).
      dict(name="soft_s32_f32", kind="soft", images=32, tokens=49, d=512, m=2048, experts=16,
           slots=3, dtype="float32"),
      # The B/16 model (experts in every other block): one routing group of images, where the host
      # and the launches show, and the whole benchmark batch.
      dict(name="model_b16_batch_8", kind="model", images=8, side=224, patch=16, d=768, m=3072,
           layers=12, experts=8, k=2, cf=1.05, bpr=True, group=8, dtype="bfloat16"),
      dict(name="model_b16_batch_512", kind="model", images=512, side=224, patch=16, d=768, m=3072,
           layers=12, experts=8, k=2, cf=1.05, bpr=True, group=8, dtype="bfloat16"),
      # Dispatch and combine, forwards and backwards, around experts of the caller's own.
      dict(name="grad_b16", kind="grad", images=128, tokens=196, group=8, d=768, experts=32, k=2,
           cf=1.0, dtype="bfloat16"),
  ]


# ------------------------------------------------------------------------------ drawn cases
def _log_int(rng, lo, hi):
  return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng):
  """Model widths: mostly multiples of 64, now and then of 32."""
  step = 64 if rng.random() < 0.8 else 32
  return step * rng.randint(192 // step, 1024 // step)


def _hidden(rng, d):
  return 4 * d if rng.random() < 0.7 else 64 * rng.randint(max(1, 2 * d // 64), 4 * d // 64)


def _dtype(rng):
  return "bfloat16" if rng.random() < 0.7 else "float32"


def draw(rng):
  kind = rng.choice(["sparse", "sparse", "sparse", "choice", "soft", "soft", "model", "grad"])
  case = dict(kind=kind)
  if kind == "model":
    patch = rng.choice([16, 32])
    group = rng.randint(1, 8)
    d = 64 * rng.randint(3, 16)
    case.update(side=patch * rng.randint(6, 18), patch=patch, d=d, m=4 * d,
                layers=2 * rng.randint(2, 6), experts=_log_int(rng, 4, 32), k=rng.randint(1, 2),
                cf=round(rng.uniform(0.5, 2.0), 2), bpr=rng.random() < 0.5, group=group,
                dtype=_dtype(rng))
    case["images"] = group * _log_int(rng, 1, 64)
  else:
    d = _width(rng)
    case.update(tokens=_log_int(rng, 49, 577), d=d, dtype=_dtype(rng))
    if kind != "grad":
      case["m"] = _hidden(rng, d)
    if kind == "soft":
      case.update(images=_log_int(rng, 4, 256), experts=_log_int(rng, 4, 128),
                  slots=rng.randint(1, 4))
      # One group's logits have to fit the router's on-chip memory.
      size = 2 if case["dtype"] == "bfloat16" else 4
      pad = lambda n: (n + 31) // 32 * 32
      fits = lambda: pad(case["tokens"]) * (4 + size * (pad(case["experts"] * case["slots"]) + 2)) < 160_000
      while not fits() and case["slots"] > 1:
        case["slots"] -= 1
      while not fits():
        case["tokens"] //= 2
    else:
      group = rng.randint(1, 8)
      case.update(images=group * max(1, _log_int(rng, 196, 50176) // (group * case["tokens"])),
                  group=group, experts=_log_int(rng, 4, 64), cf=round(rng.uniform(0.5, 2.0), 2))
      if kind != "choice":
        case["k"] = rng.choice([1, 2, 2, 2, 3, 4])
      if kind == "sparse":
        case.update(bpr=rng.random() < 0.5, skew=rng.choice([0.0, 0.0, 1.0, 2.0]))
  # No dearer than the largest listed case.
  limit = 5e12 if case["dtype"] == "bfloat16" else 3e11
  while work(case)["flops"] > limit:
    step = case.get("group", 1)
    if case["images"] > step:
      case["images"] = max(step, case["images"] // 2 // step * step)
    elif step > 1:
      case["images"] = case["group"] = step // 2
    else:
      case["tokens" if "tokens" in case else "layers"] //= 2
  return case


# ------------------------------------------------------------------------------ states
def _torch_dtype(case):
  return torch.bfloat16 if case["dtype"] == "bfloat16" else torch.float32


class _Maker:
  """Seeded tensors on the GPU."""

  def __init__(self, seed):
    self.device = torch.device("cuda:0")
    self.gen = torch.Generator(device=self.device)
    self.gen.manual_seed(int(seed))

  def normal(self, *shape, std=1.0, dtype=torch.float32):
    return (torch.randn(shape, generator=self.gen, device=self.device) * std).to(dtype)

  def tokens(self, images, tokens, d, dtype):
    """Tokens as a layer norm leaves them."""
    x = torch.randn((images, tokens, d), generator=self.gen, device=self.device)
    return torch.nn.functional.layer_norm(x, (d,)).to(dtype)

  def mlp(self, lead, d, m, dtype):
    return {"Dense_0": {"kernel": self.normal(*lead, d, m, std=d ** -0.5, dtype=dtype),
                        "bias": self.normal(*lead, m, std=0.02, dtype=dtype)},
            "Dense_1": {"kernel": self.normal(*lead, m, d, std=m ** -0.5, dtype=dtype),
                        "bias": self.normal(*lead, d, std=0.02, dtype=dtype)}}


def _capacity(case):
  """Rows per expert and group, as the dispatchers compute it."""
  tokens = _group_tokens(case) * case.get("k", 1)
  c = math.ceil(tokens * case["cf"] / case["experts"])
  c += -c % 4
  return min(c, _group_tokens(case)) if case["kind"] == "choice" else c


def _tokens_per_image(case):
  return (case["side"] // case["patch"]) ** 2 if case["kind"] == "model" else case["tokens"]


def _group_tokens(case):
  return case["group"] * _tokens_per_image(case)


def prepare(case, seed):
  mk = _Maker(seed)
  dtype = _torch_dtype(case)
  kind = case["kind"]
  if kind == "model":
    return _prepare_model(case, mk, dtype)
  d = case["d"]
  x = mk.tokens(case["images"], case["tokens"], d, dtype)
  if kind == "grad":
    g, s, e, k = case["images"] // case["group"], _group_tokens(case), case["experts"], case["k"]
    gates = torch.softmax(mk.normal(g, s, e), dim=-1)
    capacity = _capacity(case)
    routed = moe.get_top_experts_per_item_dispatcher(
        gates, "indices", num_selected_experts=k, capacity=capacity, batch_priority=True)
    return dict(kind=kind, indices=routed.indices, experts=e, capacity=capacity,
                weights=routed.combine_weights.to(torch.float32).requires_grad_(),
                x=x.view(g, s, d).requires_grad_(), grad_out=mk.normal(g, s, d, dtype=dtype))
  e, m = case["experts"], case["m"]
  group_size = case["tokens"] if kind == "soft" else _group_tokens(case)
  if kind == "soft":
    params = {"mu": mk.normal(d, e, case["slots"], std=d ** -0.5),
              "scale": torch.ones((), device=mk.device)}
    router = dict(name=_SOFT_ROUTER, num_slots=case["slots"], compute_similarity_metrics=False)
  else:
    params = {"dense": {"kernel": mk.normal(d, e, std=d ** -0.5)}}
    if kind == "choice":
      router = dict(name="NoisyTopItemsPerExpertRouter",
                    dispatcher=dict(name="einsum", capacity=_capacity(case)))
    else:
      router = dict(num_selected_experts=case["k"],
                    dispatcher=dict(name="indices", batch_priority=case["bpr"],
                                    capacity_factor=case["cf"]))
      if case["skew"]:
        router["logit_bias"] = mk.normal(e, std=case["skew"])
  layer = vit_moe.MlpMoeBlock(mlp_dim=m, num_experts=e, group_size=group_size, deterministic=True,
                              router=router, dtype=dtype)
  variables = {"params": {"Router": params, "Mlp": mk.mlp((e,), d, m, dtype)}}
  return dict(kind=kind, layer=layer, variables=variables, x=x)


def _prepare_model(case, mk, dtype):
  d, m, patch, side, layers = case["d"], case["m"], case["patch"], case["side"], case["layers"]
  heads, n = d // 64, _tokens_per_image(case)
  dev = mk.device
  moe_layers = tuple(range(1, layers, 2))
  norm = lambda: {"scale": torch.ones(d, device=dev), "bias": torch.zeros(d, device=dev)}
  proj = lambda: {"kernel": mk.normal(d, heads, 64, std=d ** -0.5),
                  "bias": torch.zeros((heads, 64), device=dev)}
  encoder = {"posembed_input": {"pos_embedding": mk.normal(1, n, d, std=0.02)},
             "encoder_norm": norm()}
  for b in range(layers):
    block = {"LayerNorm_0": norm(), "LayerNorm_1": norm(),
             "SelfAttention": {"query": proj(), "key": proj(), "value": proj(),
                               "out": {"kernel": mk.normal(heads, 64, d, std=d ** -0.5),
                                       "bias": torch.zeros(d, device=dev)}}}
    if b in moe_layers:
      block["Moe"] = {"Router": {"dense": {"kernel": mk.normal(d, case["experts"], std=d ** -0.5)}},
                      "Mlp": mk.mlp((case["experts"],), d, m, torch.float32)}
    else:
      block["Mlp"] = mk.mlp((), d, m, torch.float32)
    encoder[f"encoderblock_{b}"] = block
  variables = {"params": {
      "embedding": {"kernel": mk.normal(patch, patch, 3, d, std=(3 * patch * patch) ** -0.5),
                    "bias": torch.zeros(d, device=dev)},
      "Encoder": encoder,
      "head": {"kernel": mk.normal(d, 1000, std=d ** -0.5), "bias": torch.zeros(1000, device=dev)}}}
  model = vit_moe.VisionTransformerMoe(
      num_classes=1000, patch_size=(patch, patch), hidden_size=d, classifier="gap",
      representation_size=None, deterministic=True,
      encoder=dict(num_layers=layers, mlp_dim=m, num_heads=heads, dtype=dtype,
                   moe=dict(layers=moe_layers, num_experts=case["experts"],
                            group_size=_group_tokens(case),
                            router=dict(num_selected_experts=case["k"],
                                        dispatcher=dict(name="indices", batch_priority=case["bpr"],
                                                        capacity_factor=case["cf"])))))
  images = torch.rand((case["images"], side, side, 3), generator=mk.gen, device=dev) * 2 - 1
  return dict(kind="model", layer=model, variables=variables, x=images)


def run(state):
  if state["kind"] == "grad":
    x, w = state["x"], state["weights"]
    dispatcher = moe.ExpertIndicesDispatcher(state["indices"], w, state["experts"],
                                             state["capacity"])
    out = dispatcher.combine(dispatcher.dispatch(x))
    dx, dw = torch.autograd.grad(out, (x, w), state["grad_out"])
    return out, dx, dw
  return state["layer"].apply(state["variables"], state["x"])


# ------------------------------------------------------------------------------ what it takes
def _kept(case):
  """Assignments that find room in the buffers, from simulated logits."""
  groups = case["images"] // case["group"]
  s, e, c = _group_tokens(case), case["experts"], _capacity(case)
  if case["kind"] == "choice":
    return groups * e * c
  k, skew = case["k"], case.get("skew", 0.0)
  rng = np.random.RandomState(0)
  tries = 16 if skew else 2
  kept = 0.0
  for _ in range(tries):
    logits = rng.standard_normal((min(s, 2048), e)) + skew * rng.standard_normal(e)
    chosen = np.argsort(-logits, axis=1)[:, :k]
    counts = np.bincount(chosen.reshape(-1), minlength=e) * (s / len(logits))
    kept += np.minimum(counts, c).sum() / tries
  return float(groups * kept)


def work(case):
  kind, d = case["kind"], case["d"]
  b = 2 if case["dtype"] == "bfloat16" else 4
  t = case["images"] * _tokens_per_image(case)
  if kind == "grad":
    # forwards: x in, buffer out; buffer in, out out.  Backwards: the gradient in, the buffer's
    # gradient out and in, x's gradient out, and the buffer and the gradient for the weights'.
    rows, kept = case["experts"] * case["images"] // case["group"] * _capacity(case), _kept(case)
    return dict(bytes=b * d * (5 * t + 2 * rows + 3 * kept) + 24 * t * case["k"],
                flops=6.0 * kept * d)
  m = case["m"]
  if kind == "soft":
    slots = case["experts"] * case["slots"]
    rows = case["images"] * slots
    return dict(bytes=b * (2 * t * d + d * slots + 2 * case["experts"] * d * m),
                flops=3 * 2.0 * t * d * slots + 4.0 * rows * d * m)
  kept, e = _kept(case), case["experts"]
  used = min(e, kept)
  moe_flops = 2.0 * t * d * e + 4.0 * kept * d * m
  if kind != "model":
    return dict(bytes=b * (2 * t * d + d * e + 2 * used * d * m), flops=moe_flops)
  layers, n = case["layers"], _tokens_per_image(case)
  sparse, dense = layers // 2, layers - layers // 2
  patch = 3 * case["patch"] ** 2
  per_block = 8.0 * t * d * d + 4.0 * t * n * d
  flops = (layers * per_block + dense * 4.0 * t * d * m + sparse * moe_flops
           + 2.0 * t * patch * d + 2.0 * case["images"] * d * 1000)
  weights = b * (layers * 4 * d * d + dense * 2 * d * m + sparse * (2 * used * d * m + d * e))
  return dict(bytes=weights + 4 * (patch * d + 1000 * d + case["images"] * (3 * case["side"] ** 2 + 1000)),
              flops=flops)


def tolerance(case):
  """About four times what the same calls differ by between summation orders of the gating, of
  either expert product and of the Soft MoE router (largest seen: bfloat16 layers 4e-4 and one bit
  in the last place here and there, bfloat16 models 2e-3, float32 7e-7 and 1.2e-5)."""
  if case["dtype"] == "float32":
    return dict(rel=1e-5 if case["kind"] == "model" else 5e-6,
                max=4e-4 if case["kind"] == "model" else 6e-5)
  return dict(rel=8e-3, max=0.1) if case["kind"] == "model" else dict(rel=2e-3, max=0.08)
