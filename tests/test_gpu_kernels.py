"""Parity of each HIP kernel (called through the C ABI) against the CPU oracle."""
import os
import numpy as np
import pytest
import torch

from oracle import moe_oracle as O
from oracle import route_c
from tests.util import assert_close, dev, tdtype, to_dev, to_np

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
  from vmoe_amd import kernels
  return kernels


# ------------------------------------------------------------------ cast
def test_cast_matches_round_to_nearest_even(K):
  rng = np.random.default_rng(0)
  x = (rng.standard_normal(100003) * 10.0 ** rng.integers(-10, 10, 100003)).astype(np.float32)
  x[:4] = [0.0, -0.0, 1.00390625, 1.01171875]   # exact ties
  got = to_np(K.cast(to_dev(x), torch.bfloat16))
  np.testing.assert_array_equal(got, O.bf16_round(x))
  back = to_np(K.cast(K.cast(to_dev(x), torch.bfloat16), torch.float32))
  np.testing.assert_array_equal(back, O.bf16_round(x))


# ------------------------------------------------------------------ top-k
@pytest.mark.parametrize("E,k", [(3, 2), (8, 2), (32, 2), (32, 5), (100, 7), (1000, 3)])
def test_topk_exact_with_ties(K, E, k):
  rng = np.random.default_rng(E)
  g = rng.integers(0, 4, (257, E)).astype(np.float32) / 4     # heavy ties
  g[0] = 0.0
  val, idx = K.topk(to_dev(g), k)
  want_v, want_i = O.top_k(g, k)
  np.testing.assert_array_equal(to_np(idx), want_i)
  np.testing.assert_array_equal(to_np(val), want_v)


# ------------------------------------------------------------------ gating
GATE_CASES = [
    # G, S, D, E, K, dtype
    (2, 49, 512, 8, 2, O.F32),
    (3, 50, 64, 5, 3, O.F32),
    (2, 100, 768, 32, 2, O.BF16),
    (1, 33, 1024, 32, 2, O.BF16),
    (2, 64, 264, 40, 4, O.BF16),
    (2, 37, 128, 100, 2, O.F32),
    (1, 1568, 768, 32, 2, O.BF16),
    (1, 33000, 1024, 32, 2, O.BF16),   # streaming kernel, rings of two slots (the router kernel takes 66 KB)
    (1, 8200, 768, 32, 2, O.BF16),     # streaming kernel, rings of three slots, a last tile of 8 items
    (3, 2741, 768, 8, 2, O.BF16),      # streaming kernel, experts padded to the 32-wide tile
    (2, 4100, 256, 24, 3, O.BF16),     # streaming kernel, four chunks of k
    (1, 8192, 64, 16, 1, O.BF16),      # streaming kernel, a single chunk of k
    (2, 77, 2048, 32, 2, O.BF16),      # router kernel staged in two chunks along D
    (2, 45, 768, 16, 2, O.BF16),       # experts padded to the 32-wide tile
    (2, 45, 320, 12, 3, O.BF16),       # expert count not a multiple of 8: element-wise staging
    (3, 31, 72, 8, 1, O.BF16),         # D not a multiple of 64
    (2, 50, 256, 64, 2, O.BF16),       # two expert tiles
    (1, 70, 192, 128, 4, O.BF16),      # four expert tiles
    (1, 70, 96, 128, 4, O.F32),
]


@pytest.mark.parametrize("G,S,D,E,k,dtype", GATE_CASES)
def test_gate_topk(K, G, S, D, E, k, dtype):
  rng = np.random.default_rng(G * 1000 + S)
  x = O.cast(rng.standard_normal((G, S, D)), dtype)
  w = O.cast(rng.standard_normal((D, E)) / np.sqrt(D), dtype)
  gates, val, idx = K.gate_topk(to_dev(x, dtype), to_dev(w, dtype), k)
  gates, val, idx = to_np(gates), to_np(val), to_np(idx)
  want = O.router_gates(x, w, dtype)
  # Float part: tolerance stated by the north star (1e-5 fp32, 2e-2 bf16).
  assert_close(gates, want, 1e-5 if dtype == O.F32 else 2e-2, "gates")
  np.testing.assert_allclose(gates.sum(-1), 1.0, atol=1e-5 if dtype == O.F32 else 2e-2)
  # Integer part: the selection is exact given the kernel's own gates.
  want_v, want_i = O.top_k(gates, k)
  np.testing.assert_array_equal(idx, want_i)
  np.testing.assert_array_equal(val, want_v)
  flips = int((O.top_k(want, k)[1] != idx).any(-1).sum())
  print(f"gate_topk {dtype} items={G*S} top-k rows differing from oracle gates: {flips}")
  assert flips <= max(2, G * S // 100)


def test_gate_topk_logit_bias(K):
  rng = np.random.default_rng(5)
  G, S, D, E = 2, 40, 256, 32
  x = O.cast(rng.standard_normal((G, S, D)), O.BF16)
  w = O.cast(rng.standard_normal((D, E)) / np.sqrt(D), O.BF16)
  b = (rng.standard_normal(E) * 2).astype(np.float32)
  gates, _, _ = K.gate_topk(to_dev(x, O.BF16), to_dev(w, O.BF16), 2, logit_bias=to_dev(b))
  assert_close(to_np(gates), O.router_gates(x, w, O.BF16, b), 2e-2, "gates with bias")


@pytest.mark.parametrize("n,D,E", [(1568, 512, 8), (45, 64, 5), (4100, 384, 32), (33, 1024, 24),
                                   (8200, 64, 16), (16400, 36, 5), (33000, 32, 32)])      # 1, 2, 4 and 8 tiles a workgroup
def test_gate_topk_float32_split_k_form(K, n, D, E):
  """float32 gating deals the k range of a tile to the waves that share it, fewer the more tiles there
  are (partial logits added in wave order): the 64-bit logits bit for bit on operands whose partial sums are
  exact, within float32 rounding otherwise; logits output and logit bias included."""
  rng = np.random.default_rng(n + D)
  xi = rng.integers(-2, 3, (1, n, D)).astype(np.float32)
  wi = rng.integers(-2, 3, (D, E)).astype(np.float32) / 64
  b = (rng.integers(-8, 9, E) / 4).astype(np.float32)
  xr = rng.standard_normal((1, n, D)).astype(np.float32)
  wr = (rng.standard_normal((D, E)) / np.sqrt(D)).astype(np.float32)
  for x, w, exact in ((xi, wi, True), (xr, wr, False)):
    gates, val, idx, logits = K.gate_topk(to_dev(x), to_dev(w), 2, logit_bias=to_dev(b), return_logits=True)
    g_n, v_n, i_n = K.gate_topk(to_dev(x), to_dev(w), 2, logit_bias=to_dev(b))
    g_p, v_p, i_p = K.gate_topk(to_dev(x), to_dev(w), 2)
    want = x[0].astype(np.float64) @ w.astype(np.float64) + b
    if exact:
      np.testing.assert_array_equal(to_np(logits)[0], want)
    else:
      np.testing.assert_allclose(to_np(logits)[0], want, rtol=1e-5, atol=1e-5)
    assert_close(to_np(gates), O.router_gates(x, w, O.F32, b), 1e-5, "gates")
    assert_close(to_np(g_p), O.router_gates(x, w, O.F32), 1e-5, "gates without bias")
    for with_logits, without in ((gates, g_n), (val, v_n), (idx, i_n)):
      np.testing.assert_array_equal(to_np(with_logits), to_np(without))
    for g, v, i in ((gates, val, idx), (g_p, v_p, i_p)):
      want_v, want_i = O.top_k(to_np(g), 2)
      np.testing.assert_array_equal(to_np(i), want_i)
      np.testing.assert_array_equal(to_np(v), want_v)


@pytest.mark.parametrize("n,D,E,k", [(1, 64, 8, 8), (31, 128, 16, 1), (32, 192, 32, 2), (33, 768, 24, 3),
                                     (1568, 768, 32, 2), (196, 1024, 8, 2), (65, 1088, 32, 2),
                                     (97, 2112, 8, 1), (255 * 32, 768, 32, 2), (255 * 32 + 1, 768, 32, 2)])
def test_gate_topk_bf16_split_k_form(K, monkeypatch, n, D, E, k):
  """bfloat16 gating over fewer tiles of 32 items than CUs deals k to the waves of a tile's workgroup
  in slices of 128 (one slice, a half one, exactly one round of eight, more): against the oracle, and
  against the direct loads (VMOE_GATE_DIRECT_LOADS=1) bit for bit where every partial sum is exact."""
  rng = np.random.default_rng(n + D)
  xi = rng.integers(-2, 3, (1, n, D)).astype(np.float32)          # exact in bfloat16, sums below 2^24
  wi = rng.integers(-2, 3, (D, E)).astype(np.float32) / 64
  b = (rng.integers(-8, 9, E) / 4).astype(np.float32)
  xr = O.cast(rng.standard_normal((1, n, D)), O.BF16)
  wr = O.cast(rng.standard_normal((D, E)) / np.sqrt(D), O.BF16)
  for x, w, exact in ((xi, wi, True), (xr, wr, False)):
    xd, wd = to_dev(x, O.BF16), to_dev(w, O.BF16)
    g_s, v_s, i_s = K.gate_topk(xd, wd, k, logit_bias=to_dev(b))
    _, v_n, i_n = K.gate_topk(xd, wd, k, logit_bias=to_dev(b), return_gates=False)
    g_p, _, _ = K.gate_topk(xd, wd, k)
    monkeypatch.setenv("VMOE_GATE_DIRECT_LOADS", "1")
    g_d, v_d, i_d = K.gate_topk(xd, wd, k, logit_bias=to_dev(b))
    monkeypatch.delenv("VMOE_GATE_DIRECT_LOADS")
    np.testing.assert_array_equal(to_np(i_s), to_np(i_n))
    np.testing.assert_array_equal(to_np(v_s), to_np(v_n))
    want_v, want_i = O.top_k(to_np(g_s), k)
    np.testing.assert_array_equal(to_np(i_s), want_i)
    np.testing.assert_array_equal(to_np(v_s), want_v)
    # (2e-2 as above: one rounding of a bfloat16 logit)
    assert_close(to_np(g_s), O.router_gates(x, w, O.BF16, b), 2e-2, "gates")
    assert_close(to_np(g_p), O.router_gates(x, w, O.BF16), 2e-2, "gates without bias")
    if exact:
      np.testing.assert_array_equal(to_np(g_s), to_np(g_d))
      np.testing.assert_array_equal(to_np(i_s), to_np(i_d))
      np.testing.assert_array_equal(to_np(v_s), to_np(v_d))


@pytest.mark.parametrize("n,D,E,k,aligned", [
    (1, 8, 1, 1, True), (31, 72, 5, 2, True), (33, 264, 12, 3, True), (300, 768, 7, 2, True),
    (64, 1024, 33, 4, True), (65, 2056, 64, 2, True), (40, 832, 50, 2, True), (255 * 32, 64, 32, 2, False),
    (255 * 32 + 1, 64, 12, 2, True), (8200, 320, 31, 2, True), (8200, 768, 16, 2, False), (8193, 96, 40, 4, True)])
def test_gate_topk_bf16_any_expert_count(K, monkeypatch, n, D, E, k, aligned):
  """bfloat16 gating with router kernels that do not come in aligned blocks of 8 x 8, with more than 32
  experts or with widths that end inside a chunk: a workgroup per tile (fewer than 256 tiles of 32 items, k in
  one chunk or several), the streaming form and the direct loads add in the same order, so
  VMOE_GATE_DIRECT_LOADS=1 gives the same bits, with and without logits, bias and gates."""
  rng = np.random.default_rng(n + E)
  x = to_dev(O.cast(rng.standard_normal((1, n, D)), O.BF16), O.BF16)
  w = to_dev(O.cast(rng.standard_normal(D * E + 1) / np.sqrt(D), O.BF16), O.BF16)
  w = w[:-1].view(D, E) if aligned else w[1:].view(D, E)
  b = to_dev(rng.standard_normal(E).astype(np.float32))
  calls = [dict(return_logits=True), dict(logit_bias=b, return_logits=True), dict(logit_bias=b), dict(return_gates=False)]
  got = [K.gate_topk(x, w, k, **c) for c in calls]
  monkeypatch.setenv("VMOE_GATE_DIRECT_LOADS", "1")
  want = [K.gate_topk(x, w, k, **c) for c in calls]
  # (E % 8 == 0 on aligned router kernels without logits takes the forms that deal k in another order)
  other = aligned and E % 8 == 0 and E <= 32 and D % 64 == 0
  for c, g, r in zip(calls, got, want):
    for a, e in zip(g, r):
      if a is not None and not (other and "return_logits" not in c):
        np.testing.assert_array_equal(to_np(a), to_np(e), err_msg=str(c))
  want_v, want_i = O.top_k(to_np(got[0][0]), k)
  np.testing.assert_array_equal(to_np(got[0][2]), want_i)
  np.testing.assert_array_equal(to_np(got[0][1]), want_v)
  assert_close(to_np(got[0][0]), O.router_gates(to_np(x), to_np(w), O.BF16), 2e-2, "gates")


@pytest.mark.parametrize("n,D,E,k,aligned", [
    (1, 4, 1, 1, True), (33, 36, 5, 3, True), (100, 832, 38, 2, True), (8200, 544, 6, 1, True), (8193, 100, 33, 4, True),
    (45, 1028, 128, 4, True), (45, 260, 100, 2, False), (257 * 32, 64, 64, 2, True), (96, 2080, 32, 2, False),
    (16400, 132, 12, 2, True), (33000, 64, 16, 2, True), (32800, 64, 60, 2, True)])
def test_gate_topk_float32_any_expert_count(K, n, D, E, k, aligned):
  """float32 gating: one to eight tiles per workgroup, the router kernel in one chunk of rows or several,
  any number of experts, router kernels at any float address, widths that end inside a step of k."""
  rng = np.random.default_rng(n + E)
  x = rng.standard_normal((1, n, D)).astype(np.float32)
  w = (rng.standard_normal(D * E + 1) / np.sqrt(D)).astype(np.float32)
  wd = to_dev(w)
  w, wd = (w[:-1], wd[:-1]) if aligned else (w[1:], wd[1:])
  w, wd = w.reshape(D, E), wd.view(D, E)
  b = rng.standard_normal(E).astype(np.float32)
  for bias in (None, b):
    gates, val, idx, logits = K.gate_topk(to_dev(x), wd, k, logit_bias=None if bias is None else to_dev(bias),
                                          return_logits=True)
    exact = x[0].astype(np.float64) @ w.astype(np.float64) + (0 if bias is None else bias)
    np.testing.assert_allclose(to_np(logits)[0], exact, rtol=1e-5, atol=1e-5)
    assert_close(to_np(gates), O.router_gates(x, w, O.F32, bias), 1e-5, "gates")
    want_v, want_i = O.top_k(to_np(gates), k)
    np.testing.assert_array_equal(to_np(idx), want_i)
    np.testing.assert_array_equal(to_np(val), want_v)
    g2, v2, i2 = K.gate_topk(to_dev(x), wd, k, logit_bias=None if bias is None else to_dev(bias))
    for a, e in ((g2, gates), (v2, val), (i2, idx)):
      np.testing.assert_array_equal(to_np(a), to_np(e))


@pytest.mark.parametrize("n,D,E", [(4096, 768, 8), (20000, 384, 16), (900, 512, 32), (777, 832, 51), (6000, 1024, 128)])
@pytest.mark.parametrize("features", [2, 8, None])
def test_gate_topk_float32_keeps_float32_precision(K, n, D, E, features):
  """Logits of items with a few non-zero features, where every product's last bits show, and of dense ones: no
  further from 64 bits (2-norm) than a chain of float32 multiply-adds with two roundings more (where the waves'
  partial sums meet, and where the sums of large and small products do; the error grows as the root of their number)."""
  gen = torch.Generator(device=dev()).manual_seed(n + (features or 0))
  x = torch.randn((n, D), generator=gen, device=dev())
  w = torch.randn((D, E), generator=gen, device=dev()) * D ** -0.5
  order = torch.arange(D, device=dev()).expand(n, D)
  if features is not None:
    order = torch.rand((n, D), generator=gen, device=dev()).argsort(-1)[:, :features].sort(-1).values
    x = torch.zeros_like(x).scatter_(1, order, x.gather(1, order))
  exact = x.double() @ w.double()
  chain = torch.zeros((n, E), device=dev())
  for i in range(order.shape[1]):
    k = order[:, i]
    chain = (chain.double() + x.gather(1, k[:, None]).double() * w[k].double()).float()
  off = lambda a: ((a.double() - exact).norm() / exact.norm()).item()
  assert off(K.gate_topk(x[None], w, 1, return_logits=True)[3][0]) <= (1 + 2 / order.shape[1]) ** 0.5 * off(chain)


@pytest.mark.parametrize("n,D,E", [(45, 260, 7), (8200, 64, 16), (16400, 36, 5), (33000, 32, 32), (70, 516, 40),
                                   (33000, 64, 33), (50, 100, 100), (33000, 36, 128)])
@pytest.mark.parametrize("bias", [None, "finite", "infinite"])
def test_gate_topk_float32_infinities(K, n, D, E, bias):
  """Infinite and NaN items, an infinite router column and values that round to infinity in bfloat16 give the
  logits of float32 multiplication, at every number of tiles per workgroup; the other items' are bit for bit what
  they are without them.  A bias of -inf takes its expert out."""
  rng = np.random.default_rng(n + E)
  x = rng.standard_normal((1, n, D)).astype(np.float32)
  w = (rng.standard_normal((D, E)) / np.sqrt(D)).astype(np.float32)
  b = rng.standard_normal(E).astype(np.float32)
  if bias == "infinite":
    b[E // 2] = -np.inf
  b = None if bias is None else b
  run = lambda x, w: K.gate_topk(to_dev(x), to_dev(w), 1, logit_bias=None if b is None else to_dev(b), return_logits=True)
  clean = to_np(run(x, w)[3])[0]
  odd, rows = x.copy(), [0, 3, n // 2, n - 1]
  odd[0, 0, 0], odd[0, 3, D - 1], odd[0, n // 2, 1], odd[0, n - 1, 2] = np.inf, -np.inf, np.nan, 3.4e38
  with np.errstate(over="ignore", invalid="ignore"):
    want = odd[0, rows].astype(np.float64) @ w.astype(np.float64) + (0 if b is None else b)
  want = np.where(np.abs(want) > np.finfo(np.float32).max, np.sign(want) * np.inf, want)
  gates, _, _, logits = (to_np(t) for t in run(odd, w))
  got = logits[0, rows]
  np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
  np.testing.assert_array_equal(np.where(np.isinf(got), got, 0), np.where(np.isinf(want), want, 0))
  np.testing.assert_allclose(got[np.isfinite(want)], want[np.isfinite(want)], rtol=1e-5)
  same = np.ones(n, bool)
  same[rows] = False
  np.testing.assert_array_equal(logits[0, same], clean[same])
  assert np.isfinite(gates[0, same]).all() and (bias != "infinite" or (gates[0, same, E // 2] == 0).all())
  # A router column of infinities: its logits are infinite, the others untouched.
  if E > 1 and bias != "infinite":
    column = w.copy()
    column[D // 2, E - 1] = -np.inf
    gates, _, _, logits = (to_np(t)[0] for t in run(x, column))
    np.testing.assert_array_equal(logits[:, E - 1], np.where(x[0, :, D // 2] > 0, -np.inf, np.inf))
    np.testing.assert_array_equal(logits[:, :-1], clean[:, :-1])
    out = x[0, :, D // 2] > 0
    assert (gates[out, E - 1] == 0).all() and np.isfinite(gates[out]).all()


def test_gate_topk_streaming_and_direct_loads_agree(K, monkeypatch):
  """The two forms of the bfloat16 gating kernel (item rows through LDS by DMA, or by direct
  loads: VMOE_GATE_DIRECT_LOADS=1) add the same products in a different order of k: equal
  bit for bit where every partial sum is exact, within a few bfloat16 steps otherwise; the
  logit bias and a call without the gates output take the streaming form too."""
  rng = np.random.default_rng(11)
  n, D, E = 8192 + 40, 768, 32
  xi = rng.integers(-2, 3, (1, n, D)).astype(np.float32)          # exact in bfloat16, sums below 2^24
  wi = rng.integers(-2, 3, (D, E)).astype(np.float32) / 64
  b = (rng.integers(-8, 9, E) / 4).astype(np.float32)
  xr = O.cast(rng.standard_normal((1, n, D)), O.BF16)
  wr = O.cast(rng.standard_normal((D, E)) / np.sqrt(D), O.BF16)
  for x, w, exact in ((xi, wi, True), (xr, wr, False)):
    monkeypatch.delenv("VMOE_GATE_DIRECT_LOADS", raising=False)
    g_s, v_s, i_s = K.gate_topk(to_dev(x, O.BF16), to_dev(w, O.BF16), 2, logit_bias=to_dev(b))
    _, v_n, i_n = K.gate_topk(to_dev(x, O.BF16), to_dev(w, O.BF16), 2, logit_bias=to_dev(b), return_gates=False)
    monkeypatch.setenv("VMOE_GATE_DIRECT_LOADS", "1")
    g_d, v_d, i_d = K.gate_topk(to_dev(x, O.BF16), to_dev(w, O.BF16), 2, logit_bias=to_dev(b))
    monkeypatch.delenv("VMOE_GATE_DIRECT_LOADS")
    np.testing.assert_array_equal(to_np(i_s), to_np(i_n))
    np.testing.assert_array_equal(to_np(v_s), to_np(v_n))
    if exact:
      np.testing.assert_array_equal(to_np(g_s), to_np(g_d))
      np.testing.assert_array_equal(to_np(i_s), to_np(i_d))
      np.testing.assert_array_equal(to_np(v_s), to_np(v_d))
      assert_close(to_np(g_s), O.router_gates(x, w, O.BF16, b), 2e-2, "gates")
    else:
      gs, gd = to_np(g_s).astype(np.float64), to_np(g_d).astype(np.float64)
      # (a logit of magnitude 2 .. 4 that rounds the other way moves by 2^-6, its gate by
      # 1.6 %, and the other gates of the item through the sum)
      assert np.all(np.abs(gs - gd) <= 2.0 ** -5 * np.maximum(np.abs(gs), np.abs(gd)) + 1e-30)
      assert float((gs != gd).mean()) < 0.05
      assert int((to_np(i_s) != to_np(i_d)).any(-1).sum()) <= n // 100


def test_router_metrics(K, goldens):
  g = goldens["router_aux_losses"]
  gates = np.asarray(g["gates"], np.float32)[None]
  _, idx = K.topk(to_dev(gates), 1)
  imp, gsh, aux = K.router_metrics(to_dev(gates), idx, 0.0, 1.0)
  assert float(gsh[0]) == pytest.approx(g["gshard"], abs=1e-6)
  assert float(imp[0]) == pytest.approx(g["importance"], abs=1e-6)
  assert float(aux[0]) == pytest.approx(g["importance"], abs=1e-6)
  rng = np.random.default_rng(1)
  for (G, S, E) in [(4, 1568, 32), (3, 49, 8), (2, 100, 300)]:
    gt = O.softmax(rng.standard_normal((G, S, E)).astype(np.float32) * 2)
    _, idx = K.topk(to_dev(gt), 2)
    imp, gsh, aux = K.router_metrics(to_dev(gt), idx, 0.5, 2.0)
    want = O.router_metrics(gt, 0.5, 2.0)
    np.testing.assert_allclose(to_np(imp), want["importance_loss"], rtol=1e-4)
    np.testing.assert_allclose(to_np(gsh), want["gshard_loss"], rtol=1e-4)
    np.testing.assert_allclose(to_np(aux), want["auxiliary_loss"], rtol=1e-4)


# ------------------------------------------------------------------ slot assignment
ROUTE_CASES = [
    # G, S, E, K, C, ties
    (1, 3, 3, 2, 2, False),
    (2, 49, 8, 2, 16, False),
    (4, 64, 8, 2, 4, True),
    (3, 100, 5, 3, 7, True),
    (32, 1568, 32, 2, 100, False),   # B/16 layer
    (16, 2304, 32, 2, 72, False),    # L/16@384, heavy dropping
    (8, 1568, 8, 2, 412, False),     # full-model layer
    (2, 1568, 32, 2, 100, True),
    (2, 513, 7, 1, 30, True),
    (1, 1, 2, 2, 1, False),
    (2, 1024, 8, 2, 100, True),      # one key per thread, lane and LDS exchanges
    (3, 1025, 4, 1, 300, False),     # two keys per thread
    (2, 2304, 32, 2, 72, True),      # four
    (1, 5000, 4, 2, 700, True),      # eight
    (2, 2900, 6, 3, 1100, False),    # 8 700 choices: more than the 8 192 held in registers
]


@pytest.mark.parametrize("bpr", [False, True])
@pytest.mark.parametrize("G,S,E,k,C,ties", ROUTE_CASES)
def test_route_assign_bit_exact(K, G, S, E, k, C, ties, bpr):
  rng = np.random.default_rng(S * 7 + E)
  if ties:   # bf16-like coarse gates: many equal first-choice gates
    gates = O.bf16_round(O.softmax(rng.integers(-3, 4, (G, S, E)).astype(np.float32)))
  else:
    gates = O.softmax(rng.standard_normal((G, S, E)).astype(np.float32) * 2)
  val, idx = K.topk(to_dev(gates), k)
  indices, token_slot, slot_token, fill = K.route_assign(val, idx, E, C, bpr)
  indices, token_slot, slot_token, fill = map(to_np, (indices, token_slot, slot_token, fill))
  want_idx, want_w = route_c.route_batch(gates, k, bpr)
  np.testing.assert_array_equal(indices, want_idx)
  np.testing.assert_array_equal(to_np(val), want_w)
  if G * S <= 20000:   # the literal one-hot/cumsum restatement on the smaller cases
    d = O.get_top_experts_per_item_dispatcher(gates, "indices", k, bpr, capacity=C)
    np.testing.assert_array_equal(indices, d.indices)
  # Derived maps.
  e, p = want_idx[..., 0], want_idx[..., 1]
  kept = p < C
  gi = np.arange(G)[:, None, None]
  if G % E == 0:
    q = G // E
    row = ((gi % q) * E + gi // q) * C + p
  else:
    row = gi * C + p
  want_slot = np.where(kept, e * (G * C) + row, -1)
  np.testing.assert_array_equal(token_slot, want_slot)
  want_st = np.full(E * G * C, -1, np.int32)
  item = (np.arange(G * S).reshape(G, S, 1) + np.zeros((1, 1, k), np.int64))
  want_st[want_slot[kept]] = item[kept]
  np.testing.assert_array_equal(slot_token, want_st)
  demand = np.stack([np.bincount(e[g].ravel(), minlength=E) for g in range(G)])
  np.testing.assert_array_equal(fill, np.minimum(demand, C))


@pytest.mark.parametrize("bpr", [False, True])
@pytest.mark.parametrize("G,S,E,k,C,dtype", [(4, 64, 8, 2, 4, O.F32), (32, 1568, 32, 2, 100, O.BF16),
                                             (3, 100, 5, 3, 7, O.F32), (2, 2304, 32, 2, 72, O.BF16),
                                             (2, 50, 100, 2, 3, O.F32)])
def test_route_assign_with_metrics_equals_separate_calls(K, G, S, E, k, C, dtype, bpr):
  """One launch for slot assignment and the router's losses: every output has the bits
  of the two separate entry points."""
  rng = np.random.default_rng(S + E)
  gates = to_dev(O.cast(O.softmax(rng.standard_normal((G, S, E)).astype(np.float32) * 2), dtype), dtype)
  val, idx = K.topk(gates.float(), k)
  want = K.route_assign(val, idx, E, C, bpr)
  want_losses = K.router_metrics(gates, idx, 0.25, 1.0)
  got = K.route_assign(val, idx, E, C, bpr, metrics=(gates, 0.25, 1.0))
  for a, b in zip(got[:4], want):
    assert torch.equal(a, b)
  for a, b in zip(got[4], want_losses):
    assert torch.equal(a, b)


def test_route_assign_random_shapes(K):
  """Seeded sweep over group sizes around the sort's switch points (keys per thread,
  partial waves), expert counts, gate flavours (float32, bfloat16-valued -> 32-bit sort
  keys, coarse values with many ties, negative and zero gates) against the sequential
  C statement of the assignment."""
  rng = np.random.default_rng(2024)
  sizes = [1, 2, 3, 31, 32, 33, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513, 1000,
           1023, 1024, 1025, 1500, 2047, 2048, 2049, 3000, 4095, 4096, 4097]
  for case, S in enumerate(sizes * 2):
    E = int(rng.integers(1, 41))
    k = int(rng.integers(1, min(E, 4) + 1))
    G = int(rng.integers(1, 4))
    C = int(rng.integers(1, max(2, (S * k) // E + 3)))
    flavour = case % 4
    pow2 = 1 << max(0, (S - 1).bit_length())
    keys = 8 * max(pow2, (2 * 1024 + S + 1) // 2)   # sort keys, or the counting rank's two 1 024-word arrays and S items
    lds = keys + 8 * E * ((S * k + 31) // 32) + 4 * S + 4 * E
    if lds > 160 * 1024:      # the entry point's documented limit: such shapes are refused
      E = max(k, (160 * 1024 - keys - 4 * S) // (8 * ((S * k + 31) // 32) + 4) - 1)
    logits = rng.standard_normal((G, S, E)).astype(np.float32) * 2
    if flavour == 0:
      gates = O.softmax(logits)
    elif flavour == 1:
      gates = O.bf16_round(O.softmax(logits))
    elif flavour == 2:
      gates = O.bf16_round(O.softmax(np.round(logits)))      # many equal gates
    else:
      gates = np.round(logits * 2).astype(np.float32) / 4       # negative, zero and tied "gates"
    val, idx = K.topk(to_dev(gates), k)
    got, _, _, fill = K.route_assign(val, idx, E, C, True)
    want, want_w = route_c.route_batch(gates, k, True)
    np.testing.assert_array_equal(to_np(got), want, err_msg=f"S={S} E={E} k={k} G={G} C={C} flavour={flavour}")
    np.testing.assert_array_equal(to_np(val), want_w)
    e = want[..., 0]
    demand = np.stack([np.bincount(e[g].ravel(), minlength=E) for g in range(G)])
    np.testing.assert_array_equal(to_np(fill), np.minimum(demand, C))


def test_route_assign_golden(K, goldens):
  g = goldens["top_experts_per_item"]
  gates = np.asarray(g["gates"], np.float32)[None]
  val, idx = K.topk(to_dev(gates), 2)
  for bpr, key in ((False, "vanilla"), (True, "bpr")):
    indices, *_ = K.route_assign(val, idx, 3, g["capacity"], bpr)
    np.testing.assert_array_equal(to_np(indices)[0], np.asarray(g["indices"][key]))
    cw, dw = K.densify(indices, val, 3, g["capacity"])
    np.testing.assert_array_almost_equal(to_np(cw)[0], np.asarray(g["einsum_combine_weights"][key]))
    np.testing.assert_array_equal(to_np(dw)[0], np.asarray(g["einsum_combine_weights"][key]) > 0)
  np.testing.assert_array_almost_equal(to_np(val)[0], np.asarray(g["indices_combine_weights"]))


# ------------------------------------------------------------------ dispatch / combine
@pytest.mark.parametrize("case", ["dispatcher_experts_divide_groups",
                                  "dispatcher_groups_divide_experts"])
def test_dispatch_combine_golden(K, goldens, case):
  g = goldens[case]
  E, C = g["num_experts"], g["capacity"]
  data = np.asarray(goldens["dispatcher_data"]["data"], np.float32)
  idx = to_dev(np.asarray(g["indices"], np.int32))
  w = np.tile(np.asarray(g["indices_combine_weights_tile"], np.float32)[None, None], (2, 3, 1))
  token_slot, slot_token, counters = K.indices_to_slots(idx, E, C)
  assert to_np(counters).tolist() == [0, 0]
  buf = K.dispatch(to_dev(data.reshape(6, 4)), token_slot.view(6, 2), slot_token)
  np.testing.assert_array_equal(to_np(buf).reshape(E, 2 * C, 4), np.asarray(g["expected_dispatch"]))
  out = K.combine(buf, token_slot.view(6, 2), to_dev(w.reshape(6, 2)))
  np.testing.assert_array_almost_equal(to_np(out).reshape(2, 3, 4), np.asarray(g["expected_combine"]))


def test_indices_to_slots_flags_duplicates_and_negatives(K):
  idx = np.asarray([[[[0, 0]], [[0, 0]], [[-1, 0]]]], np.int32)   # G=1,S=3,K=1
  _, _, counters = K.indices_to_slots(to_dev(idx), 2, 2)
  assert to_np(counters).tolist() == [1, 1]


MOVE_CASES = [
    # G, S, E, K, C, D, dtype
    (2, 49, 8, 2, 16, 512, O.F32),
    (4, 33, 8, 2, 4, 64, O.F32),      # G/E not integral -> swapaxes branch
    (8, 64, 4, 2, 20, 256, O.BF16),   # G/E = 2 -> permuted branch
    (3, 50, 6, 3, 9, 72, O.BF16),
    (4, 1568, 32, 2, 100, 768, O.BF16),
    (2, 2304, 32, 2, 72, 1024, O.BF16),
]


@pytest.mark.parametrize("G,S,E,k,C,D,dtype", MOVE_CASES)
def test_dispatch_combine_bit_exact(K, G, S, E, k, C, D, dtype):
  rng = np.random.default_rng(D + S)
  gates = O.cast(O.softmax(rng.standard_normal((G, S, E)).astype(np.float32) * 2), dtype)
  x = O.cast(rng.standard_normal((G, S, D)), dtype)
  d = O.get_top_experts_per_item_dispatcher(gates, "indices", k, True, capacity=C)
  val, idx = K.topk(to_dev(gates), k)
  indices, token_slot, slot_token, _ = K.route_assign(val, idx, E, C, True)
  np.testing.assert_array_equal(to_np(indices), d.indices)
  buf = K.dispatch(to_dev(x, dtype).view(G * S, D), token_slot.view(G * S, k), slot_token)
  want_buf = d.dispatch(x)
  np.testing.assert_array_equal(to_np(buf).reshape(E, G * C, D), want_buf)
  y = O.cast(rng.standard_normal((E, G * C, D)), dtype)
  out = K.combine(to_dev(y, dtype).view(E * G * C, D), token_slot.view(G * S, k), val.view(G * S, k))
  want = O.cast(d.combine(y), dtype)
  np.testing.assert_array_equal(to_np(out).reshape(G, S, D), want)
  # Idempotence / determinism: a second run gives the same bits.
  buf2 = K.dispatch(to_dev(x, dtype).view(G * S, D), token_slot.view(G * S, k), slot_token)
  assert torch.equal(buf, buf2)


def test_dispatch_combine_round_trip_full_size(K):
  """B/16 layer size: combine(dispatch(x)) with unit weights returns x times the
  number of kept assignments of each item (size-independent property)."""
  G, S, E, k, C, D = 32, 1568, 32, 2, 100, 768
  gen = torch.Generator(device="cpu").manual_seed(0)
  gates = torch.softmax(torch.randn((G, S, E), generator=gen) * 2, -1).to(dev())
  x = torch.randn((G * S, D), generator=gen).to(torch.bfloat16).to(dev())
  val, idx = K.topk(gates, k)
  indices, token_slot, slot_token, fill = K.route_assign(val, idx, E, C, True)
  buf = K.dispatch(x, token_slot.view(G * S, k), slot_token)
  ones = torch.ones((G * S, k), dtype=torch.float32, device=dev())
  out = K.combine(buf, token_slot.view(G * S, k), ones)
  kept = (token_slot.view(G * S, k) >= 0).sum(-1, keepdim=True).to(torch.float32)
  want = (x.to(torch.float32) * kept).to(torch.bfloat16)
  assert torch.equal(out, want)
  # Every slot is either an exact copy of its item or zero; fill matches occupancy.
  st = slot_token.view(E, -1)
  assert int((st >= 0).sum()) == int(fill.sum())
  empty = (slot_token < 0)
  assert float(buf[empty].abs().max() if empty.any() else 0.0) == 0.0


# ------------------------------------------------------------------ expert MLP
MLP_CASES = [
    # E, R, D, M, dtype
    (2, 40, 64, 128, O.F32),
    (8, 512, 512, 2048, O.F32),       # S/32-style layer, full size
    (3, 100, 96, 200, O.F32),         # column tile that ends inside the matrix; second product's k not whole tiles
    (3, 100, 96, 160, O.F32),         # both products through the LDS-DMA kernel, ragged rows and columns
    (3, 100, 72, 136, O.BF16),        # ragged everything
    (2, 300, 256, 512, O.BF16),
    (3, 300, 64, 192, O.BF16),        # shortest second product the tile-walking kernel takes (6 k tiles)
    (4, 3200, 768, 3072, O.BF16),     # B/16 experts (4 of 32)
]


@pytest.mark.parametrize("prepacked", [False, True])
@pytest.mark.parametrize("E,R,D,M,dtype", MLP_CASES)
def test_expert_mlp(K, E, R, D, M, dtype, prepacked):
  if prepacked and dtype == O.F32:
    pytest.skip("float32 path reads the reference layout directly")
  rng = np.random.default_rng(R)
  x = O.cast(rng.standard_normal((E, R, D)), dtype)
  w0 = O.cast(rng.standard_normal((E, D, M)) / np.sqrt(D), dtype)
  b0 = O.cast(rng.standard_normal((E, M)) * 0.1, dtype)
  w1 = O.cast(rng.standard_normal((E, M, D)) / np.sqrt(M), dtype)
  b1 = O.cast(rng.standard_normal((E, D)) * 0.1, dtype)
  dx, dw0, db0, dw1, db1 = (to_dev(a, dtype) for a in (x, w0, b0, w1, b1))
  kw = {}
  if prepacked:
    kw = dict(w0t=K.pack_expert_weights(dw0), w1t=K.pack_expert_weights(dw1))
    np.testing.assert_array_equal(to_np(kw["w0t"]), w0.transpose(0, 2, 1))
  out = to_np(K.expert_mlp(dx, dw0, db0, dw1, db1, **kw))
  want = O.mlp_block(x, w0, b0, w1, b1, dtype)
  assert_close(out, want, 1e-5 if dtype == O.F32 else 2e-2, "expert mlp")


def test_expert_mlp_erf_gelu_and_no_bias(K):
  rng = np.random.default_rng(9)
  E, R, D, M = 2, 64, 64, 128
  x = rng.standard_normal((E, R, D)).astype(np.float32)
  w0 = (rng.standard_normal((E, D, M)) / 8).astype(np.float32)
  w1 = (rng.standard_normal((E, M, D)) / 11).astype(np.float32)
  out = to_np(K.expert_mlp(to_dev(x), to_dev(w0), None, to_dev(w1), None, approximate_gelu=False))
  assert_close(out, O.mlp_block(x, w0, None, w1, None, O.F32, approximate_gelu=False), 1e-5, "erf")


# ------------------------------------------------------------------ error handling
def test_bad_arguments_return_error_codes(K):
  from vmoe_amd import _hip as H
  x = torch.randn((1, 4, 12), device=dev()).to(torch.bfloat16)       # D % 8 != 0
  w = torch.randn((12, 4), device=dev()).to(torch.bfloat16)
  val = torch.empty((4, 2), dtype=torch.float32, device=dev())
  idx = torch.empty((4, 2), dtype=torch.int32, device=dev())
  with pytest.raises(H.VmoeError, match="aligned"):                  # the C ABI refuses the width
    H.call("vmoe_gate_topk", H.GateTopkParams(H.ptr(x), H.ptr(w), None, None, H.ptr(val),
                                              H.ptr(idx), 4, 12, 4, 2, H.BF16, None))
  gates, _, _ = K.gate_topk(x, w, 2)                                 # the wrapper pads with zeros
  want = torch.softmax((x.float() @ w.float()).to(torch.bfloat16).float(), -1)
  np.testing.assert_allclose(to_np(gates), to_np(want), rtol=1e-2, atol=1e-3)
  x = torch.zeros((1, 4, 16), dtype=torch.float32, device=dev())
  w = torch.zeros((16, 4), dtype=torch.float32, device=dev())
  with pytest.raises(H.VmoeError, match="invalid sizes"):
    K.gate_topk(x, w, 5)                                             # K > E
  with pytest.raises(H.VmoeError, match="no CPU fallback"):
    K.gate_topk(x.cpu(), w.cpu(), 2)
  with pytest.raises(TypeError):
    K.gate_topk(x.double(), w.double(), 2)
  idx = torch.zeros((1, 4, 2), dtype=torch.int32, device=dev())
  with pytest.raises(H.VmoeError, match="invalid sizes"):
    K.route_assign(None, idx, 1, 4, False)                           # K > E
  with pytest.raises(H.VmoeError, match="null"):
    K.route_assign(None, idx, 4, 4, True)                            # BPR needs the gates


# ------------------------------------------------------------------ Soft MoE
SOFT_CASES = [
    # G, S, D, n, p, dtype
    (1, 8, 16, 5, 2, O.F32),
    (3, 50, 64, 7, 3, O.F32),
    (2, 196, 768, 128, 1, O.BF16),
    (4, 100, 256, 16, 2, O.BF16),
    (1, 2, 16, 4, 2, O.F32),          # inputs smaller than mu: the scale multiplies the inputs
    # every model width of the two-role bf16 kernel and one more, ragged S and N
    (3, 77, 384, 24, 1, O.BF16),
    (2, 130, 512, 8, 5, O.BF16),
    (2, 33, 1024, 128, 1, O.BF16),
    (1, 300, 256, 104, 1, O.BF16),
    (1, 20, 768, 64, 2, O.BF16),      # inputs smaller than mu on the bf16 path
    (2, 64, 768, 20, 1, O.BF16),      # N % 8 != 0: row tiles
    (2, 64, 320, 16, 1, O.BF16),      # another width: row tiles
    # two-role kernel with 16-row item tiles (two 32-row tiles do not fit LDS beside the
    # logits): dispatch softmax from registers (S <= 256) and in three passes
    (1, 250, 768, 128, 1, O.BF16),
    (2, 260, 768, 128, 1, O.BF16),
]


@pytest.mark.parametrize("G,S,D,n,p,dtype", SOFT_CASES)
def test_soft_route(K, G, S, D, n, p, dtype):
  rng = np.random.default_rng(S + n)
  x = O.cast(rng.standard_normal((G, S, D)), dtype)
  mu = O.cast(rng.standard_normal((D, n, p)) / np.sqrt(D), dtype)
  scale = 1.75
  dw, cw, lg = K.soft_route(to_dev(x, dtype), to_dev(mu.reshape(D, n * p), dtype), scale,
                            return_logits=True)
  wl, wd, wc, _ = O.soft_router_weights(x, mu, scale, dtype)
  tol = 1e-5 if dtype == O.F32 else 2e-2
  assert_close(to_np(lg), wl.reshape(G, S, n * p), tol * (1 if dtype == O.BF16 else 4), "logits")
  assert_close(to_np(dw), wd.reshape(G, S, n * p), tol * 4, "dispatch weights")
  assert_close(to_np(cw), wc.reshape(G, S, n * p), tol * 4, "combine weights")
  _check_soft_weights_against_own_logits(to_np(lg), to_np(dw), to_np(cw), dtype, "")
  atol = 1e-4 if dtype == O.F32 else 3e-2
  np.testing.assert_allclose(to_np(dw).sum(1), 1.0, atol=atol)
  np.testing.assert_allclose(to_np(cw).sum(2), 1.0, atol=atol)


@pytest.mark.parametrize("G,S,D,N,dtype", [
    (3, 65, 64, 256, O.BF16),      # 16-row tiles, one row past the fourth
    (128, 65, 64, 160, O.BF16),    # 64-row tiles
    (256, 33, 1024, 128, O.BF16),  # 32-row tiles, widest model width
    (2, 17, 40, 17, O.BF16),       # slots that are no whole piece, width padded to whole steps
    (1, 1, 8, 1, O.BF16),
    (4, 196, 736, 74, O.BF16),
    (2, 300, 512, 520, O.BF16),    # more logits than a workgroup per group could hold
    (5, 49, 512, 48, O.F32),
    (2, 31, 102, 33, O.F32),       # rows at unaligned addresses
    (3, 130, 960, 74, O.F32),
    (140, 64, 48, 164, O.F32),     # 64-row tiles
    (128, 33, 1096, 24, O.BF16),   # 32-row tiles, rows of three pieces per lane
    (2, 33, 1536, 40, O.BF16),     # 16-row tiles, the same
    (2, 33, 4096, 24, O.BF16),     # the widest rows that tiles take, eight pieces per lane
    (3, 20, 2600, 17, O.BF16),
    (2, 20, 2048, 36, O.F32),
    (2, 33, 1100, 17, O.F32),
    (2, 40, 4104, 20, O.BF16),     # wider than any tile: a workgroup per group
    (3, 37, 2052, 12, O.F32),
    (1, 40, 4096, 1024, O.BF16),   # or more logits beside such rows than LDS holds
])
def test_soft_route_row_tiles(K, G, S, D, N, dtype):
  """Shapes whose routing runs over row tiles (and the widths past them): logits against float64 within the dtype's
  tolerance, both softmaxes against the float64 softmaxes of the returned logits, the monitoring
  sums against the returned weights; with prepared slot parameters bit for bit the same."""
  rng = np.random.default_rng(G * S + N)
  x = O.cast(rng.standard_normal((G, S, D)), dtype)
  mu = O.cast(rng.standard_normal((D, N)) / np.sqrt(D), dtype)
  scale = 1.5
  dw, cw, lg = (to_np(t) for t in K.soft_route(to_dev(x, dtype), to_dev(mu, dtype), scale, return_logits=True))
  x64, mu64 = x.astype(np.float64), mu.astype(np.float64)
  want = np.einsum("gsd,dn->gsn", x64 / np.sqrt((x64 ** 2).sum(-1, keepdims=True) + 1e-6),
                   scale * mu64 / np.sqrt((mu64 ** 2).sum(0) + 1e-6))
  # bfloat16: both operands and the logit are rounded, 2^-9 each, on a sum of unit vectors' products
  assert np.abs(lg - want).max() <= (3 * 2.0 ** -9 * scale if dtype == O.BF16 else 2e-6 * scale)
  _check_soft_weights_against_own_logits(lg, dw, cw, dtype, f"G={G} S={S} D={D} N={N}")
  prepared = {}
  for _ in range(2):
    dw2, cw2, scalars = K.soft_route(to_dev(x, dtype), to_dev(mu, dtype), scale, prepared=prepared, with_stats=True)
    np.testing.assert_array_equal(to_np(dw2), dw)
    np.testing.assert_array_equal(to_np(cw2), cw)
  d, c = dw.astype(np.float64), cw.astype(np.float64)
  np.testing.assert_allclose([float(v) for v in scalars][:4],
                             [c.min(axis=2).mean(), c.max(axis=2).mean(), d.min(axis=1).mean(), d.max(axis=1).mean()],
                             rtol=3e-6)


@pytest.mark.parametrize("G,S,D,N", [(64, 196, 64, 256), (16, 65, 1024, 128), (32, 100, 320, 44)])
def test_soft_route_row_tiles_round_like_float32_softmaxes(K, G, S, D, N):
  """Logits up to about 160 (items near slots, scale 200): both softmaxes take their exponentials and
  quotients in float32, so hardly a bfloat16 weight rounds away from the float64 softmax of the kernel's
  own logits.  Bound: exponential, sum and quotient are within 4 * 2^-24 of a weight together (l - max is
  exact there), and a weight rounds the other way only within that of a rounding boundary, of which there
  is one per 2^-8 of a weight at the densest: 2 * 2^-22 / 2^-8 of the weights.  An exponential that rounds
  max * log2(e) first is off by 2^-18 there, and 3e-4 of the weights of the first shape differ."""
  gen = torch.Generator(device=dev()).manual_seed(D)
  normal = lambda *shape: torch.randn(shape, generator=gen, device=dev())
  mu = (normal(D, N) * D ** -0.5).to(torch.bfloat16)
  near = mu.float().t()[torch.arange(G * S, device=dev()).reshape(G, S) % N]
  x = (near * D ** 0.5 * 0.7 + normal(G, S, D)).to(torch.bfloat16)
  dw, cw, lg = K.soft_route(x, mu, 200.0, return_logits=True)
  assert float(lg.float().max()) > 64
  for got, axis in ((dw, 1), (cw, 2)):
    want = torch.softmax(lg.double(), axis)
    counted = want > 1e-18          # (below, l itself is rounded on the way to l - max)
    share = float((got != want.to(torch.bfloat16))[counted].double().mean())
    assert share <= 2.0 ** -13, (axis, share)


@pytest.mark.parametrize("G,S,D,N,dtype", [(3, 65, 64, 256, O.BF16), (2, 5, 40, 17, O.BF16), (2, 300, 1024, 128, O.BF16),
                                           (2, 31, 100, 33, O.F32)])
def test_soft_route_row_tiles_keep_nan(K, G, S, D, N, dtype):
  """A NaN item: NaN combine weights of that item alone, NaN dispatch weights of every item of its group
  (the softmax over items meets it in every slot), the other groups as without it."""
  rng = np.random.default_rng(S)
  x = O.cast(rng.standard_normal((G, S, D)), dtype)
  mu = to_dev(O.cast(rng.standard_normal((D, N)) / np.sqrt(D), dtype), dtype)
  clean = [to_np(t) for t in K.soft_route(to_dev(x, dtype), mu, 1.0)]
  x[1, S // 2] = np.nan
  dw, cw = (to_np(t) for t in K.soft_route(to_dev(x, dtype), mu, 1.0))
  assert np.isnan(dw[1]).all() and np.isnan(cw[1, S // 2]).all()
  others = np.arange(S) != S // 2
  np.testing.assert_array_equal(cw[1, others], clean[1][1, others])
  for g in set(range(G)) - {1}:
    np.testing.assert_array_equal(dw[g], clean[0][g])
    np.testing.assert_array_equal(cw[g], clean[1][g])


def _check_soft_weights_against_own_logits(lg, dw, cw, dtype, tag):
  """The two softmaxes themselves.  Against the oracle the weights carry the difference of the
  logits (a bfloat16 logit that rounds the other way moves a weight by exp(step) - 1, which is
  why those comparisons are loose); against the float64 softmaxes of the logits that the kernel
  itself returned -- the values its softmaxes start from -- nothing is left but the softmax
  arithmetic and one rounding: two units in the last place of the weights' type (bfloat16: 8
  significant bits; float32: rtol 1e-5 for the float32 exponentials and sums).  A wrong
  denominator, a missing maximum or a softmax over the wrong axis does not pass."""
  lg64 = np.asarray(lg, np.float64)
  for name, got, axis in (("dispatch weights", dw, 1), ("combine weights", cw, 2)):
    e = np.exp(lg64 - lg64.max(axis=axis, keepdims=True))
    want = e / e.sum(axis=axis, keepdims=True)
    got = np.asarray(got, np.float64)
    if dtype == O.BF16:
      allowed = 2.0 ** (np.floor(np.log2(np.maximum(want, 1e-300))) - 7 + 1) + 1e-38
    else:
      allowed = 1e-5 * want + 1e-30
    bad = np.abs(got - want) > allowed
    assert not bad.any(), (f"{name} {tag}: {bad.sum()} of {bad.size} further than two units in the last "
                           f"place from the softmax of the kernel's own logits; worst ratio "
                           f"{float((np.abs(got - want) / allowed).max()):.2f}")


def test_soft_route_seeded_shapes(K):
  """Seeded sweep over the shapes of the bfloat16 fast paths (model widths, N a multiple of 8 up
  to 128, group sizes around the tile heights and around the 256 items that the
  register-resident dispatch softmax holds) against the oracle."""
  rng = np.random.default_rng(2024)
  special_s = [1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 223, 224, 225, 255, 256, 257, 300]
  for trial in range(16):
    D = int(rng.choice([256, 384, 512, 768, 1024]))
    n = int(rng.integers(1, 17)) * 8
    S = int(rng.choice(special_s)) if trial % 2 == 0 else int(rng.integers(1, 320))
    G = int(rng.integers(1, 4))
    x = O.cast(rng.standard_normal((G, S, D)), O.BF16)
    mu = O.cast(rng.standard_normal((D, n, 1)) / np.sqrt(D), O.BF16)
    scale = float(rng.uniform(0.5, 2.0))
    dw, cw, lg = K.soft_route(to_dev(x, O.BF16), to_dev(mu.reshape(D, n), O.BF16), scale,
                              return_logits=True)
    wl, wd, wc, _ = O.soft_router_weights(x, mu, scale, O.BF16)
    tag = f"G={G} S={S} D={D} N={n}"
    assert_close(to_np(lg), wl.reshape(G, S, n), 2e-2, "logits " + tag)
    assert_close(to_np(dw), wd.reshape(G, S, n), 8e-2, "dispatch weights " + tag)
    assert_close(to_np(cw), wc.reshape(G, S, n), 8e-2, "combine weights " + tag)
    _check_soft_weights_against_own_logits(to_np(lg), to_np(dw), to_np(cw), O.BF16, tag)
    np.testing.assert_allclose(to_np(dw).sum(1), 1.0, atol=3e-2, err_msg=tag)
    np.testing.assert_allclose(to_np(cw).sum(2), 1.0, atol=3e-2, err_msg=tag)


@pytest.mark.parametrize("G,S,D,N", [(5, 196, 768, 128), (2, 250, 768, 128), (3, 100, 512, 64),
                                     (2, 300, 256, 104), (2, 37, 384, 40)])
def test_soft_route_two_roles_and_single_role_agree(K, G, S, D, N):
  """The kernel whose waves split into producers and consumers against the row tiles, whose waves have
  one role (VMOE_SOFT_ROUTE_SINGLE_ROLE=1): same arithmetic per element, different summation order in
  the norms and softmax sums: a norm that rounds the other way moves a normalised item by one
  bfloat16 step, a logit by about as much, and a weight by up to exp(step) - 1, in few places."""
  rng = np.random.default_rng(G * S + N)
  x = to_dev(O.cast(rng.standard_normal((G, S, D)), O.BF16), O.BF16)
  mu = to_dev(O.cast(rng.standard_normal((D, N)) / np.sqrt(D), O.BF16), O.BF16)
  got = [to_np(a) for a in K.soft_route(x, mu, 1.3, return_logits=True)]
  os.environ["VMOE_SOFT_ROUTE_SINGLE_ROLE"] = "1"
  try:
    want = [to_np(a) for a in K.soft_route(x, mu, 1.3, return_logits=True)]
  finally:
    del os.environ["VMOE_SOFT_ROUTE_SINGLE_ROLE"]
  for name, a, b in zip(("dispatch weights", "combine weights", "logits"), got, want):
    diff = np.abs(a - b)
    floor = 2.0 ** -7 * np.abs(b).max() if name == "logits" else 0.0
    assert (diff <= 2.0 ** -5 * np.abs(b) + floor).all(), (name, float((diff / (np.abs(b) + 1e-30)).max()))
    assert (diff > 0).mean() <= 1e-3, (name, float((diff > 0).mean()))


EINSUM_CASES = [
    # G, S, E, C, D, wdtype, ddtype
    (2, 3, 2, 2, 4, O.F32, O.F32),
    (2, 3, 4, 1, 4, O.F32, O.F32),
    (4, 50, 2, 3, 40, O.F32, O.BF16),     # Bfloat16Dispatcher over float32 weights
    (8, 196, 4, 2, 96, O.BF16, O.BF16),
    (3, 33, 5, 1, 20, O.F32, O.F32),
    # all-bfloat16 cases take the bf16 matrix-core path where its limits allow
    (5, 17, 3, 8, 72, O.BF16, O.BF16),      # G % 8 != 0, ragged S and D
    (8, 256, 4, 34, 200, O.BF16, O.BF16),   # E*C = 136: two row blocks in dispatch, generic combine
    (16, 196, 128, 1, 128, O.BF16, O.BF16), # Soft MoE B/16 rows, E does not divide G
    (8, 100, 4, 8, 64, O.BF16, O.BF16),     # E divides G: interleaved buffer order
    (3, 257, 2, 4, 64, O.BF16, O.BF16),     # S above the bf16 path's limit
]


@pytest.mark.parametrize("G,S,E,C,D", [(2, 64, 8, 8, 64), (3, 65, 5, 13, 70), (4, 1, 2, 1, 3), (2, 130, 3, 43, 129)])
@pytest.mark.parametrize("wdtype", [torch.float32, torch.bool])
def test_einsum_float32_weights_in_64_bits(K, G, S, E, C, D, wdtype):
  """The generic einsum at k tiles, rows and columns that end inside (and addresses of the types' own alignment)
  against 64 bits; float32 data that count as rounded to bfloat16 give the bits of a cast in front."""
  gen = torch.Generator(device=dev()).manual_seed(S)
  w = torch.randn((G, S, E, C), generator=gen, device=dev())
  w = w > 0 if wdtype == torch.bool else w
  x = torch.randn((G, S, D), generator=gen, device=dev())
  y = torch.randn((E * G * C, D), generator=gen, device=dev())
  order = torch.arange(E * G * C, device=dev()).view(E * G * C, 1).float()       # slot rows, by a one-hot of each
  bound = lambda a, b: a.abs() @ b.abs() * max(S, E * C) * 2.0 ** -24 + 1e-30     # n roundings of partial sums
  wd = w.double().view(G, S, E * C)
  eye = torch.eye(E * C, device=dev()).view(1, E * C, E, C).expand(G, -1, -1, -1)
  rows = K.einsum_combine(eye, order, torch.float32).long().view(G, E * C)         # row of slot (g, n)
  got = K.einsum_dispatch(w, x, torch.float32)
  for g in range(G):
    want, at = wd[g].t() @ x[g].double(), got[rows[g]].double()
    assert bool(((at - want).abs() <= bound(wd[g].t(), x[g].double())).all())
  assert torch.equal(K.einsum_dispatch(w, x, torch.float32, True), K.einsum_dispatch(w, x.bfloat16(), torch.float32))
  if wdtype != torch.bool:
    got = K.einsum_combine(w, y, torch.float32)
    for g in range(G):
      data = y[rows[g]].double()
      assert bool(((got[g].double() - wd[g] @ data).abs() <= bound(wd[g], data)).all())
    assert torch.equal(K.einsum_combine(w, y, torch.float32, True), K.einsum_combine(w, y.bfloat16(), torch.float32))


@pytest.mark.parametrize("G,S,E,C,D,wdtype,ddtype", EINSUM_CASES)
def test_einsum_dispatch_combine(K, G, S, E, C, D, wdtype, ddtype):
  rng = np.random.default_rng(G + S)
  w = O.cast(O.softmax(rng.standard_normal((G, S, E * C)).astype(np.float32)), wdtype)
  w = w.reshape(G, S, E, C)
  x = O.cast(rng.standard_normal((G, S, D)), ddtype)
  d = O.EinsumDispatcher(w, w)
  out_dtype = wdtype if wdtype == ddtype else O.F32
  buf = K.einsum_dispatch(to_dev(w, wdtype), to_dev(x, ddtype), tdtype(out_dtype))
  want = O.cast(d.dispatch(x), out_dtype)
  # bf16 x bf16 products are exact in float32: only the summation order differs.
  tol = 1e-5 if out_dtype == O.F32 else 8e-3
  assert_close(to_np(buf).reshape(E, G * C, D), want, tol, "einsum dispatch")
  y = O.cast(rng.standard_normal((E, G * C, D)), ddtype)
  out = K.einsum_combine(to_dev(w, wdtype), to_dev(y, ddtype).view(E * G * C, D), tdtype(out_dtype))
  assert_close(to_np(out), O.cast(d.combine(y), out_dtype), tol, "einsum combine")


@pytest.mark.parametrize("G,S,E,C,D,offset", [
    (8, 196, 128, 2, 768, 0),    # the Soft MoE router's default capacity: 256 slots
    (3, 256, 1, 129, 72, 0),     # one past the 128-slot form; an odd row length
    (2, 257, 5, 1, 64, 0),       # one past 256 items: the items halved between waves
    (9, 512, 4, 128, 136, 0),    # the longest contraction of both directions
    (2, 513, 3, 171, 40, 0),     # one past it: the generic kernel
    (4, 31, 7, 63, 200, 0),      # 441 slots, a lone partial row tile
    (5, 300, 19, 1, 96, 3),      # weights at an address that is a multiple of 2 only
    (8, 16, 8, 2, 8, 1),
    (1, 1, 1, 1, 8, 0),
])
def test_einsum_bf16_long_rows(K, G, S, E, C, D, offset):
  """bfloat16 dispatch / combine over contractions of any length and rows of weights that start
  anywhere.  Products are exact in float32, so against the float32 oracle the result is off by its own
  rounding to bfloat16 (half of the last of 8 bits: 2**-8 of the value) and the roundings of both sums (2**-24 of the sum of
  magnitudes per term each)."""
  rng = np.random.default_rng(G * S + E)
  N = E * C
  w = O.cast(O.softmax(rng.standard_normal((G, S, N)).astype(np.float32) * 2), O.BF16)
  x = O.cast(rng.standard_normal((G, S, D)), O.BF16)
  y = O.cast(rng.standard_normal((E, G * C, D)), O.BF16)
  buf = torch.empty(w.size + offset, dtype=torch.bfloat16, device="cuda")
  wd = buf[offset:].view(G, S, E, C)
  wd.copy_(to_dev(w.reshape(G, S, E, C), O.BF16))
  d = O.EinsumDispatcher(w.reshape(G, S, E, C), w.reshape(G, S, E, C))

  def check(got, want, mag, terms, what):
    err = np.abs(got.astype(np.float64) - want)
    bound = 2.0 ** -8 * np.abs(want) + 2 * terms * 2.0 ** -24 * mag + 1e-30
    assert (err <= bound).all(), (what, float((err / bound).max()))

  got = to_np(K.einsum_dispatch(wd, to_dev(x, O.BF16), torch.bfloat16)).reshape(E, G * C, D)
  check(got, d.dispatch(x).astype(np.float64), d.dispatch(np.abs(x)), S, "dispatch")
  got = to_np(K.einsum_combine(wd, to_dev(y, O.BF16).view(E * G * C, D), torch.bfloat16))
  check(got, d.combine(y).astype(np.float64), d.combine(np.abs(y)), N, "combine")


def test_einsum_golden_and_bool_weights(K, goldens):
  data = np.asarray(goldens["dispatcher_data"]["data"], np.float32)
  for case in ("dispatcher_experts_divide_groups", "dispatcher_groups_divide_experts"):
    g = goldens[case]
    cw = np.asarray(g["einsum_combine_weights"], np.float32)
    E, C = g["num_experts"], g["capacity"]
    buf = K.einsum_dispatch(to_dev(cw > 0), to_dev(data), torch.float32)
    np.testing.assert_array_almost_equal(to_np(buf).reshape(E, 2 * C, 4), np.asarray(g["expected_dispatch"]))
    out = K.einsum_combine(to_dev(cw), buf, torch.float32)
    np.testing.assert_array_almost_equal(to_np(out), np.asarray(g["expected_combine"]))


# ------------------------------------------------------------------ packed expert rows
@pytest.mark.parametrize("G,S,E,Kk,C,bpr", [(4, 64, 4, 2, 20, True), (8, 50, 8, 2, 16, False), (8, 128, 8, 2, 30, False), (32, 1568, 32, 2, 100, True),
                                            (3, 33, 5, 1, 8, True), (300, 16, 4, 2, 6, False),
                                            (64, 128, 4, 2, 6, True), (9, 300, 7, 2, 40, True), (2, 200, 300, 2, 3, False),
                                            (32, 49, 8, 2, 16, False),      # S/32 layer: a block of 256 assignments touches four groups
                                            (40, 19, 8, 2, 6, True)])        # 38 per group: eight groups per block, the most the one-launch form takes
def test_compact_rows(K, G, S, E, Kk, C, bpr):
  """token_row = e*G*C + (kept items of expert e in the groups before g) + position."""
  rng = np.random.default_rng(G * S + E)
  gates = O.softmax(rng.standard_normal((G, S, E)).astype(np.float32) * 2)
  val, idx = K.topk(to_dev(gates), Kk)
  indices, token_slot, slot_token, fill = K.route_assign(val, idx, E, C, bpr)
  token_row, rows, row_token = K.compact_rows(fill, token_slot, C)
  f = to_np(fill)
  np.testing.assert_array_equal(to_np(rows), f.sum(0))
  ind = to_np(indices)
  prefix = np.cumsum(f, axis=0) - f                         # (G, E)
  e, pos = ind[..., 0], ind[..., 1]
  kept = pos < C
  want = np.where(kept, e * (G * C) + np.take_along_axis(
      prefix[:, None, :].repeat(S, 1), e, axis=2) + pos, -1)
  np.testing.assert_array_equal(to_np(token_row), want)
  # row_token is the inverse map on the packed rows
  tr, rt = to_np(token_row).reshape(G * S, Kk), to_np(row_token).reshape(-1)
  items = np.repeat(np.arange(G * S), Kk).reshape(G * S, Kk)
  np.testing.assert_array_equal(rt[tr[tr >= 0]], items[tr >= 0])
  # a bijection onto the first rows of every expert
  r = to_np(token_row)[kept]
  assert len(np.unique(r)) == r.size
  for ee in range(E):
    mine = r[(r // (G * C)) == ee] - ee * G * C
    assert sorted(mine) == list(range(f.sum(0)[ee]))


@pytest.mark.parametrize("E,R,D,M", [
    (8, 416, 512, 2048),      # one expert per die; first product 64 x 128 tiles, second 64 x 64
    (5, 700, 512, 1024),      # 64 x 64 tiles; runs that begin and end inside an expert
    (3, 1000, 512, 1536),     # 64 x 128 and 64 x 64
])
def test_expert_mlp_float32_products_on_the_dma_kernel(K, monkeypatch, E, R, D, M):
  """Float32 products on float32 matrix instructions (float32_products=True): the LDS-DMA kernel (64 x 128 or
  64 x 64 tiles, one run of the tile list per die, rows past a count skipped in blocks of 32)
  against the register-staged kernel and the oracle; dense, over ragged rows and over gathered ones;
  the same bits in a call of four times the rows, which takes 64 x 128 tiles for either product."""
  monkeypatch.delenv("VMOE_F32_GEMM", raising=False)
  rng = np.random.default_rng(E + R)
  x = rng.standard_normal((E, R, D)).astype(np.float32)
  w0 = (rng.standard_normal((E, D, M)) / np.sqrt(D)).astype(np.float32)
  b0 = (rng.standard_normal((E, M)) * 0.1).astype(np.float32)
  w1 = (rng.standard_normal((E, M, D)) / np.sqrt(M)).astype(np.float32)
  b1 = (rng.standard_normal((E, D)) * 0.1).astype(np.float32)
  items = rng.standard_normal((R + 7, D)).astype(np.float32)
  x_rows = rng.integers(0, R + 7, (E, R)).astype(np.int32)
  weights = [to_dev(a) for a in (w0, b0, w1, b1)]
  rows = rng.integers(0, R + 1, E).astype(np.int32)
  rows[:3] = [R, 0, 33]
  run = lambda x, **kw: to_np(K.expert_mlp(to_dev(x), *weights, float32_products=True, **kw))
  ragged = lambda x, **kw: run(x, out=torch.full((E, R, D), 7.0, device=dev()), rows_per_expert=to_dev(rows), **kw)
  dense = run(x)
  assert_close(dense, O.mlp_block(x, w0, b0, w1, b1, O.F32), 1e-5, "dense")
  some, gathered, indexed = ragged(x), ragged(items, x_rows=to_dev(x_rows)), run(items[x_rows])
  for e, n in enumerate(rows):
    np.testing.assert_array_equal(some[e, :n], dense[e, :n], err_msg=f"ragged: expert {e}")
    np.testing.assert_array_equal(gathered[e, :n], indexed[e, :n], err_msg=f"gathered: expert {e}")
    assert (some[e, n:] == 7.0).all() and (gathered[e, n:] == 7.0).all(), f"expert {e}: written past its rows"
  assert E * -(-4 * R // 64) * (D // 128) >= 512
  np.testing.assert_array_equal(run(np.tile(x, (1, 4, 1))), np.tile(dense, (1, 4, 1)))    # same order of k
  # the default products round in another order: they are not what ran above
  assert (to_np(K.expert_mlp(to_dev(x), *weights)) != dense).any()
  monkeypatch.setenv("VMOE_F32_GEMM", "plain")
  plain = to_np(K.expert_mlp(to_dev(x), *weights))
  assert_close(dense, plain, 1e-5, "against plain")                                       # other order of k
  assert (plain != dense).any()


@pytest.mark.parametrize("width", [36, 64, 100])
@pytest.mark.parametrize("approximate", [True, False])
def test_expert_mlp_float32_gelu(K, monkeypatch, width, approximate):
  """The GELU of float32 MLPs through products with the identity, which are exact: tanhf where the width is no
  multiple of 32, else within the roundings of x / (1 + 2^z) on the hardware's exp2 and reciprocal; the same as behind
  products on float32 instructions."""
  from scipy.special import erfc
  x = np.concatenate([np.linspace(-14, 14, 20 * width), np.logspace(-30, 2, 10 * width),
                      -np.logspace(-30, 2, 10 * width)]).astype(np.float32).reshape(1, 40, width)
  eye = to_dev(np.eye(width, dtype=np.float32)[None])
  run = lambda **kw: to_np(K.expert_mlp(to_dev(x), eye, None, eye, None, approximate_gelu=approximate, **kw))
  monkeypatch.delenv("VMOE_F32_GEMM", raising=False)
  got = run()
  # (three bfloat16 values end at 2^-133: below 2^-110 a value loses its last bits)
  np.testing.assert_allclose(got, run(float32_products=True), rtol=0, atol=2.0 ** -133)
  monkeypatch.setenv("VMOE_F32_GEMM", "plain")
  plain = run()
  v = x.astype(np.float64)
  if not approximate or width % 32 != 0:
    np.testing.assert_array_equal(got, plain)
  u = 2 * np.sqrt(2 / np.pi) * (v + 0.044715 * v ** 3)
  with np.errstate(over="ignore"):
    want = v / (1 + np.exp(-u)) if approximate else 0.5 * v * erfc(-v / np.sqrt(2))
  # tanhf, erff: two units in the last place of a number up to one, the sum half a one, which x / 2 scales
  bound = 2.0 ** -24 * (3 * np.abs(v) + np.abs(want))
  if approximate and width % 32 == 0:
    # z: three roundings and two rounded constants, each 2^-24 of |u|, which the exponential makes relative; exp2, the
    # sum, the reciprocal and the product: 2^-24 each, twice that for the two hardware functions.  Below 2^-120 it ends.
    bound = 2.0 ** -24 * (6 + 5 * np.abs(u)) * np.abs(want) + 2.0 ** -120
  elif approximate:
    bound += 2.0 ** -24 * 5 * np.abs(u) * np.abs(v) / np.cosh(np.minimum(np.abs(u) / 2, 300)) ** 2 / 4    # of tanh's argument
  assert (np.abs(got - want) <= bound + 2.0 ** -148).all()


def test_expert_mlp_float32_over_the_size_of_the_call(K, monkeypatch):
  """The tile, and with it the order of float32 sums, depends on the size of the call: the same items
  through the same experts stay as close to 64 bits at every size as float32 matrix instructions
  are (2-norm, a twentieth for the differing order of few sums; see test_expert_mlp_float32_split_tiles)."""
  monkeypatch.delenv("VMOE_F32_GEMM", raising=False)
  rng = np.random.default_rng(5)
  E, D, M, n = 8, 512, 2048, 16
  x = rng.standard_normal((E, 784, D)).astype(np.float32)
  w0 = (rng.standard_normal((E, D, M)) / np.sqrt(D)).astype(np.float32)
  w1 = (rng.standard_normal((E, M, D)) / np.sqrt(M)).astype(np.float32)
  u = x[:, :n].astype(np.float64) @ w0
  want = (u / (1 + np.exp(-2 * np.sqrt(2 / np.pi) * (u + 0.044715 * u ** 3)))) @ w1
  off = lambda a: np.linalg.norm(a - want) / np.linalg.norm(want)
  run = lambda R: to_np(K.expert_mlp(to_dev(x[:, :R]), to_dev(w0), None, to_dev(w1), None))[:, :n]
  outs = {R: run(R) for R in (16, 49, 98, 196, 392, 784)}
  monkeypatch.setenv("VMOE_F32_GEMM", "plain")
  most = 1.05 * off(run(n))
  assert all(off(out) <= most for out in outs.values()), ({R: off(out) for R, out in outs.items()}, most)
  assert len({out.tobytes() for out in outs.values()}) > 1        # (several tiles were taken)


@pytest.mark.parametrize("E,R,D,M", [(3, 129, 96, 260), (5, 33, 100, 132), (2, 64, 800, 128), (70, 3, 36, 64)])
def test_expert_mlp_float32_split_tiles(K, monkeypatch, E, R, D, M):
  """Every tile of the float32 products on bfloat16 MFMAs (three bfloat16 values per operand), at
  sizes that end inside a tile of rows, columns or k and for more experts than lanes: no further from
  64 bits than the float32 MFMA kernel (VMOE_F32_GEMM=plain; 2-norm, a twentieth for the differing
  order of few sums), also where the operands' scales lie 2^80 apart; ragged rows bit for bit as dense ones,
  nothing past them; gathered rows bit for bit as rows indexed beforehand."""
  rng = np.random.default_rng(E + R)
  up = 2.0 ** 80
  x = rng.standard_normal((E, R, D)).astype(np.float32)
  w0 = (rng.standard_normal((E, D, M)) / np.sqrt(D)).astype(np.float32)
  b0 = (rng.standard_normal((E, M)) * 0.1).astype(np.float32)
  w1 = (rng.standard_normal((E, M, D)) / np.sqrt(M)).astype(np.float32)
  b1 = (rng.standard_normal((E, D)) * 0.1).astype(np.float32)
  rows = rng.integers(0, R + 1, E).astype(np.int32)
  rows[:2] = [R, 0]
  items = rng.standard_normal((R + 7, D)).astype(np.float32)
  x_rows = rng.integers(0, R + 7, (E, R)).astype(np.int32)

  def want(xx):
    h = xx.astype(np.float64) @ w0.astype(np.float64) + b0[:, None]
    h = 0.5 * h * (1 + np.tanh(np.sqrt(2 / np.pi) * (h + 0.044715 * h ** 3)))
    return h @ w1.astype(np.float64) + b1[:, None]

  exact = want(x)
  off = lambda a: np.linalg.norm(to_np(a) - exact) / np.linalg.norm(exact)
  rest = [to_dev(a) for a in (w0, b0, w1, b1)]
  monkeypatch.setenv("VMOE_F32_GEMM", "plain")
  plain = off(K.expert_mlp(to_dev(x), *rest))
  for tile in range(7):
    monkeypatch.setenv("VMOE_F32_GEMM", f"tile{tile}")
    dense = K.expert_mlp(to_dev(x), *rest)
    assert off(dense) <= 1.05 * plain, (tile, off(dense), plain)
    scaled = K.expert_mlp(to_dev((x / up).astype(np.float32)), to_dev((w0 * up).astype(np.float32)), *rest[1:])
    assert off(scaled) <= 1.05 * plain, (tile, off(scaled), plain)
    ragged = torch.full((E, R, D), 7.0, device=dev())
    K.expert_mlp(to_dev(x), *rest, out=ragged, rows_per_expert=to_dev(rows))
    dense, ragged = to_np(dense), to_np(ragged)
    for e, n in enumerate(rows):
      np.testing.assert_array_equal(ragged[e, :n], dense[e, :n], err_msg=f"tile {tile}, expert {e}")
      assert (ragged[e, n:] == 7.0).all(), f"tile {tile}, expert {e} wrote past its rows"
    if D % 32 == 0:
      full = to_dev(np.full(E, R, np.int32))
      got = K.expert_mlp(to_dev(items), *rest, rows_per_expert=full, x_rows=to_dev(x_rows))
      ref = K.expert_mlp(to_dev(items[x_rows]), *rest, rows_per_expert=full)
      np.testing.assert_array_equal(to_np(got), to_np(ref))


@pytest.mark.parametrize("tile", range(7))
def test_expert_mlp_float32_weights_at_any_address(K, monkeypatch, tile):
  """Weights one, two and three floats past a 16-byte boundary: the bits of aligned ones."""
  monkeypatch.setenv("VMOE_F32_GEMM", f"tile{tile}")
  E, R, D, M = 3, 70, 100, 132
  gen = torch.Generator().manual_seed(tile)
  mk = lambda *s: torch.randn(s, generator=gen).to(dev())
  x, w0, b0, w1, b1 = mk(E, R, D), mk(E, D, M), mk(E, M), mk(E, M, D), mk(E, D)
  want = K.expert_mlp(x, w0, b0, w1, b1)
  for shift in (1, 2, 3):
    moved = [torch.empty(w.numel() + shift, device=dev())[shift:].view(w.shape).copy_(w) for w in (w0, b0, w1, b1)]
    assert all(w.data_ptr() % 16 == 4 * shift for w in moved)
    assert torch.equal(K.expert_mlp(x, *moved), want)


@pytest.mark.parametrize("tile", range(7))
def test_expert_mlp_float32_split_tiles_infinities(K, monkeypatch, tile):
  """Infinite and NaN operands, and finite ones that round to infinity in bfloat16, give what float32
  multiplication gives (VMOE_F32_GEMM=plain): infinities of the same sign, NaN in the same places, the
  other items bit for bit what they are without them."""
  rng = np.random.default_rng(3)
  E, R, D, M = 2, 70, 64, 132
  x = rng.standard_normal((E, R, D)).astype(np.float32)
  w0 = np.abs(rng.standard_normal((E, D, M)) / np.sqrt(D)).astype(np.float32)
  w1 = (rng.standard_normal((E, M, D)) / np.sqrt(M)).astype(np.float32)
  w1[:, :, ::2] = np.abs(w1[:, :, ::2])
  w1[:, :, 1::4] *= -1
  w1[:, :, 3::4] = -np.abs(w1[:, :, 3::4])
  w0[1, 5] = 1e-38
  odd = x.copy()
  odd[0, 3, 7], odd[0, 69, 0], odd[1, 20, 63], odd[1, 33, 5] = np.inf, -np.inf, np.nan, 3.4e38
  run = lambda a: to_np(K.expert_mlp(to_dev(a), to_dev(w0), None, to_dev(w1), None))
  monkeypatch.setenv("VMOE_F32_GEMM", "plain")
  want = run(odd)
  monkeypatch.setenv("VMOE_F32_GEMM", f"tile{tile}")
  got, clean = run(odd), run(x)
  assert np.isinf(want[0, 3]).any() and np.isnan(want[1, 20]).all() and np.isfinite(want[1, 33]).all()
  np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
  np.testing.assert_array_equal(np.where(np.isinf(got), got, 0), np.where(np.isinf(want), want, 0))
  ok = np.isfinite(want)
  assert_close(got[ok], want[ok], 1e-5, "finite values")
  same = np.ones((E, R), bool)
  for e, r in ((0, 3), (0, 69), (1, 20), (1, 33)):
    same[e, r] = False
  np.testing.assert_array_equal(got[same], clean[same])


@pytest.mark.parametrize("tile", [7, 8])
def test_expert_mlp_float32_four_groups_along_k(K, monkeypatch, tile):
  """The tiles whose four groups take turns: the checks above, and against 64 bits where k leaves some of the groups
  nothing, ends inside a group's share, or ends inside a k tile; ragged rows bit for bit as well."""
  test_expert_mlp_float32_weights_at_any_address(K, monkeypatch, tile)
  test_expert_mlp_float32_split_tiles_infinities(K, monkeypatch, tile)
  monkeypatch.setenv("VMOE_F32_GEMM", f"tile{tile}")
  for E, R, D, M in [(2, 33, 4, 36), (3, 65, 100, 260), (2, 129, 36, 132), (5, 7, 288, 68), (2, 64, 1028, 64)]:
    gen = torch.Generator(device=dev()).manual_seed(D)
    mk = lambda *s: torch.randn(s, generator=gen, device=dev())
    x, w0, b0, w1, b1 = mk(E, R, D), mk(E, D, M) * D ** -0.5, mk(E, M), mk(E, M, D) * M ** -0.5, mk(E, D)
    got = K.expert_mlp(x, w0, b0, w1, b1)
    h = torch.nn.functional.gelu(torch.bmm(x.double(), w0.double()) + b0.double()[:, None], approximate="tanh")
    want = torch.bmm(h, w1.double()) + b1.double()[:, None]
    # (2-norm: sums of float32 products in float32 are off by less than 2^-24 times the square root of their number)
    assert ((got.double() - want).norm() / want.norm()).item() <= max(D, M) ** 0.5 * 2.0 ** -23
    rows = torch.randint(0, R + 1, (E,), generator=gen, device=dev(), dtype=torch.int32)
    rows[0] = R
    ragged = torch.full_like(got, 7.0)
    K.expert_mlp(x, w0, b0, w1, b1, out=ragged, rows_per_expert=rows)
    for e, n in enumerate(rows.tolist()):
      assert torch.equal(ragged[e, :n], got[e, :n]) and bool((ragged[e, n:] == 7.0).all())


def test_expert_mlp_float32_seeded_shapes(K):
  """A seeded sweep of float32 expert MLPs over odd shapes (rows short of a block, widths that
  end inside a tile, k that is or is not whole 32-wide tiles, many or few experts), dense and
  over ragged rows, against the oracle at 1e-5: whichever kernel the shape takes."""
  rng = np.random.default_rng(2024)
  for case in range(14):
    E = int(rng.choice([1, 2, 3, 8, 11, 40]))
    R = int(rng.choice([1, 7, 31, 33, 64, 65, 130, 257]))
    D = int(rng.choice([32, 36, 64, 96, 100, 160, 224]))
    M = int(rng.choice([32, 40, 64, 128, 132, 192, 288]))
    x = rng.standard_normal((E, R, D)).astype(np.float32)
    w0 = (rng.standard_normal((E, D, M)) / np.sqrt(D)).astype(np.float32)
    b0 = (rng.standard_normal((E, M)) * 0.1).astype(np.float32)
    w1 = (rng.standard_normal((E, M, D)) / np.sqrt(M)).astype(np.float32)
    b1 = (rng.standard_normal((E, D)) * 0.1).astype(np.float32)
    rows = rng.integers(0, R + 1, E).astype(np.int32)
    rows[0] = R
    want = O.mlp_block(x, w0, b0, w1, b1, O.F32)
    args = [to_dev(a) for a in (x, w0, b0, w1, b1)]
    dense = to_np(K.expert_mlp(*args))
    assert_close(dense, want, 1e-5, f"case {case}: E={E} R={R} D={D} M={M} dense")
    ragged = torch.full((E, R, D), 7.0, dtype=torch.float32, device=dev())
    K.expert_mlp(*args, out=ragged, rows_per_expert=to_dev(rows))
    ragged = to_np(ragged)
    for e, n in enumerate(rows):
      np.testing.assert_array_equal(ragged[e, :n], dense[e, :n], err_msg=f"case {case}: E={E} R={R} D={D} M={M} expert {e}")
      assert (ragged[e, n:] == 7.0).all(), f"case {case}: expert {e} wrote past its rows"


def test_expert_mlp_bfloat16_seeded_shapes(K):
  """The same sweep in bfloat16 (widths in multiples of 8): dense against the oracle, ragged
  rows bit for bit against the dense call and nothing written past them, and, where the shape
  allows it, rows gathered from the items bit for bit against rows indexed beforehand."""
  rng = np.random.default_rng(2025)
  gathered = 0
  for case in range(14):
    E = int(rng.choice([1, 2, 3, 8, 11, 40]))
    R = int(rng.choice([1, 7, 31, 33, 64, 65, 130, 257, 300]))
    D = int(rng.choice([32, 40, 64, 96, 104, 160, 256]))
    M = int(rng.choice([32, 48, 64, 128, 136, 192, 512]))
    T = int(rng.choice([R, 3 * R + 5]))
    name = f"case {case}: E={E} R={R} D={D} M={M} T={T}"
    items = O.cast(rng.standard_normal((T, D)).astype(np.float32), O.BF16)
    w0 = O.cast((rng.standard_normal((E, D, M)) / np.sqrt(D)).astype(np.float32), O.BF16)
    b0 = O.cast((rng.standard_normal((E, M)) * 0.1).astype(np.float32), O.BF16)
    w1 = O.cast((rng.standard_normal((E, M, D)) / np.sqrt(M)).astype(np.float32), O.BF16)
    b1 = O.cast((rng.standard_normal((E, D)) * 0.1).astype(np.float32), O.BF16)
    rows = rng.integers(0, R + 1, E).astype(np.int32)
    rows[0] = R
    x_rows = rng.integers(0, T, (E, R)).astype(np.int32)
    x = items[x_rows]                                                      # (E, R, D)
    want = O.mlp_block(x, w0, b0, w1, b1, O.BF16)
    wd = [to_dev(a, O.BF16) for a in (w0, b0, w1, b1)]
    dense = K.expert_mlp(to_dev(x, O.BF16), *wd)
    assert_close(to_np(dense), want, 2e-2, name + " dense")
    ragged = torch.full((E, R, D), 7.0, dtype=torch.bfloat16, device=dev())
    K.expert_mlp(to_dev(x, O.BF16), *wd, out=ragged, rows_per_expert=to_dev(rows))
    for e, n in enumerate(rows):
      assert torch.equal(ragged[e, :n], dense[e, :n]), name + f" expert {e}"
      assert (to_np(ragged[e, n:]) == 7.0).all(), name + f": expert {e} wrote past its rows"
    if K.expert_mlp_can_gather(torch.bfloat16, D, T):
      gathered += 1
      for e, n in enumerate(rows):
        x_rows[e, n:] = 2 ** 30                                            # never followed
      got = torch.full((E, R, D), 7.0, dtype=torch.bfloat16, device=dev())
      K.expert_mlp(to_dev(items, O.BF16), *wd, out=got, rows_per_expert=to_dev(rows),
                   x_rows=to_dev(x_rows))
      assert torch.equal(got, ragged), name + " gathered"
  assert gathered >= 4


@pytest.mark.parametrize("dtype", [O.F32, O.BF16])
def test_expert_mlp_gathers_its_rows_from_the_items(K, dtype):
  """x_rows: the first product reads row r of expert e from item x_rows[e][r] of the (T, D)
  matrix of items.  Bit for bit what the same call computes on a buffer built by indexing;
  entries past an expert's count (here out of range on purpose) are never followed."""
  rng = np.random.default_rng(17)
  E, R, D, M, T = 6, 200, 96, 160, 500
  items = to_dev(O.cast(rng.standard_normal((T, D)).astype(np.float32), dtype), dtype)
  w0 = to_dev(O.cast(rng.standard_normal((E, D, M)).astype(np.float32) / np.sqrt(D), dtype), dtype)
  w1 = to_dev(O.cast(rng.standard_normal((E, M, D)).astype(np.float32) / np.sqrt(M), dtype), dtype)
  b0 = to_dev(O.cast(rng.standard_normal((E, M)).astype(np.float32) * 0.1, dtype), dtype)
  b1 = to_dev(O.cast(rng.standard_normal((E, D)).astype(np.float32) * 0.1, dtype), dtype)
  rows = np.asarray([200, 0, 1, 65, 128, 199], np.int32)
  x_rows = np.full((E, R), 2 ** 30, np.int32)
  for e, n in enumerate(rows):
    x_rows[e, :n] = rng.integers(0, T, n)
  assert K.expert_mlp_can_gather(tdtype(dtype), D, T)
  got = torch.full((E, R, D), 7.0, dtype=tdtype(dtype), device=dev())
  K.expert_mlp(items, w0, b0, w1, b1, out=got, rows_per_expert=to_dev(rows), x_rows=to_dev(x_rows))
  buf = items[torch.from_numpy(np.where(x_rows < T, x_rows, 0)).to(dev()).long()]      # (E, R, D)
  want = torch.full((E, R, D), 7.0, dtype=tdtype(dtype), device=dev())
  K.expert_mlp(buf, w0, b0, w1, b1, out=want, rows_per_expert=to_dev(rows))
  assert torch.equal(got, want)
  for e, n in enumerate(rows):
    assert (to_np(got[e, n:]) == 7.0).all()
  full = O.mlp_block(to_np(buf).astype(np.float32), to_np(w0), to_np(b0), to_np(w1), to_np(b1), dtype)
  for e, n in enumerate(rows):
    assert_close(to_np(got[e, :n]), full[e, :n], 1e-5 if dtype == O.F32 else 2e-2, f"expert {e}")


@pytest.mark.parametrize("dtype", [O.F32, O.BF16])
@pytest.mark.parametrize("E", [5, 20])      # fewer / more experts than dies in the launch plan
def test_expert_mlp_rows_per_expert(K, dtype, E):
  """Leading rows equal the full computation bit for bit; the other rows are not written."""
  rng = np.random.default_rng(3)
  R, D, M = 300, 64, 128
  x = to_dev(O.cast(rng.standard_normal((E, R, D)).astype(np.float32), dtype), dtype)
  w0 = to_dev(O.cast(rng.standard_normal((E, D, M)).astype(np.float32) / 8, dtype), dtype)
  w1 = to_dev(O.cast(rng.standard_normal((E, M, D)).astype(np.float32) / 11, dtype), dtype)
  b0 = to_dev(O.cast(rng.standard_normal((E, M)).astype(np.float32) * 0.1, dtype), dtype)
  b1 = to_dev(O.cast(rng.standard_normal((E, D)).astype(np.float32) * 0.1, dtype), dtype)
  full = K.expert_mlp(x, w0, b0, w1, b1)
  rows = np.asarray(([300, 0, 1, 129, 256] * 4)[:E], np.int32)
  out = torch.full_like(full, 7.0)
  x_bad = x.clone()
  for e, n in enumerate(rows):
    x_bad[e, n:] = float("nan")                      # rows past the count must not matter
  K.expert_mlp(x_bad, w0, b0, w1, b1, out=out, rows_per_expert=to_dev(rows))
  for e, n in enumerate(rows):
    np.testing.assert_array_equal(to_np(out[e, :n]), to_np(full[e, :n]))
    assert (to_np(out[e, n:]) == 7.0).all()


@pytest.mark.parametrize("E,R,D,M", [
    (5, 65, 1024, 512),      # one row past a 64-row tile
    (24, 130, 384, 512),     # two rows past a 128-row tile, as many experts as make three rounds of the dies
    (16, 257, 320, 640),     # one row past two 128-row tiles; columns end inside tiles of 128 and 192
    (12, 400, 512, 768),     # rows that end inside tiles of every height
    (8, 52, 96, 3072),       # long k over few rows, k not a multiple of 64 in the first product
    (3, 33, 136, 264),       # k that ends inside a 32-wide step
    (70, 3, 64, 200),        # more experts than rows, one short row tile each
    (3, 1, 800, 136),        # one row that ends in the first half of the last 128-wide k stage
    (5, 2, 40, 72),          # and rows shorter than that half
])
def test_expert_mlp_small_tiles(K, E, R, D, M):
  """bfloat16 products over few rows per expert (on the tiles that the choice by size takes; the tests below name
  them) against a float32 restatement with the same rounding points; ragged rows bit for bit against the dense call,
  nothing written past a count, and rows gathered from the items bit for bit as well."""
  rng = np.random.default_rng(E * 1000 + R)
  bf = torch.bfloat16
  mk = lambda scale, *s: to_dev(O.cast(rng.standard_normal(s).astype(np.float32) * scale, O.BF16), O.BF16)
  T = R + 7
  items, w0, b0 = mk(1, T, D), mk(D ** -0.5, E, D, M), mk(0.1, E, M)
  w1, b1 = mk(M ** -0.5, E, M, D), mk(0.1, E, D)
  x_rows = torch.from_numpy(rng.integers(0, T, (E, R)).astype(np.int32)).to(dev())
  x = items[x_rows.long()]
  dense = K.expert_mlp(x, w0, b0, w1, b1)
  for e in range(E):
    h = ((x[e].float() @ w0[e].float()).to(bf).float() + b0[e].float()).to(bf)
    h = torch.nn.functional.gelu(h.float(), approximate="tanh").to(bf)
    y = ((h.float() @ w1[e].float()).to(bf).float() + b1[e].float()).to(bf)
    np.testing.assert_allclose(to_np(dense[e]), to_np(y), rtol=2e-2, atol=2e-2, err_msg=f"expert {e}")
  rows = rng.integers(0, R + 1, E).astype(np.int32)
  rows[:3] = [R, 0, 1]
  bad = x_rows.clone()
  for e, n in enumerate(rows):
    bad[e, n:] = 2 ** 30                                  # never followed
  ragged, gathered = torch.full_like(dense, 7.0), torch.full_like(dense, 7.0)
  K.expert_mlp(x, w0, b0, w1, b1, out=ragged, rows_per_expert=to_dev(rows))
  for e, n in enumerate(rows):
    assert torch.equal(ragged[e, :n], dense[e, :n]), f"expert {e}"
    assert (to_np(ragged[e, n:]) == 7.0).all(), f"expert {e} wrote past its rows"
  if K.expert_mlp_can_gather(bf, D, T):
    K.expert_mlp(items, w0, b0, w1, b1, out=gathered, rows_per_expert=to_dev(rows), x_rows=bad)
    assert torch.equal(gathered, ragged)


@pytest.mark.parametrize("tile", range(8))
def test_expert_mlp_every_small_tile(K, monkeypatch, tile):
  """Each tile of kRowsTiles (0, 1, 2 and 4 are gemm_bf16_rows_kernel's, the others gemm_bf16_mid_kernel's;
  VMOE_ROW_TILES names one for both products) through the checks above, at a shape whose row, column and k tiles
  all end inside and one of a row."""
  monkeypatch.setenv("VMOE_ROW_TILES", str(tile))
  test_expert_mlp_small_tiles(K, 3, 131, 136, 264)
  test_expert_mlp_small_tiles(K, 9, 1, 192, 72)


@pytest.mark.parametrize("tile", [3, 5, 6, 7, 13, 14, 15, 16])
def test_expert_mlp_medium_tiles(K, monkeypatch, tile):
  """The tiles of the kernel for a few hundred to a few thousand rows: the checks of the small tiles with and
  without a launch plan, at one row past a tile of each height, k and columns that end inside, and bit
  for bit what the smallest tile computes (same order of sums), also without a bias and with biases at an
  odd element."""
  for E, R, D, M in [(3, 131, 136, 264), (9, 1, 192, 72), (17, 257, 320, 200), (9, 193, 96, 1032), (3, 1100, 64, 8)]:
    monkeypatch.setenv("VMOE_ROW_TILES", str(tile))
    test_expert_mlp_small_tiles(K, E, R, D, M)
    rng = np.random.default_rng(E)
    mk = lambda scale, *s: to_dev(O.cast(rng.standard_normal(s).astype(np.float32) * scale, O.BF16), O.BF16)
    x, w0, w1 = mk(1, E, R, D), mk(D ** -0.5, E, D, M), mk(M ** -0.5, E, M, D)
    b0, b1 = mk(0.1, E * M + 1)[1:].view(E, M), mk(0.1, E * D + 1)[1:].view(E, D)
    for biases in ((None, None), (b0, b1)):
      for approximate in (True, False):
        args = (x, w0, biases[0], w1, biases[1])
        monkeypatch.setenv("VMOE_ROW_TILES", str(tile))
        got = K.expert_mlp(*args, approximate_gelu=approximate)
        monkeypatch.setenv("VMOE_ROW_TILES", "0")
        want = K.expert_mlp(*args, approximate_gelu=approximate)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("second", ["eight", "narrow"])
@pytest.mark.parametrize("rows", [1, 16, 33, 63, 64, 65, 96, 97, 127, 128, 129, 161, 193, 255, 256, 257, 449])
def test_expert_mlp_last_tiles_of_the_large_kernels(K, monkeypatch, rows, second):
  """The large tiles multiply the live row blocks of an expert's last tile only: every number of them, at one row
  either side, in dense and ragged calls (experts without a row, with one tile and with several among them), bit for
  bit what the smallest tile computes (same order of sums), and nothing written past the live rows."""
  E, D, M = 5, 320, 456 if second == "eight" else 392
  M += -M % 64                                             # (k of the second product: whole 64s, from 256 on)
  rng = np.random.default_rng(rows)
  mk = lambda scale, *s: to_dev(O.cast(rng.standard_normal(s).astype(np.float32) * scale, O.BF16), O.BF16)
  x, w0, w1 = mk(1, E, rows, D), mk(D ** -0.5, E, D, M), mk(M ** -0.5, E, M, D)
  b0, b1 = mk(0.1, E, M), mk(0.1, E, D)
  counts = torch.tensor([rows, 0, min(rows, 1), (rows + 1) // 2, max(rows - 30, 0)], dtype=torch.int32, device=dev())

  def run(large, live):
    monkeypatch.setenv("VMOE_ROW_TILES", "off" if large else "0")
    monkeypatch.setenv("VMOE_SECOND_PRODUCT", second if large else "")
    out = torch.full((E, rows, D), 7.0, dtype=torch.bfloat16, device=dev())
    K.expert_mlp(x, w0, b0, w1, b1, out=out, rows_per_expert=live)
    return out

  for live in (None, counts):
    got, want = run(True, live), run(False, live)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    for e, n in enumerate(counts.tolist() if live is not None else []):
      assert bool((got[e, n:] == 7.0).all())


@pytest.mark.parametrize("second", ["eight", "narrow"])
@pytest.mark.parametrize("E", [100, 150])                   # (below and above two rounds of tiles per die: 500 and 750)
def test_expert_mlp_short_last_tiles_of_long_launches(K, monkeypatch, E, second):
  """Last tiles of 129 to 192 rows, whose idle waves take part in the product of a launch of few rounds and stay out of it in
  a longer one: bit for bit what the smallest tile computes, and nothing written past the live rows."""
  R, D, M = 161, 1280 if second == "eight" else 960, 256
  rng = np.random.default_rng(E)
  mk = lambda scale, *s: to_dev(O.cast(rng.standard_normal(s).astype(np.float32) * scale, O.BF16), O.BF16)
  x, w0, w1 = mk(1, E, R, D), mk(D ** -0.5, E, D, M), mk(M ** -0.5, E, M, D)
  b0, b1 = mk(0.1, E, M), mk(0.1, E, D)
  counts = torch.from_numpy(rng.choice([0, 1, 128, 129, 160, 161], E).astype(np.int32)).to(dev())
  out = []
  for tiles, kernel in (("off", second), ("0", "")):
    monkeypatch.setenv("VMOE_ROW_TILES", tiles)
    monkeypatch.setenv("VMOE_SECOND_PRODUCT", kernel)
    for live in (None, counts):
      out.append(torch.full((E, R, D), 7.0, dtype=torch.bfloat16, device=dev()))
      K.expert_mlp(x, w0, b0, w1, b1, out=out[-1], rows_per_expert=live)
  assert torch.equal(out[0].view(torch.int16), out[2].view(torch.int16))
  assert torch.equal(out[1].view(torch.int16), out[3].view(torch.int16))


@pytest.mark.parametrize("E,R,D,M", [(5, 800, 832, 3328), (3, 1500, 512, 2048), (12, 896, 448, 1088), (21, 140, 704, 2816),
                                     (5, 8, 64, 136), (4, 2576, 96, 2048)])
def test_expert_mlp_of_full_experts(K, E, R, D, M):
  """A call that says that every row is live may take other tiles (these shapes do), and gives the same bits; so does
  one that says it of rows that are not."""
  rng = np.random.default_rng(R)
  mk = lambda scale, *s: to_dev(O.cast(rng.standard_normal(s).astype(np.float32) * scale, O.BF16), O.BF16)
  T = R + 5
  items, w0, b0 = mk(1, T, D), mk(D ** -0.5, E, D, M), mk(0.1, E, M)
  w1, b1 = mk(M ** -0.5, E, M, D), mk(0.1, E, D)
  x_rows = torch.from_numpy(rng.integers(0, T, (E, R)).astype(np.int32)).to(dev())
  for counts in ([R] * E, rng.integers(0, R + 1, E)):
    live = torch.as_tensor(np.asarray(counts, np.int32), device=dev())
    got, want = (torch.full((E, R, D), 7.0, dtype=torch.bfloat16, device=dev()) for _ in range(2))
    for out, full in ((got, True), (want, False)):
      K.expert_mlp(items, w0, b0, w1, b1, out=out, rows_per_expert=live, x_rows=x_rows, full_rows=full)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("tile", range(8, 13))
@pytest.mark.parametrize("E,R,D,M", [
    (130, 64, 640, 776),     # several tiles per workgroup, column tiles and k that end inside
    (40, 33, 768, 2048),     # one and two tiles, part of a row tile
    (3, 128, 712, 1040),     # a full row tile where the tile has 128, else the small tiles
    (9, 1, 640, 648),
])
def test_expert_mlp_tiles_walked_by_a_workgroup(K, monkeypatch, tile, E, R, D, M):
  """The tile-walking kernel for few rows: the checks of the small tiles, and bit for bit what those
  compute (same order of sums), also without a bias and with biases at an odd element."""
  monkeypatch.setenv("VMOE_ROW_TILES", str(tile))
  test_expert_mlp_small_tiles(K, E, R, D, M)
  rng = np.random.default_rng(E)
  mk = lambda scale, *s: to_dev(O.cast(rng.standard_normal(s).astype(np.float32) * scale, O.BF16), O.BF16)
  x, w0, w1 = mk(1, E, R, D), mk(D ** -0.5, E, D, M), mk(M ** -0.5, E, M, D)
  b0, b1 = mk(0.1, E * M + 1)[1:].view(E, M), mk(0.1, E * D + 1)[1:].view(E, D)
  for biases in ((None, None), (b0, b1)):
    for approximate in (True, False):
      args = (x, w0, biases[0], w1, biases[1])
      monkeypatch.setenv("VMOE_ROW_TILES", str(tile))
      got = K.expert_mlp(*args, approximate_gelu=approximate)
      monkeypatch.setenv("VMOE_ROW_TILES", "7")
      want = K.expert_mlp(*args, approximate_gelu=approximate)
      assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("S,E,k,C,spread", [
    (511, 7, 2, 60, 1.0), (513, 8, 1, 70, 1.0), (1925, 7, 4, 300, 1.0), (2048, 4, 2, 512, 0.5), (4100, 32, 2, 130, 1.0),
    (900, 8, 2, 120, 1e-3),        # gates closer than a bin: sorted
    (700, 8, 2, 90, 0.02),         # long bins, counted
    (600, 4, 2, 150, 40.0),        # gates that reach 1 and 0
])
def test_float32_gates_ranked_by_counting(K, S, E, k, C, spread):
  """Batch priority and experts choice over float32 gates (bins by their high halves, low halves and items
  inside a bin) against a stable sort, equal gates and gates one bit apart among them."""
  rng = np.random.default_rng(S)
  G = 2
  logits = (rng.standard_normal((G, S, E)) * spread).astype(np.float32)
  logits[:, 5::7] = logits[:, 3:4]                              # equal gates
  gates = O.softmax(logits).astype(np.float32)
  gates[:, 11::13] = np.nextafter(gates[:, 11::13], np.float32(0))
  g = to_dev(gates)
  val, idx = K.topk(g, k)
  for bpr in (True, False):
    indices, token_slot, slot_token, fill = (to_np(t) for t in K.route_assign(val, idx, E, C, bpr)[:4])
    v, i = to_np(val), to_np(idx)
    for n in range(G):
      order = np.argsort(-v[n, :, 0], kind="stable") if bpr else np.arange(S)
      seen, pos = np.zeros(E, np.int64), np.zeros((S, k), np.int64)
      for j in range(k):
        for s in order:
          pos[s, j] = seen[i[n, s, j]]
          seen[i[n, s, j]] += 1
      np.testing.assert_array_equal(indices[n, ..., 1], pos)
  cols = K.top_items_metrics(g, C)
  want = np.argsort(-gates, axis=1, kind="stable")              # (G, rank, E)
  slot_token = to_np(cols[2]).reshape(E, G, C)
  for n in range(G):
    np.testing.assert_array_equal(slot_token[:, n], (n * S + want[n, :C]).T)


def test_expert_mlp_planned_launch_random_fill(K):
  """bf16 expert products over packed rows with a die-balanced launch plan: random row
  counts (empty, one row, tile boundaries, full), expert counts below and above the
  number of dies, row capacities below and above a tile."""
  rng = np.random.default_rng(11)
  dtype = O.BF16
  for E, R, D, M in [(1, 700, 64, 96), (3, 130, 96, 64), (8, 520, 64, 128), (9, 257, 128, 64),
                     (17, 300, 64, 64), (40, 100, 64, 96), (64, 33, 96, 64),
                     (5, 520, 64, 224), (12, 700, 520, 192)]:   # tile-walking second product
    x = to_dev(O.cast(rng.standard_normal((E, R, D)).astype(np.float32), dtype), dtype)
    w0 = to_dev(O.cast(rng.standard_normal((E, D, M)).astype(np.float32) / 8, dtype), dtype)
    w1 = to_dev(O.cast(rng.standard_normal((E, M, D)).astype(np.float32) / 11, dtype), dtype)
    b0 = to_dev(O.cast(rng.standard_normal((E, M)).astype(np.float32) * 0.1, dtype), dtype)
    b1 = to_dev(O.cast(rng.standard_normal((E, D)).astype(np.float32) * 0.1, dtype), dtype)
    full = K.expert_mlp(x, w0, b0, w1, b1)
    for trial in range(3):
      special = np.asarray([0, 1, 127, 128, 129, 255, 256, 257, R], np.int64)
      rows = np.where(rng.random(E) < 0.5, rng.integers(0, R + 1, E), rng.choice(special, E))
      rows = np.minimum(rows, R).astype(np.int32)
      out = torch.full_like(full, 7.0)
      K.expert_mlp(x, w0, b0, w1, b1, out=out, rows_per_expert=to_dev(rows))
      for e, n in enumerate(rows):
        np.testing.assert_array_equal(to_np(out[e, :n]), to_np(full[e, :n]),
                                      err_msg=f"E={E} R={R} rows={rows.tolist()} expert {e}")
        assert (to_np(out[e, n:]) == 7.0).all(), f"E={E} R={R} rows={rows.tolist()} expert {e}"


def test_expert_mlp_planned_launch_random_fill_on_large_tiles(K, monkeypatch):
  """The same on the tiles that read a plan: these shapes choose the small ones, which need none."""
  monkeypatch.setenv("VMOE_ROW_TILES", "off")
  test_expert_mlp_planned_launch_random_fill(K)


@pytest.mark.parametrize("E,R,D,M,dtype", [c for c in MLP_CASES if c[-1] == O.BF16])
def test_expert_mlp_on_large_tiles(K, monkeypatch, E, R, D, M, dtype):
  monkeypatch.setenv("VMOE_ROW_TILES", "off")
  test_expert_mlp(K, E, R, D, M, dtype, True)


def test_expert_mlp_bfloat16_seeded_shapes_on_large_tiles(K, monkeypatch):
  """The sweep on the large tiles and, where k is no multiple of 32, the register-staged kernel."""
  monkeypatch.setenv("VMOE_ROW_TILES", "off")
  test_expert_mlp_bfloat16_seeded_shapes(K)


def test_expert_mlp_operands_of_2_gib(K):
  """An expert's rows of 2 GiB beside a k that is no multiple of 32: the register-staged kernel (every
  other size takes a kernel that loads through LDS).  Dense, then with a count that ends inside a tile."""
  R, D, M = 1 << 27, 8, 8
  gen = torch.Generator(device=dev()).manual_seed(1)
  mk = lambda scale, *s: torch.randn(s, generator=gen, device=dev(), dtype=torch.bfloat16) * scale
  x, w0, b0, w1, b1 = mk(1, 1, R, D), mk(D ** -0.5, 1, D, M), mk(0.1, 1, M), mk(M ** -0.5, 1, M, D), mk(0.1, 1, D)
  out = K.expert_mlp(x, w0, b0, w1, b1)
  bf = torch.bfloat16
  for at in (0, R // 2 - 100, R - 5000):
    rows = x[0, at:at + 5000].float()
    h = ((rows @ w0[0].float()).to(bf).float() + b0[0].float()).to(bf)
    h = torch.nn.functional.gelu(h.float(), approximate="tanh").to(bf)
    y = ((h.float() @ w1[0].float()).to(bf).float() + b1[0].float()).to(bf)
    np.testing.assert_allclose(to_np(out[0, at:at + 5000]), to_np(y), rtol=2e-2, atol=5e-2, err_msg=f"rows from {at}")
  n = R - 77
  ragged = torch.full_like(out, 7.0)
  K.expert_mlp(x, w0, b0, w1, b1, out=ragged, rows_per_expert=torch.tensor([n], dtype=torch.int32, device=dev()))
  assert torch.equal(ragged[0, :n], out[0, :n]) and bool((ragged[0, n:] == 7.0).all())


@pytest.mark.parametrize("E,R,D,M", [(64, 384, 1024, 128), (32, 1152, 1024, 256), (90, 384, 520, 160)])
def test_expert_mlp_wide_second_product(K, E, R, D, M):
  """Shapes whose second product takes the wide kernel (384 x 256 tiles, eight waves; it runs
  where the tile-walking 256 x 256 kernel does not apply, and VMOE_SECOND_PRODUCT=wide asks
  for it wherever it applies itself): all rows against the oracle, then packed rows with a
  launch plan (row counts around the tile height, empty experts) bit for bit against the
  dense launch."""
  os.environ["VMOE_SECOND_PRODUCT"] = "wide"
  try:
    _wide_second_product(K, E, R, D, M)
  finally:
    del os.environ["VMOE_SECOND_PRODUCT"]


def _wide_second_product(K, E, R, D, M):
  rng = np.random.default_rng(E + R)
  dtype = O.BF16
  x = O.cast(rng.standard_normal((E, R, D)).astype(np.float32), dtype)
  w0 = O.cast(rng.standard_normal((E, D, M)).astype(np.float32) / np.sqrt(D), dtype)
  w1 = O.cast(rng.standard_normal((E, M, D)).astype(np.float32) / np.sqrt(M), dtype)
  b0 = O.cast(rng.standard_normal((E, M)).astype(np.float32) * 0.1, dtype)
  b1 = O.cast(rng.standard_normal((E, D)).astype(np.float32) * 0.1, dtype)
  dx, dw0, db0, dw1, db1 = (to_dev(a, dtype) for a in (x, w0, b0, w1, b1))
  full = K.expert_mlp(dx, dw0, db0, dw1, db1)
  pick = np.unique(np.concatenate([[0, E - 1], rng.integers(0, E, 4)]))
  want = O.mlp_block(x[pick], w0[pick], b0[pick], w1[pick], b1[pick], dtype)
  assert_close(to_np(full)[pick], want, 2e-2, "wide second product")
  nobias = K.expert_mlp(dx, dw0, db0, dw1, None)
  want = O.mlp_block(x[pick[:2]], w0[pick[:2]], b0[pick[:2]], w1[pick[:2]], None, dtype)
  assert_close(to_np(nobias)[pick[:2]], want, 2e-2, "wide second product, no bias")
  special = np.asarray([0, 1, 95, 96, 97, 383, 384, 385, R - 1, R], np.int64)
  for trial in range(3):
    rows = np.where(rng.random(E) < 0.5, rng.integers(0, R + 1, E), rng.choice(special, E))
    rows = np.minimum(rows, R).astype(np.int32)
    out = torch.full_like(full, 7.0)
    K.expert_mlp(dx, dw0, db0, dw1, db1, out=out, rows_per_expert=to_dev(rows))
    got, ref = to_np(out), to_np(full)
    for e, n in enumerate(rows):
      np.testing.assert_array_equal(got[e, :n], ref[e, :n], err_msg=f"rows={rows.tolist()} expert {e}")
      assert (got[e, n:] == 7.0).all(), f"rows={rows.tolist()} expert {e}"


def _sparse_signs(rng, shape, nonzeros, axis):
  """Entries in {-1, 0, 1} with exactly `nonzeros` non-zero entries along `axis`."""
  shape = list(shape)
  n = shape.pop(axis)
  flat = np.zeros((int(np.prod(shape)), n), np.float32)
  for row in flat:
    pos = rng.choice(n, size=min(nonzeros, n), replace=False)
    row[pos] = rng.choice(np.asarray([-1.0, 1.0], np.float32), size=pos.size)
  return np.ascontiguousarray(np.moveaxis(flat.reshape(*shape, n), -1, axis))


@pytest.mark.parametrize("E,R,D,M", [
    (2, 96, 64, 256),         # one-tile-per-workgroup first product (2 k tiles), tile-walking second product
    (3, 200, 72, 136),        # widths outside the fast path: register-staged kernel, k edge
    (64, 384, 1024, 128),     # wide second product
    (2, 300, 256, 2048),      # long k loops on both kernels' steady state
])
def test_matrix_core_results_are_read_whole(K, E, R, D, M):
  """Every accumulator register of the matrix-core loops must be complete when the
  epilogue reads it: a v_mfma_f32_32x32x16_bf16 result read too early comes back with
  its last register stale, which showed as wrong rows 27 and 31 of every 32-row tile (the
  kernels put a fixed gap of wait states between the loop and the first read).  Operands
  are small integers chosen so that every product, sum and rounding step of the MLP is
  exact in bfloat16 and the GELU is the identity (pre-activations of 8 and more): the
  result must equal the float64 answer bit for bit, in particular rows 27 and 31."""
  rng = np.random.default_rng(D + M)
  x = rng.integers(-1, 2, (E, R, D)).astype(np.float32)
  w0 = _sparse_signs(rng, (E, D, M), 8, axis=1)             # |x @ w0| <= 8
  b0 = np.full((E, M), 16.0, np.float32)                    # hidden = 16 + (x @ w0) in [8, 24]
  w1 = _sparse_signs(rng, (E, M, D), 4, axis=1)             # |hidden @ w1| <= 96
  b1 = rng.integers(-3, 4, (E, D)).astype(np.float32)
  hidden = np.einsum("erd,edm->erm", x.astype(np.float64), w0.astype(np.float64)) + 16.0
  assert hidden.min() >= 8 and hidden.max() <= 24
  want = np.einsum("erm,emd->erd", hidden, w1.astype(np.float64)) + b1[:, None, :]
  assert np.abs(want).max() <= 128
  dtype = O.BF16
  got = to_np(K.expert_mlp(*(to_dev(a, dtype) for a in (x, w0, b0, w1, b1)))).astype(np.float64)
  rows = np.arange(R)
  late = (rows % 32 == 27) | (rows % 32 == 31)
  np.testing.assert_array_equal(got[:, late], want[:, late], err_msg="rows 27 / 31 of a 32-row tile")
  np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("E,R,D,M", [(2, 96, 64, 256), (3, 200, 72, 136), (2, 300, 256, 2048)])
def test_matrix_core_results_are_read_whole_on_large_tiles(K, monkeypatch, E, R, D, M):
  """The shapes above that choose the small tiles, on the kernels named beside them."""
  monkeypatch.setenv("VMOE_ROW_TILES", "off")
  test_matrix_core_results_are_read_whole(K, E, R, D, M)


def test_gating_logits_are_read_whole(K):
  """The gating kernel's matrix-core loop under the same check: integer operands, exact
  float32 logits, all rows (27 and 31 of each 32-item tile first)."""
  rng = np.random.default_rng(3)
  G, S, D, E = 3, 100, 256, 32
  x = rng.integers(-2, 3, (G, S, D)).astype(np.float32)
  w = rng.integers(-1, 2, (D, E)).astype(np.float32)
  want = (x.astype(np.float64) @ w.astype(np.float64))          # |sum| <= 512: exact in float32
  want_bf = np.asarray(O.cast(want.astype(np.float32), O.BF16), np.float64)   # the logits are rounded to the dtype
  for dtype, ref in ((O.F32, want), (O.BF16, want_bf)):
    _, _, _, logits = K.gate_topk(to_dev(x, dtype), to_dev(w, dtype), 2, return_logits=True)
    got = to_np(logits).astype(np.float64).reshape(G * S, E)
    rows = np.arange(G * S)
    late = (rows % 32 == 27) | (rows % 32 == 31)
    np.testing.assert_array_equal(got[late], ref.reshape(G * S, E)[late], err_msg=f"{dtype}: rows 27 / 31")
    np.testing.assert_array_equal(got, ref.reshape(G * S, E), err_msg=dtype)


def test_resident_delivery_probe(K):
  """The load-only kernel over shared, L2-resident tiles runs to its end for both request shapes
  and reports the bytes it moved; bad arguments come back as error codes."""
  from vmoe_amd import _hip as H
  buf = torch.zeros(3 * 512 * 1024 + 100, dtype=torch.uint8, device=dev())      # three tiles and a bit
  for seg in (128, 64):
    assert K.resident_delivery_probe(buf, 1024, 8, 2, seg) == 256 * 2 * 8 * 65536
  torch.cuda.synchronize()
  with pytest.raises(H.VmoeError, match="invalid sizes"):
    K.resident_delivery_probe(buf, 1024, 9, 2, 128)          # 9 k tiles of 128 bytes > row
  with pytest.raises(H.VmoeError, match="invalid sizes"):
    K.resident_delivery_probe(buf, 1024, 8, 2, 32)
  with pytest.raises(H.VmoeError, match="invalid sizes"):
    K.resident_delivery_probe(buf[:1000], 1024, 8, 2, 128)   # not one whole tile


def test_operand_delivery_probe(K):
  """The load-only measurement kernel reports the operand bytes of the 256 x 256 tiling
  and refuses what the tiling refuses."""
  from vmoe_amd import _hip as H
  a = torch.randn((3, 700, 256), device=dev()).to(torch.bfloat16)
  bt = torch.randn((3, 520, 256), device=dev()).to(torch.bfloat16)
  moved = K.operand_delivery_probe(a, bt)
  torch.cuda.synchronize()
  assert moved == 3 * 3 * 3 * 512 * 256 * 2          # 3 batches x (3 x 3) tiles x 512 rows x K x 2 bytes
  assert K.operand_delivery_probe(a[0], bt[0]) == 3 * 3 * 512 * 256 * 2
  assert K.operand_delivery_probe(a, bt, k_tile=64) == moved     # same tiles, 128-byte row segments
  torch.cuda.synchronize()
  with pytest.raises(H.VmoeError):                     # K not a multiple of 64
    K.operand_delivery_probe(a[:, :, :96].contiguous(), bt[:, :, :96].contiguous(), k_tile=64)
  with pytest.raises(H.VmoeError):                     # K not a multiple of 32
    K.operand_delivery_probe(a[:, :, :40].contiguous(), bt[:, :, :40].contiguous())
  with pytest.raises(ValueError):
    K.operand_delivery_probe(a.float(), bt.float())


@pytest.mark.parametrize("G,S,E,k,C,D,M", [
    (4, 1568, 32, 2, 100, 256, 512),     # headline routing shapes, a narrow MLP
    (2, 1568, 8, 2, 412, 128, 256),      # few experts, many rows each
    (3, 300, 5, 3, 200, 128, 192),       # expert count that does not divide 256
])
def test_expert_mlp_with_compaction_in_the_planning_launch(K, monkeypatch, G, S, E, k, C, D, M):
  """expert_mlp(compact=...) (vmoe_compact_rows_planned + vmoe_expert_mlp_planned) against
  vmoe_compact_rows followed by vmoe_expert_mlp: the integer maps bit for bit, the output
  rows of kept assignments bit for bit as well (the same kernels run on the same plan)."""
  rng = np.random.default_rng(G * 100 + E)
  gates = O.softmax(rng.standard_normal((G, S, E)).astype(np.float32) * 2)
  val, idx = K.topk(to_dev(gates), k)
  _, token_slot, _, fill = K.route_assign(val, idx, E, C, True)
  items = to_dev(O.cast(rng.standard_normal((G * S, D)), O.BF16), O.BF16)
  w0 = to_dev(O.cast(rng.standard_normal((E, D, M)) / np.sqrt(D), O.BF16), O.BF16)
  w1 = to_dev(O.cast(rng.standard_normal((E, M, D)) / np.sqrt(M), O.BF16), O.BF16)
  b0 = to_dev(O.cast(rng.standard_normal((E, M)) * 0.1, O.BF16), O.BF16)
  b1 = to_dev(O.cast(rng.standard_normal((E, D)) * 0.1, O.BF16), O.BF16)
  w0t, w1t = K.pack_expert_weights(w0), K.pack_expert_weights(w1)
  token_row, rows, row_token = K.compact_rows(fill, token_slot, C)
  want = K.expert_mlp(items, None, b0, None, b1, w0t=w0t, w1t=w1t, rows_per_expert=rows, x_rows=row_token)
  for separate in (False, True):
    if separate:
      monkeypatch.setenv("VMOE_PLAN_SEPARATE_LAUNCH", "1")
    else:
      monkeypatch.delenv("VMOE_PLAN_SEPARATE_LAUNCH", raising=False)
    for _ in range(2):
      got, maps = K.expert_mlp(items, None, b0, None, b1, w0t=w0t, w1t=w1t,
                               compact=(fill, token_slot, C))
      assert (K._last_planned is not None and K._last_planned[8] is got) != separate, "wrong entry points"
      np.testing.assert_array_equal(to_np(maps[0]), to_np(token_row))
      np.testing.assert_array_equal(to_np(maps[1]), to_np(rows))
      r = to_np(rows)
      g_np, w_np = to_np(got), to_np(want)
      rt_g, rt_w = to_np(maps[2]), to_np(row_token)
      for e in range(E):
        np.testing.assert_array_equal(rt_g[e, :r[e]], rt_w[e, :r[e]])
        np.testing.assert_array_equal(g_np[e, :r[e]], w_np[e, :r[e]])
  monkeypatch.delenv("VMOE_PLAN_SEPARATE_LAUNCH", raising=False)


@pytest.mark.parametrize("G,S,E,k,C,D,M", [(4, 1568, 32, 2, 100, 256, 512), (2, 1568, 8, 2, 412, 128, 256),
                                           (3, 300, 5, 3, 200, 128, 192)])
def test_expert_mlp_with_compaction_in_the_planning_launch_on_large_tiles(K, monkeypatch, G, S, E, k, C, D, M):
  """The shapes above choose small tiles for one product or both; here the launch plans both."""
  monkeypatch.setenv("VMOE_ROW_TILES", "off")
  test_expert_mlp_with_compaction_in_the_planning_launch(K, monkeypatch, G, S, E, k, C, D, M)


def test_expert_mlp_hidden_layer_beyond_4_gib(K):
  """A hidden layer of 4.3 GiB: the second product cannot address it with 32-bit byte
  offsets from its start, which the tile-walking kernel needs, so the one-tile-per-
  workgroup kernel (offsets per expert) must take over.  Sampled rows of every expert
  against a float32 restatement on the device."""
  rng = np.random.default_rng(31)
  E, R, D, M = 8, 70000, 64, 4096
  assert E * R * M * 2 >= 1 << 32
  bf = torch.bfloat16
  gen = torch.Generator(device=dev())
  gen.manual_seed(5)
  x = torch.randn((E, R, D), generator=gen, device=dev()).to(bf)
  w0 = (torch.randn((E, D, M), generator=gen, device=dev()) / D ** 0.5).to(bf)
  w1 = (torch.randn((E, M, D), generator=gen, device=dev()) / M ** 0.5).to(bf)
  b0 = (torch.randn((E, M), generator=gen, device=dev()) * 0.1).to(bf)
  b1 = (torch.randn((E, D), generator=gen, device=dev()) * 0.1).to(bf)
  out = K.expert_mlp(x, w0, b0, w1, b1)
  pick = torch.from_numpy(np.unique(np.concatenate(
      [[0, 1, 255, 256, R - 257, R - 2, R - 1], rng.integers(0, R, 50)]))).to(dev())
  for e in range(E):
    h = ((x[e, pick].float() @ w0[e].float()).to(bf).float() + b0[e].float()).to(bf)
    h = torch.nn.functional.gelu(h.float(), approximate="tanh").to(bf)
    y = ((h.float() @ w1[e].float()).to(bf).float() + b1[e].float()).to(bf)
    np.testing.assert_allclose(to_np(out[e, pick]), to_np(y), rtol=2e-2, atol=2e-2, err_msg=f"expert {e}")
  del out, x
  torch.cuda.empty_cache()


@pytest.mark.parametrize("with_bias", [True, False])
def test_expert_mlp_second_product_walks_several_tiles(K, with_bias):
  """The second product's workgroups walk a list of tiles and fetch a tile's first
  operands while they finish the tile before: enough tiles (480 of 256 x 256, 60 per die)
  that most workgroups compute two, dense and over packed rows with a launch plan, the
  last column tile 8 wide.  Checked against a float32 restatement with the bfloat16
  rounding points of flax's Dense (accumulator, + bias) on the device, tolerance one
  bfloat16 step; packed rows against the dense result bit for bit."""
  rng = np.random.default_rng(23)
  E, R, D, M = 16, 2321, 520, 256
  bf = torch.bfloat16
  x = to_dev(O.cast(rng.standard_normal((E, R, D)).astype(np.float32), O.BF16), O.BF16)
  w0 = to_dev(O.cast(rng.standard_normal((E, D, M)).astype(np.float32) / np.sqrt(D), O.BF16), O.BF16)
  w1 = to_dev(O.cast(rng.standard_normal((E, M, D)).astype(np.float32) / np.sqrt(M), O.BF16), O.BF16)
  b0 = to_dev(O.cast(rng.standard_normal((E, M)).astype(np.float32) * 0.1, O.BF16), O.BF16) if with_bias else None
  b1 = to_dev(O.cast(rng.standard_normal((E, D)).astype(np.float32) * 0.1, O.BF16), O.BF16) if with_bias else None
  full = K.expert_mlp(x, w0, b0, w1, b1)
  for e in range(E):                       # one expert at a time: plain 2-D products
    h = (x[e].float() @ w0[e].float()).to(bf)
    if with_bias:
      h = (h.float() + b0[e].float()).to(bf)
    h = torch.nn.functional.gelu(h.float(), approximate="tanh").to(bf)
    y = (h.float() @ w1[e].float()).to(bf)
    if with_bias:
      y = (y.float() + b1[e].float()).to(bf)
    np.testing.assert_allclose(to_np(full[e]), to_np(y), rtol=2e-2, atol=2e-2, err_msg=f"expert {e}")
  rows = rng.integers(0, R + 1, E).astype(np.int32)
  rows[:4] = [R, 0, 257, 1]
  out = torch.full_like(full, 7.0)
  K.expert_mlp(x, w0, b0, w1, b1, out=out, rows_per_expert=to_dev(rows))
  for e, n in enumerate(rows):
    np.testing.assert_array_equal(to_np(out[e, :n]), to_np(full[e, :n]), err_msg=f"expert {e}")
    assert (to_np(out[e, n:]) == 7.0).all(), f"expert {e}"


@pytest.mark.parametrize("which", ["eight", "narrow"])
@pytest.mark.parametrize("E,R,D,M", [
    (64, 1100, 768, 256),     # 960 / 1280 tiles: the kernels' own range; four k tiles (the shortest k they take)
    (40, 1300, 1024, 512),    # four column tiles of 256, five and a third of 192
    (3, 500, 520, 1024),      # forced: a column tile that ends inside the tile, few tiles per die
    (5, 257, 264, 320),       # forced: one row past a tile, k of five tiles
])
def test_expert_mlp_second_product_on_eight_waves(K, monkeypatch, E, R, D, M, which):
  """The eight-wave forms of the second product (two waves per SIMD, output leaving through lane
  exchanges instead of LDS; "eight": 256 x 256 tiles and 32 x 32 x 16 MFMAs, "narrow": 256 x 192
  tiles and 16 x 16 x 32 MFMAs) against the four-wave tile-walking kernel with whole tiles:
  all add the same products in the same order of k, so the outputs must agree bit for bit;
  dense and over packed rows with a launch plan (rows past a count are not written)."""
  rng = np.random.default_rng(E * 100 + M)
  args = [to_dev(O.cast(a, O.BF16), O.BF16) for a in (
      rng.standard_normal((E, R, D)).astype(np.float32),
      rng.standard_normal((E, D, M)).astype(np.float32) / np.sqrt(D),
      rng.standard_normal((E, M)).astype(np.float32) * 0.1,
      rng.standard_normal((E, M, D)).astype(np.float32) / np.sqrt(M),
      rng.standard_normal((E, D)).astype(np.float32) * 0.1)]
  rows = rng.integers(0, R + 1, E).astype(np.int32)
  rows[:3] = [R, 0, 257][:min(3, E)]
  outs = {}
  for kernel in (which, "shared"):
    monkeypatch.setenv("VMOE_SECOND_PRODUCT", kernel)
    monkeypatch.setenv("VMOE_WHOLE_TILES", "1")
    dense = K.expert_mlp(*args)
    ragged = torch.full_like(dense, 7.0)
    K.expert_mlp(*args, out=ragged, rows_per_expert=to_dev(rows))
    outs[kernel] = (to_np(dense), to_np(ragged))
    assert K.expert_mlp_status() == (0, 0)
  monkeypatch.delenv("VMOE_SECOND_PRODUCT")
  monkeypatch.delenv("VMOE_WHOLE_TILES")
  np.testing.assert_array_equal(outs[which][0], outs["shared"][0])
  for e, n in enumerate(rows):
    np.testing.assert_array_equal(outs[which][1][e, :n], outs["shared"][1][e, :n], err_msg=f"expert {e}")
    np.testing.assert_array_equal(outs[which][1][e, :n], outs[which][0][e, :n], err_msg=f"expert {e}")
    assert (outs[which][1][e, n:] == 7.0).all(), f"expert {e}"
  # and against a float32 restatement of one expert
  e = E - 1
  x, w0, b0, w1, b1 = (a[e].float() for a in args)
  bf = torch.bfloat16
  h = ((x @ w0).to(bf).float() + b0).to(bf)
  h = torch.nn.functional.gelu(h.float(), approximate="tanh").to(bf)
  want = ((h.float() @ w1).to(bf).float() + b1).to(bf)
  np.testing.assert_allclose(outs[which][0][e], to_np(want), rtol=2e-2, atol=2e-2)


SHARED_ROUND_CASES = [
    (16, 2321, 520, 1024),    # 60 tiles per die: one round, then 28 tiles shared by 32 workgroups (pieces of 12-16 k tiles)
    (32, 768, 768, 768),      # 36 per die: 4 tiles in pieces of 4 k tiles, chains of three
    (12, 2048, 1024, 512),    # 48 per die: 16 tiles, each halved
    (40, 1300, 768, 1280),    # 90 per die: two rounds, then 26 tiles
    (3, 500, 768, 1024),      # 2-3 tiles per die: no whole round, every tile in many pieces
]


@pytest.mark.parametrize("E,R,D,M", SHARED_ROUND_CASES)
def test_expert_mlp_second_product_shares_partial_round(K, monkeypatch, E, R, D, M):
  """The tile-walking second product cuts the tiles of a die's last, partial round along k
  among the die's workgroups; the float32 sums travel from piece to piece through memory.
  Against the same experts computed one at a time and against a float32 restatement: a cut
  changes the order of one float32 addition per output, so an output may differ from the
  uncut computation by one bfloat16 step (few do); dense and over packed rows with a launch
  plan (random row counts move the cuts); rows past a count are not written."""
  monkeypatch.setenv("VMOE_SECOND_PRODUCT", "shared")      # whatever the launch geometry would choose
  rng = np.random.default_rng(E * 1000 + R)
  bf = torch.bfloat16
  x = to_dev(O.cast(rng.standard_normal((E, R, D)).astype(np.float32), O.BF16), O.BF16)
  w0 = to_dev(O.cast(rng.standard_normal((E, D, M)).astype(np.float32) / np.sqrt(D), O.BF16), O.BF16)
  w1 = to_dev(O.cast(rng.standard_normal((E, M, D)).astype(np.float32) / np.sqrt(M), O.BF16), O.BF16)
  b0 = to_dev(O.cast(rng.standard_normal((E, M)).astype(np.float32) * 0.1, O.BF16), O.BF16)
  b1 = to_dev(O.cast(rng.standard_normal((E, D)).astype(np.float32) * 0.1, O.BF16), O.BF16)
  full = K.expert_mlp(x, w0, b0, w1, b1)
  again = K.expert_mlp(x, w0, b0, w1, b1)
  assert torch.equal(full, again), "two runs of the same launch differ"
  ref = []
  for e in range(E):                       # one expert at a time: plain 2-D products
    h = ((x[e].float() @ w0[e].float()).to(bf).float() + b0[e].float()).to(bf)
    h = torch.nn.functional.gelu(h.float(), approximate="tanh").to(bf)
    ref.append(((h.float() @ w1[e].float()).to(bf).float() + b1[e].float()).to(bf))
  ref = to_np(torch.stack(ref)).astype(np.float64)

  def check(got, n_rows, what):
    for e, n in enumerate(n_rows):
      np.testing.assert_allclose(got[e, :n], ref[e, :n], rtol=2e-2, atol=2e-2, err_msg=f"{what} expert {e}")

  got_full = to_np(full).astype(np.float64)
  bias1 = to_np(b1).astype(np.float64)
  check(got_full, [R] * E, "dense")
  for trial in range(4):
    rows = rng.integers(0, R + 1, E).astype(np.int32)
    rows[:3] = [R, 0, 257]
    out = torch.full_like(full, 7.0)
    K.expert_mlp(x, w0, b0, w1, b1, out=out, rows_per_expert=to_dev(rows))
    got = to_np(out).astype(np.float64)
    check(got, rows, f"rows={rows.tolist()}")
    differ = 0
    for e, n in enumerate(rows):
      assert (got[e, n:] == 7.0).all(), f"rows={rows.tolist()} expert {e}"
      d = np.abs(got[e, :n] - got_full[e, :n])
      # one step of the rounded accumulator (output minus bias), carried through the rounded sum with the bias
      step = 2.0 ** -6 * (np.abs(got_full[e, :n]) + np.abs(bias1[e])[None, :])
      assert (d <= step + 1e-30).all(), "more than one bfloat16 step from the dense launch"
      differ += int((d > 0).sum())
    assert differ <= 0.02 * max(1, int(rows.sum())) * D, f"{differ} outputs differ from the dense launch"
  assert K.expert_mlp_status() == (0, 0), "a piece gave up its wait, or a launch found no plan"


@pytest.mark.parametrize("E,R,D,M", [(12, 2048, 1024, 512), (3, 500, 768, 1024)])
def test_shared_partial_round_is_exact_on_exact_operands(K, monkeypatch, E, R, D, M):
  """The same cuts on operands whose every product, sum and rounding step is exact (small
  integers, GELU the identity): whatever the order of the additions, the result must
  equal the float64 answer bit for bit, dense and over packed rows."""
  monkeypatch.setenv("VMOE_SECOND_PRODUCT", "shared")      # whatever the launch geometry would choose
  rng = np.random.default_rng(D + M)
  x = rng.integers(-1, 2, (E, R, D)).astype(np.float32)
  w0 = _sparse_signs(rng, (E, D, M), 8, axis=1)
  b0 = np.full((E, M), 16.0, np.float32)
  w1 = _sparse_signs(rng, (E, M, D), 4, axis=1)
  b1 = rng.integers(-3, 4, (E, D)).astype(np.float32)
  hidden = np.einsum("erd,edm->erm", x.astype(np.float64), w0.astype(np.float64)) + 16.0
  want = np.einsum("erm,emd->erd", hidden, w1.astype(np.float64)) + b1[:, None, :]
  assert hidden.min() >= 8 and hidden.max() <= 24 and np.abs(want).max() <= 128
  dev_args = [to_dev(a, O.BF16) for a in (x, w0, b0, w1, b1)]
  got = to_np(K.expert_mlp(*dev_args)).astype(np.float64)
  np.testing.assert_array_equal(got, want)
  rows = rng.integers(0, R + 1, E).astype(np.int32)
  rows[0] = R
  out = torch.full((E, R, D), 7.0, dtype=torch.bfloat16, device=dev())
  K.expert_mlp(*dev_args, out=out, rows_per_expert=to_dev(rows))
  got = to_np(out).astype(np.float64)
  for e, n in enumerate(rows):
    np.testing.assert_array_equal(got[e, :n], want[e, :n], err_msg=f"expert {e}")
    assert (got[e, n:] == 7.0).all()
  assert K.expert_mlp_status() == (0, 0), "a piece gave up its wait, or a launch found no plan"


def test_shared_round_wait_that_gives_up_is_loud(K, monkeypatch):
  """The bounded wait of the shared round, forced from the host: with
  VMOE_STREAMK_TEST_GIVE_UP the pieces wait (for a handful of polls) for a deposit count that
  is never reached.  Every kernel still runs to its end; the pieces that gave up are counted
  in the status words and their outputs are NaN, not sums that were never delivered.  The
  count stays when later calls on the same workspace go well."""
  monkeypatch.setenv("VMOE_SECOND_PRODUCT", "shared")      # whatever the launch geometry would choose
  E, R, D, M = 3, 500, 768, 1024           # 2-3 tiles per die: every tile is shared
  rng = np.random.default_rng(5)
  args = [to_dev(O.cast(a, O.BF16), O.BF16) for a in (
      rng.standard_normal((E, R, D)).astype(np.float32),
      rng.standard_normal((E, D, M)).astype(np.float32) / np.sqrt(D),
      rng.standard_normal((E, M)).astype(np.float32) * 0.1,
      rng.standard_normal((E, M, D)).astype(np.float32) / np.sqrt(M),
      rng.standard_normal((E, D)).astype(np.float32) * 0.1)]
  ws = torch.zeros(K.expert_mlp_workspace_bytes(E, R, D, M, torch.bfloat16, prepacked=False),
                   dtype=torch.uint8, device=dev())
  good = K.expert_mlp(*args, workspace=ws)
  torch.cuda.synchronize()
  assert K.expert_mlp_status() == (0, 0)
  assert not torch.isnan(good).any()
  monkeypatch.setenv("VMOE_STREAMK_TEST_GIVE_UP", "4")
  bad = K.expert_mlp(*args, workspace=ws)
  torch.cuda.synchronize()
  monkeypatch.delenv("VMOE_STREAMK_TEST_GIVE_UP")
  abandoned, mismatches = K.expert_mlp_status()
  assert abandoned >= 1 and mismatches == 0
  nan_rows = torch.isnan(bad).any(-1)
  assert nan_rows.any(), "a piece gave up but no output row says so"
  ok = ~nan_rows
  assert torch.equal(bad[ok], good[ok]), "rows that are not NaN must be the product"
  again = K.expert_mlp(*args, workspace=ws)
  torch.cuda.synchronize()
  assert torch.equal(again, good)
  assert K.expert_mlp_status() == (abandoned, 0), "the status words only grow"


def test_expert_mlp_planned_is_repeatable_and_checks_its_plan(K):
  """vmoe_expert_mlp_planned twice after one vmoe_compact_rows_planned (unchanged routing: a
  serving loop, a graph of the experts alone) gives the same output both times -- each call
  resets the exchange counters of its shared round -- and a call on a workspace whose plans
  were never written runs nothing and says so in the status words."""
  _planned_repeats_and_checks_its_plan(K, 4, 1568, 32, 2, 100, 256, 512)


@pytest.mark.parametrize("G,S,E,k,C,D,M,second", [
    (4, 1568, 32, 2, 100, 256, 512, "shared"),     # 64 tiles of the second product: shared pieces on every die
    (4, 1568, 32, 2, 100, 256, 512, "eight"),
    (16, 1568, 8, 2, 400, 768, 1024, None),        # takes the large tiles by itself
])
def test_expert_mlp_planned_on_large_tiles_is_repeatable(K, monkeypatch, G, S, E, k, C, D, M, second):
  """The same where both products read a plan, with the exchange counters of the shared round (its
  memory is part of the workspace) and without."""
  if second is not None:
    monkeypatch.setenv("VMOE_ROW_TILES", "off")
    need = {}
    for which in ("shared", "eight"):
      monkeypatch.setenv("VMOE_SECOND_PRODUCT", which)
      need[which] = K.expert_mlp_workspace_bytes(E, G * C, D, M, torch.bfloat16, prepacked=True)
    assert need["shared"] > need["eight"] + (1 << 24), "the shared kernel does not take the shape"
    monkeypatch.setenv("VMOE_SECOND_PRODUCT", second)
  _planned_repeats_and_checks_its_plan(K, G, S, E, k, C, D, M)


def _planned_repeats_and_checks_its_plan(K, G, S, E, k, C, D, M):
  from vmoe_amd import _hip as H
  rng = np.random.default_rng(23)
  gates = O.softmax(rng.standard_normal((G, S, E)).astype(np.float32) * 2)
  val, idx = K.topk(to_dev(gates), k)
  _, token_slot, _, fill = K.route_assign(val, idx, E, C, True)
  items = to_dev(O.cast(rng.standard_normal((G * S, D)), O.BF16), O.BF16)
  w0 = to_dev(O.cast(rng.standard_normal((E, D, M)) / np.sqrt(D), O.BF16), O.BF16)
  w1 = to_dev(O.cast(rng.standard_normal((E, M, D)) / np.sqrt(M), O.BF16), O.BF16)
  b0 = to_dev(O.cast(rng.standard_normal((E, M)) * 0.1, O.BF16), O.BF16)
  b1 = to_dev(O.cast(rng.standard_normal((E, D)) * 0.1, O.BF16), O.BF16)
  w0t, w1t = K.pack_expert_weights(w0), K.pack_expert_weights(w1)
  first, maps = K.expert_mlp(items, None, b0, None, b1, w0t=w0t, w1t=w1t, compact=(fill, token_slot, C))
  first = first.clone()
  rows = to_np(maps[1])
  for _ in range(2):
    out = K.expert_mlp_replay_planned()
    first_np, out_np = to_np(first), to_np(out)
    for e in range(E):
      np.testing.assert_array_equal(out_np[e, :rows[e]], first_np[e, :rows[e]], err_msg=f"expert {e}")
  assert K.expert_mlp_status() == (0, 0)
  # a workspace that was never planned: every product launch leaves at once
  R = G * C
  ws = torch.randint(0, 255, (K.expert_mlp_workspace_bytes(E, R, D, M, torch.bfloat16, prepacked=True) + (1 << 20),),
                     dtype=torch.uint8, device=dev())
  out = torch.full((E, R, D), 7.0, dtype=torch.bfloat16, device=dev())
  p = H.ExpertMlpParams(H.ptr(items), None, H.ptr(b0), None, H.ptr(b1), H.ptr(w0t), H.ptr(w1t), H.ptr(out),
                        H.ptr(ws), ws.numel(), E, R, D, M, H.BF16, H.GELU_TANH, H.ptr(maps[1]),
                        H.ptr(maps[2]), G * S)
  need = H.lib().vmoe_expert_mlp_workspace_bytes(H.ctypes.byref(p))
  assert need <= ws.numel()
  H.call("vmoe_expert_mlp_planned", p)
  torch.cuda.synchronize()
  addr = H.ctypes.c_void_p()
  H.check(H.lib().vmoe_expert_mlp_status(H.ctypes.byref(p), H.ctypes.byref(addr)), "vmoe_expert_mlp_status")
  words = ws[addr.value - ws.data_ptr():][:8].view(torch.int32).cpu()
  assert int(words[H.MLP_STATUS_PLAN_MISMATCHES]) == 2, "both products must report the missing plan"
  assert int(words[H.MLP_STATUS_ABANDONED_WAITS]) == 0
  assert (to_np(out) == 7.0).all(), "a launch without a valid plan must not write"


@pytest.mark.parametrize("G,S,E,k,C,D,M", [(1, 49, 3, 2, 40, 64, 104), (2, 784, 8, 2, 208, 256, 512),
                                           (16, 1568, 8, 2, 400, 768, 1024)])
def test_expert_mlp_float32_biases(K, G, S, E, k, C, D, M):
  """Float32 biases of a bfloat16 MLP, rounded inside the call (beside the row compaction where there is
  one): the bits of biases rounded beforehand, for both, one of them, one in bfloat16, a strided one,
  and after an edit that raises no version."""
  rng = np.random.default_rng(E + D)
  mk = lambda scale, *s: to_dev((rng.standard_normal(s) * scale).astype(np.float32))
  bf = lambda t: t if t is None else t.to(torch.bfloat16)
  x, xe = bf(mk(1, G * S, D)), bf(mk(1, E, G * C, D))
  kw = dict(w0t=bf(mk(D ** -0.5, E, M, D)), w1t=bf(mk(M ** -0.5, E, D, M)))
  val, idx = K.topk(to_dev(O.softmax(rng.standard_normal((G, S, E)).astype(np.float32))), k)
  _, token_slot, _, fill = K.route_assign(val, idx, E, C, True)
  rows = to_dev(rng.integers(0, G * C + 1, E).astype(np.int32))
  b0, b1 = mk(0.3, E, M), mk(0.3, E, D)
  strided = mk(0.3, D, E).t()

  def both(p0, p1):
    r0, r1 = bf(p0), bf(p1 if p1 is None else p1.contiguous())
    for more in (dict(), dict(rows_per_expert=rows)):
      got, want = (K.expert_mlp(xe, None, a, None, c, out=torch.zeros_like(xe), **kw, **more) for a, c in ((p0, p1), (r0, r1)))
      assert torch.equal(got, want)
    got, maps = K.expert_mlp(x, None, p0, None, p1, compact=(fill, token_slot, C), **kw)
    want, _ = K.expert_mlp(x, None, r0, None, r1, compact=(fill, token_slot, C), **kw)
    for e, n in enumerate(to_np(maps[1])):
      assert torch.equal(got[e, :n], want[e, :n])
    return got, maps

  for p0, p1 in ((b0, b1), (None, b1), (b0, None), (bf(b0), b1), (b0, strided)):
    both(p0, p1)
  b0.data.add_(1)
  both(b0, b1)
  got, maps = K.expert_mlp(x, None, b0, None, b1, compact=(fill, token_slot, C), **kw)
  want = got.clone()
  got.zero_()
  assert K.expert_mlp_replay_planned() is got
  for e, n in enumerate(to_np(maps[1])):
    assert torch.equal(got[e, :n], want[e, :n])


@pytest.mark.parametrize("G,S,E,k,C,D,M", [(1, 196, 8, 2, 52, 768, 3072), (2, 300, 5, 3, 200, 128, 192)])
def test_expert_mlp_planned_over_few_rows(K, G, S, E, k, C, D, M):
  """Products on the small tiles need no plan: vmoe_compact_rows_planned takes such a call all the
  same, and expert_mlp_replay_planned repeats it, not an earlier, larger one."""
  rng = np.random.default_rng(G * S + E)
  mk = lambda scale, *s: to_dev(O.cast(rng.standard_normal(s) * scale, O.BF16), O.BF16)

  def call(G, S, E, k, C, D, M):
    val, idx = K.topk(to_dev(O.softmax(rng.standard_normal((G, S, E)).astype(np.float32))), k)
    _, token_slot, _, fill = K.route_assign(val, idx, E, C, True)
    return K.expert_mlp(mk(1, G * S, D), None, mk(0.1, E, M), None, mk(0.1, E, D), w0t=mk(D ** -0.5, E, M, D),
                        w1t=mk(M ** -0.5, E, D, M), compact=(fill, token_slot, C))

  call(4, 1568, 32, 2, 100, 256, 512)
  out, maps = call(G, S, E, k, C, D, M)
  want, rows = out.clone(), to_np(maps[1])
  assert rows.sum() > 0 and not torch.isnan(want).all()
  out.fill_(7.0)
  assert K.expert_mlp_replay_planned() is out
  for e in range(E):
    np.testing.assert_array_equal(to_np(out[e, :rows[e]]), to_np(want[e, :rows[e]]), err_msg=f"expert {e}")
    assert (to_np(out[e, rows[e]:]) == 7.0).all(), f"expert {e} wrote past its rows"
  assert K.expert_mlp_status() == (0, 0)


def test_expert_mlp_replay_of_items_that_are_a_view(K):
  """A planned call on items that are not contiguous reads a copy of them; repeating it does, too."""
  G, S, E, k, C, D, M = 4, 392, 8, 2, 100, 256, 512
  rng = np.random.default_rng(5)
  mk = lambda scale, *s: to_dev(O.cast(rng.standard_normal(s) * scale, O.BF16), O.BF16)
  val, idx = K.topk(to_dev(O.softmax(rng.standard_normal((G, S, E)).astype(np.float32))), k)
  _, token_slot, _, fill = K.route_assign(val, idx, E, C, True)
  items = mk(1, D, G * S).t()
  assert not items.is_contiguous()
  out, maps = K.expert_mlp(items, None, mk(0.1, E, M), None, mk(0.1, E, D), w0t=mk(D ** -0.5, E, M, D),
                           w1t=mk(M ** -0.5, E, D, M), compact=(fill, token_slot, C))
  want, rows = out.clone(), to_np(maps[1])
  out.fill_(7.0)
  assert K.expert_mlp_replay_planned() is out
  for e in range(E):
    np.testing.assert_array_equal(to_np(out[e, :rows[e]]), to_np(want[e, :rows[e]]), err_msg=f"expert {e}")


@pytest.mark.parametrize("G,S,D,N", [(6, 196, 768, 128), (3, 250, 768, 128), (2, 37, 384, 40),
                                     (4, 100, 512, 64), (2, 256, 256, 8), (1, 1, 768, 8),
                                     (2, 300, 256, 104), (2, 33, 1024, 128), (2, 64, 768, 20)])
def test_soft_route_with_stats(K, G, S, D, N):
  """vmoe_soft_route_stats: the weights are those of vmoe_soft_route bit for bit, and the
  scalars are the means of vmoe/projects/soft_moe/router.py:119-125 of exactly those stored
  weights, whether the routing launch takes the partial sums itself (bfloat16, up to 256 items,
  widths up to 768) or the separate launch runs (the last three shapes)."""
  rng = np.random.default_rng(G * S + N)
  x = to_dev(O.cast(rng.standard_normal((G, S, D)), O.BF16), O.BF16)
  mu = to_dev(O.cast(rng.standard_normal((D, N)) / np.sqrt(D), O.BF16), O.BF16)
  dw0, cw0 = K.soft_route(x, mu, 1.2)
  dw, cw, scalars = K.soft_route(x, mu, 1.2, with_stats=True)
  np.testing.assert_array_equal(to_np(dw), to_np(dw0))
  np.testing.assert_array_equal(to_np(cw), to_np(cw0))
  d, c = to_np(dw).astype(np.float64), to_np(cw).astype(np.float64)
  want = [c.min(axis=2).mean(), c.max(axis=2).mean(), d.min(axis=1).mean(), d.max(axis=1).mean()]
  got = [float(v) for v in scalars]
  np.testing.assert_allclose(got[:4], want, rtol=3e-6)
  assert got[4] == 0.0
  np.testing.assert_allclose(got[:4], [float(v) for v in K.soft_router_stats(cw, dw)][:4], rtol=3e-6)


@pytest.mark.parametrize("G,S,N,dtype", [(3, 50, 16, O.F32), (4, 196, 128, O.BF16), (2, 7, 300, O.BF16), (3, 196, 128, O.F32),
                          (2, 9, 96, O.BF16), (5, 33, 8, O.BF16), (2, 300, 512, O.BF16),
                          (2, 9, 8192, O.BF16), (3, 5, 1024, O.F32),
                          # rows of more than 1 024 pieces, or values where they are no whole pieces
                          (1, 5, 8200, O.BF16), (2, 9, 1030, O.BF16), (3, 20, 1025, O.F32)])
def test_soft_router_stats(K, G, S, N, dtype):
  """The four means of vmoe/projects/soft_moe/router.py:119-125 in one kernel."""
  rng = np.random.default_rng(G + S + N)
  cw = O.cast(O.softmax(rng.standard_normal((G, S, N)).astype(np.float32), axis=2), dtype)
  dw = O.cast(O.softmax(rng.standard_normal((G, S, N)).astype(np.float32), axis=1), dtype)
  got = [float(v) for v in K.soft_router_stats(to_dev(cw, dtype), to_dev(dw, dtype))]
  want = [cw.min(axis=2).mean(), cw.max(axis=2).mean(), dw.min(axis=1).mean(), dw.max(axis=1).mean()]
  np.testing.assert_allclose(got[:4], want, rtol=2e-6)
  assert got[4] == 0.0   # auxiliary_loss


def _wrapper_calls():
  """(entry points, call(K) -> the tensors that it writes) for every wrapper that has two forms."""
  gen = torch.Generator(device=dev()).manual_seed(3)
  bf, f32 = torch.bfloat16, torch.float32
  mk = lambda dtype, *s: torch.randn(s, generator=gen, device=dev()).to(dtype)
  G, S, D, E, k, C, M = 3, 98, 128, 8, 2, 28, 192
  for dtype in (bf, f32):
    x, w, bias = mk(dtype, G, S, D), mk(dtype, D, E), mk(f32, E)
    yield "vmoe_gate_topk", lambda K, x=x, w=w, b=bias: K.gate_topk(x, w, k, logit_bias=b)
    yield "vmoe_gate_topk", lambda K, x=x, w=w: K.gate_topk(x, w, k, return_logits=True)
    gates = torch.softmax(mk(f32, G, S, E), -1).to(dtype)
    yield "vmoe_top_items_metrics", lambda K, g=gates: K.top_items_metrics(g, 30)
    routed = lambda K, g=gates, **kw: K.route_assign(*K.topk(g.float(), k), E, C, True, **kw)
    yield "vmoe_route_assign", routed
    yield "vmoe_route_assign_metrics", lambda K, r=routed, g=gates: (lambda o: (*o[:4], *o[4]))(r(K, metrics=(g, 0.3, 0.7)))
    items, buf, weights = x.view(G * S, D), mk(dtype, E * G * C, D), mk(f32, G * S, k)
    slots = lambda K, r=routed: (lambda o: (o[1].view(G * S, k), o[2]))(r(K))
    yield "vmoe_dispatch", lambda K, x=items, t=slots: (K.dispatch(x, *t(K)),)
    yield "vmoe_combine", lambda K, y=buf, t=slots, w=weights: (K.combine(y, t(K)[0], w),)
    yield ("vmoe_combine_backward_data", lambda K, x=items, t=slots, w=weights:
           (K.combine_backward_data(x, t(K)[0], w, t(K)[1], E * G * C),))
    yield "vmoe_combine_backward_weights", lambda K, x=items, y=buf, t=slots: (K.combine_backward_weights(x, y, t(K)[0]),)
    yield ("vmoe_combine_backward", lambda K, x=items, y=buf, t=slots, w=weights:
           K.combine_backward(x, y, t(K)[0], w, t(K)[1]))
    yield "vmoe_dispatch_backward", lambda K, y=buf, t=slots: (K.dispatch_backward(y, t(K)[0]),)
    pairs = torch.stack([torch.arange(G * S * k, device=dev()) % (E + 1), torch.arange(G * S * k, device=dev()) // 8], -1)
    yield "vmoe_indices_to_slots", lambda K, i=pairs.view(G, S, k, 2): K.indices_to_slots(i, E, C)
    wts = mk(dtype, G, S, E, 5)
    yield "vmoe_einsum_dispatch", lambda K, w=wts, x=x: (K.einsum_dispatch(w, x, x.dtype),)
    yield "vmoe_einsum_combine", lambda K, w=wts, y=mk(dtype, E * G * 5, D): (K.einsum_combine(w, y, y.dtype),)
    yield "vmoe_cast", lambda K, x=x: (K.cast(x, f32 if x.dtype == bf else bf),)
    yield ("vmoe_add_layer_norm", lambda K, r=mk(f32, G, S, D), x=x, s=mk(f32, D), b=mk(f32, D):
           K.add_layer_norm(r, x, s, b, 1e-6, x.dtype))
    if dtype == bf:
      q, kk, v = mk(bf, 2, 37, 3, 64), mk(bf, 2, 41, 3, 64), mk(bf, 2, 41, 3, 64)
      yield "vmoe_attention", lambda K, q=q, kk=kk, v=v: (K.attention(q, kk, v, 0.125),)
    yield ("vmoe_soft_route_stats", lambda K, x=x, mu=mk(dtype, D, 24):
           (lambda o: (*o[:2], *o[2]))(K.soft_route(x, mu, 1.5, with_stats=True)))
    w0, b0, w1, b1 = mk(dtype, E, D, M), mk(dtype, E, M), mk(dtype, E, M, D), mk(dtype, E, D)
    mlp = dict(w0=w0, b0=b0, w1=w1, b1=b1)
    if dtype == bf:
      mlp = dict(mlp, w0=None, w1=None, w0t=w0.transpose(1, 2).contiguous(), w1t=w1.transpose(1, 2).contiguous())
    out = lambda dtype=dtype: torch.full((E, G * C, D), 7.0, dtype=dtype, device=dev())
    yield "vmoe_expert_mlp", lambda K, y=buf, m=mlp, o=out: (K.expert_mlp(y.view(E, G * C, D), out=o(), **m),)
    rows = torch.tensor([0, 1, 63, 64, 65, 84, 7, 30], dtype=torch.int32, device=dev())
    picks = torch.randint(0, G * S, (E, G * C), generator=gen, device=dev(), dtype=torch.int32)
    yield ("vmoe_expert_mlp", lambda K, x=items, m=mlp, o=out, r=rows, p=picks:
           (K.expert_mlp(x, out=o(), rows_per_expert=r, x_rows=p, **m),))

    def packed(K, x=items, m=mlp, o=out, r=routed):
      _, token_slot, _, fill = r(K)
      got, (token_row, n, row_token) = K.expert_mlp(x, out=o(), compact=(fill, token_slot, C), **m)
      return (got, token_row, n, *(row_token[e, :c] for e, c in enumerate(n.tolist())))
    yield ("vmoe_compact_rows_planned" if dtype == bf else "vmoe_compact_rows"), packed


def test_wrappers_make_the_same_call_from_python_and_natively(K):
  """Each wrapper of the layers' calls is made through the native host side or, bracketed for a timing
  sink, from Python: the same entry point with the same parameters, so the same bits."""
  from vmoe_amd import _hip
  for name, call in _wrapper_calls():
    native = call(K)
    sink = {}
    _hip.set_timing_sink(sink)
    try:
      python = call(K)
    finally:
      _hip.set_timing_sink(None)
    assert len(sink.get(name, ())) >= 1, (name, list(sink))
    assert len(native) == len(python), name
    for i, (a, b) in enumerate(zip(native, python)):
      assert (a is None) == (b is None), (name, i)
      if a is not None:
        assert a.dtype == b.dtype and a.shape == b.shape and a.device == b.device, (name, i)
        assert torch.equal(a, b), (name, i, a.dtype)
