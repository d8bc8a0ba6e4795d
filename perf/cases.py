"""The work that users of the embedding path have it do, as timed cases.

Each case is one pass through the public entry points of
`jax_tpu_embedding.sparsecore.lib.nn.embedding`:

  preprocess  embedding.preprocess_sparse_dense_matmul_input of one batch of
              one id per sample and feature: the CSR buffers, up to what the
              stats say was written (with more ids per sample how much that
              is depends on the ids, and serve covers the preprocessing);
  lookup      embedding.tpu_sparse_dense_matmul of a preprocessed batch: the
              activations of every feature;
  update      embedding.tpu_sparse_dense_matmul_grad of a preprocessed batch:
              the updated tables and slot variables;
  serve       preprocess and lookup of one request or scored batch;
  train       a whole training step on a new batch: preprocessing enqueued,
              lookup, update, then the batch's stats.

Tables, batches and id distributions are those of this repository's benchmark
configurations (bench.py), smaller tables where three copies would not fit the
card, and generic sizes between them. Ids are drawn from a truncated power law
(or uniformly), which is what categorical features look like: a few rows are
in nearly every sample and most rows are never touched.
"""

import math
import os
import random
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _p in (ROOT, os.path.join(ROOT, "jax-tpu-embedding_amd")):
  if _p not in sys.path:
    sys.path.insert(0, _p)

# What a case holds, with the values that the listed cases leave out:
#   kind         see above
#   tables       tables; table t has dims[t % len(dims)] columns and combiner
#                combiners[t * len(combiners) // tables]
#   features     input features; feature f looks up table f % tables
#   dims         embedding widths, as text ("8,16")
#   vocab_min, vocab_max   rows per table, log-uniform between the two
#   batch        samples
#   ids_min, ids_max       ids per sample and feature (equal: dense input)
#   lengths      "uniform" or "power" (n^-1.5) over [ids_min, ids_max]
#   zipf         exponent of the ids' power law; 0: uniform ids. "1.05,0"
#                alternates between the tables
#   weighted     whether every id has a weight, U(0, 1)
#   combiners    "sum", "mean", "sqrtn", or several as text
#   optimizer    "sgd", "adagrad" or "adam"
#   csr_only     the lookup gets the four CSR arrays and nothing else, as from
#                a preprocessing elsewhere
#   host         ids come as numpy arrays in host memory
#   minibatching enable_minibatching, with limits that split the batch
DEFAULTS = dict(tables=1, dims="128", vocab_min=100_000, vocab_max=100_000,
                batch=1024, ids_min=1, ids_max=1, lengths="uniform",
                zipf="1.1", weighted=False, combiners="sum",
                optimizer="adagrad", csr_only=False, host=False,
                minibatching=False)


def listed():
  # The headline shape: 26 one-hot features over 26 tables in one stack.
  onehot = dict(tables=26, features=26, dims="128", vocab_min=10,
                vocab_max=40_000_000, batch=65536, zipf="1.1")
  # Weighted bags of 20-80 ids over 8 large tables in two stacks.
  weighted = dict(tables=8, features=8, dims="64", vocab_min=10_000_000,
                  vocab_max=10_000_000, batch=32768, ids_min=20, ids_max=80,
                  zipf="1.2", weighted=True, combiners="sqrtn,mean",
                  optimizer="sgd")
  return [
      # An online request: a few samples, ids from the host.
      dict(name="serve_small", kind="serve", tables=4, features=4, dims="32",
           batch=64, ids_max=16, zipf="1.05", combiners="mean", host=True),
      # A small model's training step, where launches and host work count.
      dict(name="train_small", kind="train", tables=1, features=1, dims="16",
           batch=1024, ids_max=16, zipf="1.05", optimizer="sgd"),
      dict(name="onehot_preprocess", kind="preprocess", **onehot),
      dict(name="onehot_lookup", kind="lookup", **onehot),
      dict(name="onehot_update", kind="update", **onehot),
      # The same batch scored: preprocessing, then the lookup.
      dict(name="weighted_serve", kind="serve", **weighted),
      dict(name="weighted_lookup", kind="lookup", **weighted),
      dict(name="weighted_update", kind="update", **weighted),
      # Long dense rows and very hot ids: one feature of 50 ids, Adagrad.
      dict(name="bag_train", kind="train", tables=1, features=1, dims="128",
           vocab_min=20_000_000, vocab_max=20_000_000, batch=131072,
           ids_min=50, ids_max=50, zipf="1.3"),
      # Many features of mixed widths and ragged lengths, shared tables.
      dict(name="mixed_train", kind="train", tables=12, features=40,
           dims="8,16,32,64,128,256", vocab_min=10_000, vocab_max=5_000_000,
           batch=16384, ids_max=500, lengths="power", zipf="0,1.05",
           combiners="mean"),
      # CSR arrays made elsewhere, an odd batch and a width that is padded.
      dict(name="csr_lookup", kind="lookup", tables=6, features=6, dims="100",
           vocab_min=1000, vocab_max=1_000_000, batch=20011, ids_min=0,
           ids_max=30, zipf="1.1", combiners="mean", csr_only=True),
      # Two slot variables at a middle size, few ids per sample.
      dict(name="adam_update", kind="update", tables=10, features=10,
           dims="48", vocab_min=10_000, vocab_max=2_000_000, batch=8192,
           ids_max=10, zipf="1.05", optimizer="adam"),
  ]


def _log_int(rng, lo, hi):
  return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
  """One more case of the same ranges, no dearer than the largest above."""
  while True:
    kind = rng.choice(["preprocess", "lookup", "update", "serve", "train"])
    tables = _log_int(rng, 1, 26)
    ids_max = rng.choice([1, _log_int(rng, 1, 100), _log_int(rng, 1, 100)])
    if kind == "preprocess":
      ids_max = 1
    dims = rng.choice([str(_log_int(rng, 8, 256)), "16", "32", "64", "128",
                       "8,64", "16,128", "32,100"])
    c = dict(
        kind=kind, tables=tables,
        features=tables * rng.choice([1, 1, 1, 2]), dims=dims,
        vocab_min=_log_int(rng, 10, 1000),
        vocab_max=_log_int(rng, 10_000, 20_000_000),
        batch=_log_int(rng, 64, 131072), ids_max=ids_max,
        ids_min=rng.choice([0, 1, ids_max]),
        lengths=rng.choice(["uniform", "uniform", "power"]),
        zipf=rng.choice(["0", "1.05", "1.1", "1.2", "1.3", "0,1.05"]),
        weighted=rng.random() < 0.25,
        combiners=rng.choice(["sum", "mean", "sqrtn"]),
        optimizer=rng.choice(["sgd", "adagrad", "adagrad", "adam"]),
        csr_only=kind in ("lookup", "update") and rng.random() < 0.25,
        host=rng.random() < (0.5 if kind == "serve" else 0.2),
        minibatching=kind == "train" and rng.random() < 0.2)
    if c["lengths"] == "power" or kind == "preprocess":
      c["ids_min"] = max(1, c["ids_min"])
    widest = max(_ints(dims))
    rows = sum(_vocabs(_full(c)))
    ids = c["batch"] * c["features"] * c["ids_max"]
    if (rows * widest <= 2_000_000_000 and ids <= 8_000_000 and
        ids * widest <= 600_000_000 and
        c["batch"] * c["features"] * widest <= 250_000_000 and
        (not c["minibatching"] or ids <= 2_000_000) and
        (not c["host"] or ids <= 1_000_000)):
      return c


# ---------------------------------------------------------------------------
# Layout and inputs.
# ---------------------------------------------------------------------------


def _full(case):
  return {**DEFAULTS, **case}


def _ints(text):
  return [int(x) for x in str(text).split(",")]


def _vocabs(c):
  """Rows of each table: the model's, not the batch's, so no seed."""
  u = np.random.default_rng(0).uniform(
      math.log(c["vocab_min"]), math.log(c["vocab_max"]), size=c["tables"])
  return [int(x) for x in np.floor(np.exp(u) + 1e-6)]


def _tables(c):
  """Per table (vocabulary, dim, combiner, zipf, stack) and the stacks'
  (name, tables, padded dim): tables of one width and combiner share one."""
  dims, comb = _ints(c["dims"]), c["combiners"].split(",")
  zipf = [float(x) for x in str(c["zipf"]).split(",")]
  tabs, stacks = [], {}
  for t, v in enumerate(_vocabs(c)):
    d, m = dims[t % len(dims)], comb[t * len(comb) // c["tables"]]
    name = f"s_{d}_{m}"
    tabs.append((v, d, m, zipf[t % len(zipf)], name))
    stacks.setdefault(name, []).append(t)
  return tabs, stacks


def _round8(n):
  return -(-int(n) // 8) * 8


def _offsets(c):
  """First row of each table in its stack, and rows per stack (tables follow
  each other, each rounded up to 8 rows)."""
  tabs, stacks = _tables(c)
  off, rows = {}, {}
  for name, members in stacks.items():
    pos = 0
    for t in members:
      off[t] = pos
      pos += _round8(tabs[t][0])
    rows[name] = pos
  return off, rows


def _mean_length(c):
  lo, hi = c["ids_min"], c["ids_max"]
  n = np.arange(lo, hi + 1, dtype=np.float64)
  if c["lengths"] == "power":
    p = n ** -1.5
    return float((n * p).sum() / p.sum())
  return float(n.mean())


def _limit(c, features):
  """Ids per partition that a stack of `features` features is sized for: the
  mean count plus what ragged lengths vary by."""
  n = c["batch"] * features
  most = n * c["ids_max"]
  if c["ids_min"] == c["ids_max"]:
    return max(8, _round8(most))
  return max(8, _round8(min(most, 1.05 * _mean_length(c) * n +
                            8 * c["ids_max"] * math.sqrt(n))))


def _specs(c):
  """Feature specs, stacked by width and combiner."""
  from jax_tpu_embedding.sparsecore.lib.nn import embedding_spec  # pylint: disable=g-import-not-at-top
  from jax_tpu_embedding.sparsecore.lib.nn import table_stacking  # pylint: disable=g-import-not-at-top
  import logging  # pylint: disable=g-import-not-at-top

  opt = {"sgd": lambda: embedding_spec.SGDOptimizerSpec(learning_rate=0.01),
         "adagrad": lambda: embedding_spec.AdagradOptimizerSpec(
             learning_rate=0.01, initial_accumulator_value=0.1),
         "adam": lambda: embedding_spec.AdamOptimizerSpec(
             learning_rate=0.001)}[c["optimizer"]]()
  tabs, stacks = _tables(c)
  per_stack = {n: sum(f % c["tables"] in m for f in range(c["features"]))
               for n, m in stacks.items()}
  limits = {n: _limit(c, k) for n, k in per_stack.items()}
  if c["minibatching"]:
    # A third of a partition's ids per minibatch: the batch is split.
    limits = {n: max(256, _round8(v / 3)) for n, v in limits.items()}
  tables = [embedding_spec.TableSpec(
      name=f"t{t:02d}", vocabulary_size=v, embedding_dim=d,
      initializer=embedding_spec.normal(0.01), optimizer=opt, combiner=m,
      max_ids_per_partition=limits[s], max_unique_ids_per_partition=limits[s])
            for t, (v, d, m, _, s) in enumerate(tabs)]
  feats = [embedding_spec.FeatureSpec(
      name=f"f{f:02d}", table_spec=tables[f % c["tables"]],
      input_shape=[c["batch"], c["ids_max"]],
      output_shape=[c["batch"], tabs[f % c["tables"]][1]])
           for f in range(c["features"])]
  level = logging.getLogger().level
  logging.getLogger().setLevel(logging.ERROR)
  for name, members in stacks.items():
    limit = lambda *_, v=limits[name]: v
    table_stacking.stack_tables(
        feats, [f"t{t:02d}" for t in members], 1, 1, stack_name=name,
        stack_to_max_ids_per_partition=limit,
        stack_to_max_unique_ids_per_partition=limit)
  logging.getLogger().setLevel(level)
  return feats


def _ids(c, seed):
  """Per feature (ids int32 on the GPU, row splits int64 on the host, weights
  or None)."""
  tabs, _ = _tables(c)
  host = np.random.default_rng([seed, 7])
  gen = torch.Generator(device="cuda")
  gen.manual_seed(seed * 4 + 1)
  out = []
  lo, hi, batch = c["ids_min"], c["ids_max"], c["batch"]
  for f in range(c["features"]):
    vocab, _, _, a, _ = tabs[f % c["tables"]]
    if lo == hi:
      lens = np.full(batch, lo, np.int64)
    elif c["lengths"] == "power":
      n = np.arange(lo, hi + 1)
      p = n.astype(np.float64) ** -1.5
      lens = host.choice(n, size=batch, p=p / p.sum())
    else:
      lens = host.integers(lo, hi + 1, size=batch)
    splits = np.zeros(batch + 1, np.int64)
    np.cumsum(lens, out=splits[1:])
    n = int(splits[-1])
    u = torch.rand(n, dtype=torch.float64, device="cuda", generator=gen)
    if a == 0:
      k = (u * vocab).floor_()
    else:
      # Inverse of the distribution function of x^-a on [1, vocab + 1).
      span = 1.0 - float(vocab + 1) ** (1.0 - a)
      k = (1.0 - u * span).pow_(1.0 / (1.0 - a)).floor_().sub_(1.0)
    ids = k.clamp_(0, vocab - 1).to(torch.int32)
    w = None
    if c["weighted"]:
      w = torch.rand(n, device="cuda", generator=gen)
    out.append((ids, splits, w))
  return out


def _variables(c, seed):
  """Stack name -> (table, slots...)."""
  tabs, stacks = _tables(c)
  _, rows = _offsets(c)
  gen = torch.Generator(device="cuda")
  gen.manual_seed(seed * 4 + 2)
  out = {}
  for name, members in stacks.items():
    shape = (rows[name], _round8(tabs[members[0]][1]))
    table = torch.empty(shape, device="cuda").normal_(0.0, 0.01,
                                                      generator=gen)
    slots = ()
    if c["kind"] in ("update", "train"):
      if c["optimizer"] == "adagrad":
        slots = (torch.full(shape, 0.1, device="cuda"),)
      elif c["optimizer"] == "adam":
        slots = (torch.zeros(shape, device="cuda"),
                 torch.zeros(shape, device="cuda"))
    out[name] = (table, slots)
  return out


def _gradients(c, seed):
  """Upstream gradients of every feature's activations."""
  tabs, _ = _tables(c)
  gen = torch.Generator(device="cuda")
  gen.manual_seed(seed * 4 + 3)
  return [torch.empty((c["batch"], tabs[f % c["tables"]][1]),
                      device="cuda").normal_(0.0, 1.0, generator=gen)
          for f in range(c["features"])]


# ---------------------------------------------------------------------------
# The passes.
# ---------------------------------------------------------------------------

STEP = 9  # optimizer step of the updates (Adam's bias correction)


def _preprocess(s, enqueue=False):
  fn = (s["embedding"].enqueue_preprocess_sparse_dense_matmul_input if enqueue
        else s["embedding"].preprocess_sparse_dense_matmul_input)
  return fn(s["features"], s["weights"], s["specs"], 1, 1,
            num_sc_per_device=1, enable_minibatching=s["minibatching"])


def prepare(case, seed):
  from jax_tpu_embedding.sparsecore.lib.core import pybind_input_preprocessing  # pylint: disable=g-import-not-at-top
  from jax_tpu_embedding.sparsecore.lib.nn import embedding  # pylint: disable=g-import-not-at-top

  c = _full(case)
  feats, weights = [], []
  for ids, splits, w in _ids(c, seed):
    if c["host"]:
      ids, w = ids.cpu().numpy(), None if w is None else w.cpu().numpy()
    if c["ids_min"] == c["ids_max"]:
      feats.append(ids.reshape(c["batch"], -1))
      weights.append(None if w is None else w.reshape(c["batch"], -1))
    else:
      feats.append(pybind_input_preprocessing.RaggedIds(ids, splits))
      weights.append(None if w is None else
                     pybind_input_preprocessing.RaggedIds(w, splits))
  s = {"embedding": embedding, "kind": c["kind"], "specs": _specs(c),
       "features": feats, "weights": weights if c["weighted"] else None,
       "minibatching": c["minibatching"]}
  if c["kind"] != "preprocess":
    s["variables"] = {
        n: embedding.EmbeddingVariables(t, slots)
        for n, (t, slots) in _variables(c, seed).items()}
  if c["kind"] in ("update", "train"):
    s["gradients"] = _gradients(c, seed)
  if c["kind"] in ("lookup", "update"):
    pre, _ = _preprocess(s)
    if c["csr_only"]:
      pre = embedding.PreprocessedInput(pre.sparse_dense_matmul_input,
                                        pre.num_minibatches)
    s["batch"] = pre
  return s


def _lookup(s, pre):
  return s["embedding"].tpu_sparse_dense_matmul(
      pre, s["variables"], s["specs"], global_device_count=1,
      num_sc_per_device=1, enable_minibatching=s["minibatching"])


def _update(s, pre):
  out = s["embedding"].tpu_sparse_dense_matmul_grad(
      s["gradients"], pre, s["variables"], s["specs"], step=STEP,
      global_device_count=1, num_sc_per_device=1,
      enable_minibatching=s["minibatching"])
  return {n: [v.table, *v.slot] for n, v in out.items()}


def run(s):
  kind = s["kind"]
  if kind == "lookup":
    return _lookup(s, s["batch"])
  if kind == "update":
    return _update(s, s["batch"])
  if kind == "train":
    pre, stats = _preprocess(s, enqueue=True)
    acts = _lookup(s, pre)
    new = _update(s, pre)
    stats.result()
    return {"activations": acts, "variables": new}
  pre, stats = _preprocess(s)
  if kind == "serve":
    return _lookup(s, pre)
  out = {}
  for name in pre.lhs_row_pointers:
    n = int(stats.required_buffer_size_per_sc[name][0])
    out[name] = {"ids": pre.lhs_embedding_ids[name][:n],
                 "samples": pre.lhs_sample_ids[name][:n],
                 "gains": pre.lhs_gains[name][:n],
                 "entries": pre.lhs_row_pointers[name][:1]}
  return out


# ---------------------------------------------------------------------------
# Work, tolerances, exact results.
# ---------------------------------------------------------------------------


def _distinct(vocab, a, draws):
  """Expected distinct values among `draws` draws of the id distribution."""
  if a == 0:
    return -vocab * math.expm1(draws * math.log1p(-1.0 / vocab)
                               if vocab > 1 else -50.0)
  edges = np.unique(np.floor(np.exp(np.linspace(
      0.0, math.log(vocab + 1), 4000))))
  edges[-1] = vocab + 1
  span = 1.0 - float(vocab + 1) ** (1.0 - a)
  cdf = (1.0 - edges ** (1.0 - a)) / span
  count = np.diff(edges)
  p = np.diff(cdf) / count
  return float((count * -np.expm1(draws * np.log1p(-np.minimum(
      p, 1 - 1e-12)))).sum())


def work(case):
  """Bytes: each input element and each touched row read once, each output
  written once. Flops: a multiply and an add per gathered value, and about
  ten operations per updated value."""
  c = _full(case)
  tabs, _ = _tables(c)
  mean = _mean_length(c)
  ids = c["batch"] * mean  # per feature
  feats = [f % c["tables"] for f in range(c["features"])]
  entries = {t: c["batch"] * _distinct(tabs[t][0], tabs[t][3], mean)
             if mean > 1 else ids for t in set(feats)}
  rows = {t: _distinct(tabs[t][0], tabs[t][3], ids * feats.count(t))
          for t in set(feats)}
  slots = {"sgd": 0, "adagrad": 1, "adam": 2}[c["optimizer"]]
  b = fl = 0.0
  kind = c["kind"]
  for t in feats:
    dim, n = tabs[t][1], entries[t]
    if kind in ("preprocess", "serve", "train"):
      b += ids * (8 if c["weighted"] else 4)
      b += 0 if c["ids_min"] == c["ids_max"] else 8 * c["batch"]
    if kind in ("preprocess", "train"):
      b += 12 * n
    if kind in ("lookup", "update"):
      b += 12 * n
    if kind in ("lookup", "serve", "train"):
      b += 4 * dim * c["batch"]
      fl += 2 * n * dim
    if kind in ("update", "train"):
      b += 4 * dim * c["batch"]
      fl += 2 * n * dim
  for t in set(feats):
    dim = tabs[t][1]
    if kind in ("lookup", "serve", "train"):
      b += 4 * dim * rows[t]
    if kind in ("update", "train"):
      b += 8 * dim * rows[t] * (1 + slots)
      fl += 10 * dim * rows[t]
  return {"bytes": b, "flops": fl}


def tolerance(case):
  c = _full(case)
  if c["kind"] == "preprocess":
    return "exact"  # ids and positions; gains follow a fixed float rule
  # 32-bit sums in another order. The hottest rows add up tens of thousands
  # of contributions, hence the larger single difference.
  if c["kind"] in ("lookup", "serve"):
    return {"rel": 1e-6, "max": 2e-5}
  return {"rel": 1e-6, "max": 1e-3}


def _gains(c, combiner, ids, splits, w):
  """The weight of each id in its sample's sum, in 64 bits, and its sample."""
  lens = torch.from_numpy(np.diff(splits)).cuda()
  sample = torch.repeat_interleave(
      torch.arange(c["batch"], device="cuda"), lens)
  g = (torch.ones(ids.numel(), dtype=torch.float64, device="cuda")
       if w is None else w.double())
  if combiner != "sum":
    d = torch.zeros(c["batch"], dtype=torch.float64, device="cuda")
    d.index_add_(0, sample, g if combiner == "mean" else g * g)
    g = g / (d if combiner == "mean" else d.sqrt())[sample]
  return g, sample


def exact(case, seed):
  c = _full(case)
  tabs, stacks = _tables(c)
  off, _ = _offsets(c)
  feats = []
  for f, (ids, splits, w) in enumerate(_ids(c, seed)):
    t = f % c["tables"]
    gain, sample = _gains(c, tabs[t][2], ids, splits, w)
    feats.append((t, ids.long() + off[t], gain, sample))
  if c["kind"] == "preprocess":
    # Entries ascending by (row, sample), the gains of equal ones added up,
    # padded to a multiple of 8 with NaN.
    out = {}
    for name, members in stacks.items():
      # Stacked samples: feature after feature.
      mine = [x for x in feats if x[0] in members]
      total = c["batch"] * len(mine)
      key = torch.cat([r * total + i * c["batch"] + s
                       for i, (_, r, _, s) in enumerate(mine)])
      uniq, inv = torch.unique(key, return_inverse=True)
      g = torch.full((_round8(uniq.numel()),), math.nan, dtype=torch.float64,
                     device="cuda")
      g[:uniq.numel()] = 0.0
      g.index_add_(0, inv, torch.cat([x[2] for x in mine]))
      out[name] = {"ids": None, "samples": None, "gains": g, "entries": None}
    return out
  values = _variables(c, seed)
  acts = []
  if c["kind"] in ("lookup", "serve", "train"):
    for t, rows, gain, sample in feats:
      table, dim = values[tabs[t][4]][0], tabs[t][1]
      a = torch.zeros((c["batch"], dim), dtype=torch.float64, device="cuda")
      for k in range(0, rows.numel(), 2_000_000):
        part = slice(k, k + 2_000_000)
        a.index_add_(0, sample[part],
                     table[rows[part], :dim].double() * gain[part, None])
      acts.append(a)
    if c["kind"] != "train":
      return acts
  grads = _gradients(c, seed)
  new = {}
  for name, members in stacks.items():
    table, slots = values.pop(name)
    touched = torch.unique(torch.cat([x[1] for x in feats
                                      if x[0] in members]))
    g = torch.zeros((touched.numel(), table.shape[1]), dtype=torch.float64,
                    device="cuda")
    for (t, rows, gain, sample), grad in zip(feats, grads):
      if t not in members:
        continue
      at = torch.searchsorted(touched, rows)
      for k in range(0, rows.numel(), 2_000_000):
        part = slice(k, k + 2_000_000)
        up = grad[sample[part]].double() * gain[part, None]
        if up.shape[1] < g.shape[1]:
          up = torch.nn.functional.pad(up, (0, g.shape[1] - up.shape[1]))
        g.index_add_(0, at[part], up)
    old = [x[touched].double() for x in (table, *slots)]
    whole = [x.double() for x in (table, *slots)]
    del table, slots
    if c["optimizer"] == "sgd":
      upd = [old[0] - 0.01 * g]
    elif c["optimizer"] == "adagrad":
      acc = old[1] + g * g
      upd = [old[0] - 0.01 * g / acc.sqrt(), acc]
    else:
      # The hyperparameters are 32-bit scalars.
      step, b1, b2 = STEP + 1, float(np.float32(0.9)), float(np.float32(0.999))
      c2 = math.sqrt(1 - b2 ** step)
      m = old[1] + (1 - b1) * (g - old[1])
      v = old[2] + (1 - b2) * (g * g - old[2])
      alpha = 0.001 * c2 / (1 - b1 ** step)
      upd = [old[0] - alpha * m / (v.sqrt() + 1e-8 * c2), m, v]
    for x, y in zip(whole, upd):
      x[touched] = y
    new[name] = whole
  if c["kind"] == "update":
    return new
  return {"activations": acts, "variables": new}
