"""Stacks of different widths on forked side streams, which calls take when
their rows are many (_native.SIDE_STREAM_MIN_BYTES): lookups and updates with
the limit at zero equal the same calls on one stream bit for bit, repeatedly
and from a stream of the caller's own, and the limit decides which way a call
goes: by the entries that are known (none at all among them), and an update by
its slot variables too."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from jax_tpu_embedding.sparsecore import _native  # pylint: disable=g-import-not-at-top,wrong-import-position
from jax_tpu_embedding.sparsecore.lib.nn import embedding  # pylint: disable=g-import-not-at-top,wrong-import-position
from test_gpu_streams import _clone, _grads, _ids, _specs_three_stacks, _state, _step  # pylint: disable=g-import-not-at-top,wrong-import-position


@pytest.mark.parametrize("own_stream", [False, True])
@pytest.mark.parametrize("multi_hot", [False, True])
def test_forced_side_streams_equal_one_stream(multi_hot, own_stream,
                                              monkeypatch):
  if not torch.cuda.is_available():
    pytest.skip("no GPU")
  feats = _specs_three_stacks(4096)
  ids = _ids(np.random.default_rng(8), feats, multi_hot)
  grads = _grads(feats, 6)
  init = _state(feats, 4)
  forks = []
  fork = _native.side_streams
  monkeypatch.setattr(_native, "side_streams",
                      lambda n: forks.append(n) or fork(n))
  runs = []
  stream = torch.cuda.Stream() if own_stream else torch.cuda.current_stream()
  for limit in (0, 1 << 60):
    monkeypatch.setattr(_native, "SIDE_STREAM_MIN_BYTES", limit)
    state = _clone(init)
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
      pre, _ = embedding.preprocess_sparse_dense_matmul_input(
          ids, None, feats, 1, 1, num_sc_per_device=1)
      forks.clear()
      for _ in range(3):
        acts = _step(pre, state, feats, grads)
    torch.cuda.synchronize()
    assert bool(forks) == (limit == 0)
    runs.append((state, acts))
  for a, b in zip(runs[0][1], runs[1][1]):
    assert torch.equal(a, b)
  for name, a in runs[0][0].items():
    b = runs[1][0][name]
    for x, y in zip((a.table, *a.slot), (b.table, *b.slot)):
      assert torch.equal(x, y)


def test_what_a_call_counts(monkeypatch):
  if not torch.cuda.is_available():
    pytest.skip("no GPU")
  feats = _specs_three_stacks(4096)
  ids = _ids(np.random.default_rng(8), feats, True)
  state = _state(feats, 4)
  grads = _grads(feats, 6)
  forks = []
  fork = _native.side_streams
  monkeypatch.setattr(_native, "side_streams",
                      lambda n: forks.append(n) or fork(n))
  pre, _ = embedding.preprocess_sparse_dense_matmul_input(
      ids, None, feats, 1, 1, num_sc_per_device=1)
  csr_only = embedding.PreprocessedInput(pre.sparse_dense_matmul_input,
                                         pre.num_minibatches)
  kw = dict(global_device_count=1, num_sc_per_device=1)

  def rows(entries_of):
    return sum(4 * spec.stack_embedding_dim *
               (entries_of(name) + spec.total_sample_count)
               for name, spec in embedding.get_stacked_table_specs(
                   feats).items())

  def forked(limit, call):
    monkeypatch.setattr(_native, "SIDE_STREAM_MIN_BYTES", limit)
    forks.clear()
    call()
    return bool(forks)

  known = rows(lambda n: pre.csr_num_entries[n])
  buffers = rows(lambda n: csr_only.sparse_dense_matmul_input[1][n].numel())
  assert known < buffers
  update = lambda p: lambda: embedding.tpu_sparse_dense_matmul_grad(
      grads, p, state, feats, **kw)
  lookup = lambda p: lambda: embedding.tpu_sparse_dense_matmul(
      p, state, feats, **kw)
  # One slot: half as much again, rounded per stack.
  assert forked(known * 3 // 2 - 3, update(pre))
  assert not forked(known * 3 // 2 + 1, update(pre))
  assert forked(buffers * 3 // 2 - 3, update(csr_only))
  assert forked(known, lookup(pre)) and not forked(known + 1, lookup(pre))
  assert forked(buffers, lookup(csr_only))
  assert not forked(buffers + 1, lookup(csr_only))
  # A batch without ids is known to hold none.
  pre.csr_num_entries = {n: 0 for n in pre.csr_num_entries}
  empty = rows(lambda n: 0)
  assert not forked(empty * 3 // 2 + 1, update(pre))
  torch.cuda.synchronize()
