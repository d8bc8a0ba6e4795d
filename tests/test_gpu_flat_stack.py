"""The preprocessing of a stack on one device and one SparseCore, whose sort
reads the sample view and writes the CSR (preprocess.hip, UniqueStack::flat):
sizes around its extraction blocks, its work-groups and the one work-group of
small stacks (16,384 ids), key widths
around its digits, inputs of
one id, of copies only, of ids outside the table only, and a static buffer
smaller than the input (the general path). The route that merges after the
sort gives the same CSR, stats and views bit for bit."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from test_gpu_grouping_routes import _compare, _ragged, _specs, _weights  # pylint: disable=g-import-not-at-top,wrong-import-position


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("ids", [1, 255, 256, 257, 1023, 1025, 4097, 16383,
                                 16384, 16385, 40000])
def test_sizes_around_the_work_groups(ids, weighted):
  if not torch.cuda.is_available():
    pytest.skip("no GPU")
  rng = np.random.default_rng(ids)
  lens = np.bincount(rng.integers(0, 1 + ids // 9, size=ids))
  vocab = 5 if ids == 1023 else 3000 if ids < 16384 else 2_000_000
  specs = _specs([("a", vocab)], len(lens), "mean", 1, 1, 1 << 16)
  feats = [_ragged(rng, lens, vocab, bad=0.01 if ids > 1000 else 0)]
  _compare((ids, weighted), feats, _weights(rng, feats) if weighted else None,
           specs)


@pytest.mark.parametrize("what", ["copies", "outside", "small buffer"])
def test_nothing_left_or_little_room(what):
  if not torch.cuda.is_available():
    pytest.skip("no GPU")
  rng = np.random.default_rng(3)
  lens = np.full(300, 20)
  feats = [_ragged(rng, lens, 1 if what != "outside" else 50,
                   bad=1.0 if what == "outside" else 0)]
  limit = 512 if what == "small buffer" else 1 << 14
  specs = _specs([("a", 50)], len(lens), "sum", 1, 1, limit)
  _compare(what, feats, None, specs)


@pytest.mark.parametrize("bits", [8, 9, 10, 16, 17, 18, 19, 24, 25, 27, 28])
def test_key_widths_around_the_digits(bits):
  """Key widths where one pass of wider digits replaces two, and their
  neighbours, over more than one of either tile."""
  if not torch.cuda.is_available():
    pytest.skip("no GPU")
  rng = np.random.default_rng(bits)
  lens = rng.integers(0, 20, size=1000)
  specs = _specs([("a", 2**bits)], len(lens), "sum", 1, 1, 1 << 16)
  feats = [_ragged(rng, lens, 2**bits)]
  _compare(bits, feats, None, specs)
