"""The preprocessing of a stack on one device and one SparseCore, whose sort
reads the sample view and writes the CSR (preprocess.hip, UniqueStack::flat):
sizes around its extraction blocks, its work-groups and the one work-group of
small stacks (16,384 ids); key widths around its digits, each in one
work-group and in the passes of several tiles; inputs of one id, of copies
only, of ids outside the table only; a static buffer smaller than the input
(the general path); and stacks of every route in one call. The route that
merges after the sort gives the same CSR, stats and views bit for bit."""

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


# One pass (8, and 9 of the wide digits), then widths where a pass of wide
# digits replaces two (17, 18, 25-27) and their neighbours.
BITS = [8, 9, 10, 16, 17, 18, 19, 24, 25, 27, 28]


@pytest.mark.parametrize("rows", [1000, 3000])
@pytest.mark.parametrize("bits", BITS)
def test_key_widths_around_the_digits(bits, rows):
  """About 9,500 ids (one work-group) and 28,500: 14 tiles of 2,048."""
  if not torch.cuda.is_available():
    pytest.skip("no GPU")
  rng = np.random.default_rng(bits)
  lens = rng.integers(0, 20, size=rows)
  assert (lens.sum() > 2**14) == (rows > 1000)
  specs = _specs([("a", 2**bits)], len(lens), "sum", 1, 1, 1 << 16)
  feats = [_ragged(rng, lens, 2**bits)]
  _compare((bits, rows), feats, None, specs)


@pytest.mark.parametrize("bits", [17, 26])
def test_wide_digits_of_large_work_groups(bits):
  """More than 2^21 ids: the tiles of 4,096."""
  if not torch.cuda.is_available():
    pytest.skip("no GPU")
  rng = np.random.default_rng(bits)
  specs = _specs([("a", 2**bits)], 1 << 14, "sum", 1, 1, 1 << 22)
  ids = rng.integers(0, 2**bits, size=(1 << 14, 130)).astype(np.int32)
  ids[rng.random(ids.shape) < 0.01] = -3
  _compare((bits, "large"), [ids], None, specs)


@pytest.mark.parametrize("weighted", [False, True])
def test_stacks_of_every_route_in_one_call(weighted):
  """A small, a narrow, a wide and a large wide stack, and one of more ids than
  its buffer has positions (the general path), in one call."""
  if not torch.cuda.is_available():
    pytest.skip("no GPU")
  rng = np.random.default_rng(9)
  specs, feats = [], []
  for name, bits, rows, most, limit, drawn in (
      ("small", 20, 500, 20, 1 << 15, 2**20),
      ("narrow", 16, 3000, 20, 1 << 16, 2**16),
      ("wide", 18, 3000, 20, 1 << 16, 2**18),
      ("large", 17, 1 << 14, 259, 1 << 22, 2**17),
      # Copies of one id: fewer entries than positions, but more ids.
      ("short", 18, 3000, 20, 1 << 12, 1)):
    specs += _specs([(name, 2**bits)], rows, "mean", 1, 1, limit)
    feats.append(_ragged(rng, rng.integers(0, most + 1, size=rows), drawn,
                         bad=0.01))
  assert sum(len(r) for r in feats[3]) > 2**21
  _compare("routes", feats, _weights(rng, feats) if weighted else None, specs)
