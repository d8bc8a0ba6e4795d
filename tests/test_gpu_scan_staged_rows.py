"""Weighted rows at the edges of the extraction's 32-id comparison masks
(preprocess.hip, ScanStagedRow): lengths around 8, 32, 64, 96 and 128 ids with
one, few or many distinct ids, so that copies fall before, on and after every
mask boundary, and a dense feature of 33. The route that merges after the sort
gives the same CSR, gains, stats and views bit for bit."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from test_gpu_grouping_routes import _compare, _ragged, _specs, _weights  # pylint: disable=g-import-not-at-top,wrong-import-position

EDGES = [0, 1, 2, 7, 8, 9, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 128, 129]


@pytest.mark.parametrize("combiner", ["sum", "mean", "sqrtn"])
@pytest.mark.parametrize("vocab", [1, 3, 64, 5000])
def test_copies_across_mask_edges(combiner, vocab):
  if not torch.cuda.is_available():
    pytest.skip("no GPU")
  rng = np.random.default_rng(vocab)
  lens = rng.permutation(np.repeat(EDGES, 8))
  specs = _specs([("a", vocab), ("b", vocab)], len(lens), combiner, 1, 1,
                 1 << 16)
  feats = [_ragged(rng, lens, vocab, bad=0.02),
           rng.integers(0, vocab, size=(len(lens), 33)).astype(np.int32)]
  _compare((combiner, vocab), feats, _weights(rng, feats), specs)
