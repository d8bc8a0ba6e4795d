"""Lookups of narrow rows around the entries from which a sub-group takes a
range twice as long (segreduce.h, TakesLong), for the 4-, 8- and 16-lane
layouts with 4- and 16-byte loads, dense and per-feature activations.

With tables, gradients and gains of small integers every order of summation is
exact, and the results equal a plain index_add bit for bit (the updates of the
same entries too; their ranges have one length). With random floats the two
lengths still add up in one order: neither the buffer that the entries came in
nor what the caller says of their number changes a bit, and the sums are as
close to 64 bits as sums of short pieces are."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
  if not torch.cuda.is_available():
    pytest.skip("no GPU")
  torch.cuda.set_device(0)


from jax_tpu_embedding.sparsecore.lib.core.primitives import _device  # pylint: disable=g-import-not-at-top,wrong-import-position
from jax_tpu_embedding.sparsecore.lib.core.primitives import sparse_dense_matmul_csr as fwd  # pylint: disable=g-import-not-at-top,wrong-import-position
from jax_tpu_embedding.sparsecore.lib.core.primitives import sparse_dense_matmul_grad_with_sgd as sgd  # pylint: disable=g-import-not-at-top,wrong-import-position

LONG = 1 << 19
DIMS = (3, 13, 16, 20, 64)  # 4, 16, 4, 8 and 16 lanes


def _csr(rng, n, entries, rows, batch):
  """`entries` entries ascending by (row, sample) in a buffer of n: a hot row
  over many blocks, rows of two to forty entries, rows of one; samples of one
  to many entries, and some of none."""
  sizes = np.r_[30000, rng.choice([1, 1, 1, 2, 3, 40], size=entries)]
  sizes = sizes[:np.searchsorted(np.cumsum(sizes), entries) + 1]
  sizes[-1] -= sizes.sum() - entries
  rng.shuffle(sizes)
  assert len(sizes) <= rows
  eid = np.repeat(np.sort(rng.choice(rows, len(sizes), replace=False)), sizes)
  # Distinct ascending samples of a run: every seventh from a random one.
  k = np.arange(entries) - np.repeat(np.cumsum(sizes) - sizes, sizes)
  first = rng.integers(0, batch - batch // 8 - 7 * 40, size=len(sizes))
  sid = np.where(np.repeat(sizes, sizes) > 40, k,
                 np.repeat(first, sizes) + 7 * k)
  gains = rng.integers(1, 4, size=entries)
  out = [np.full(n, 2**31 - 1, np.int32), np.full(n, 2**31 - 1, np.int32),
         np.full(n, np.nan, np.float32)]
  for o, x in zip(out, (eid, sid, gains)):
    o[:entries] = x
  rp = np.zeros(8, np.int32)
  rp[0] = entries
  return (rp, *out), eid, sid, gains


@pytest.mark.parametrize("mapped", [False, True])
@pytest.mark.parametrize("dim", DIMS)
def test_long_ranges_are_exact(dim, mapped):
  rng = np.random.default_rng(dim)
  batch, rows = 40000, 300_000 if dim < 20 else 150_000
  for n, entries in ((LONG - 1, LONG - 9), (LONG, LONG - 1000),
                     (LONG + 777, LONG + 777)):
    csr, eid, sid, gains = _csr(rng, n, entries, rows, batch)
    dev = [torch.from_numpy(x).cuda() for x in csr]
    table = torch.from_numpy(rng.integers(-4, 5, size=(rows, dim))).float()
    grad = torch.from_numpy(rng.integers(-4, 5, size=(batch, dim))).float()
    e, s = torch.from_numpy(eid).long(), torch.from_numpy(sid).long()
    g = torch.from_numpy(gains).float()[:, None]
    act = torch.zeros(batch, dim).index_add_(0, s, table[e] * g)
    up = torch.zeros(rows, dim).index_add_(0, e, grad[s] * g)
    kw = dict(max_ids_per_partition=n, max_unique_ids_per_partition=n,
              num_sc_per_device=1, csr_num_entries=entries)
    t_dev = table.cuda()
    blocks, width, grad_dev = None, dim, grad.cuda()
    if mapped:  # three blocks, the middle one narrower, a gap before the last
      width = dim - (4 if dim % 4 == 0 else 1)
      cut = [(0, 10001, dim), (10001, 17000, width), (30000, 10000, dim)]
      blocks = _device.RowBlocks(batch, dim, [
          (a, torch.full((k, w), 7.0, device="cuda"), w) for a, k, w in cut])
      masked = torch.zeros_like(grad)
      for a, k, w in cut:
        masked[a:a + k, :w] = grad[a:a + k, :w]
      up = torch.zeros(rows, dim).index_add_(0, e, masked[s] * g)
      grad_dev = _device.RowBlocks(batch, dim, [
          (a, grad[a:a + k, :w].contiguous().cuda(), w) for a, k, w in cut])
    got = fwd.tpu_sparse_dense_matmul_csr_primitive.bind(
        *dev, 1, t_dev, device_batch_size=batch, activation_blocks=blocks,
        **kw)
    if mapped:
      for (a, out, w), (_, k, _) in zip(blocks.blocks, cut):
        assert torch.equal(out.cpu(), act[a:a + k, :w])
    else:
      assert torch.equal(got.cpu(), act)
    sgd.tpu_sparse_dense_matmul_grad_with_sgd_primitive.bind(
        *dev, 1, t_dev, grad_dev, 0.5, **kw)
    assert torch.equal(t_dev.cpu(), table - up * 0.5)


@pytest.mark.parametrize("dim", DIMS)
def test_one_order_whatever_the_buffer_and_the_count(dim):
  rng = np.random.default_rng(dim + 1)
  batch, rows = 40000, 300_000
  table = torch.from_numpy(
      rng.normal(size=(rows, dim)).astype(np.float32)).cuda()
  for entries in (LONG // 2 - 5, LONG + 4097):
    csr, eid, sid, _ = _csr(rng, entries, entries, rows, batch)
    gains = rng.random(entries, dtype=np.float32)
    results = []
    # The buffer's positions, and the entry count that the caller gives (None:
    # unknown, the buffer's size stands in; a small count asks for the short
    # ranges, unless the buffer is much larger).
    for n, count in ((entries, entries), (entries, None), (entries, 1000),
                     (3 * LONG, entries), (3 * LONG, None), (3 * LONG, 1000),
                     (4 * LONG, 1000)):
      dev = [torch.from_numpy(csr[0]).cuda()]
      for x, fill in ((eid.astype(np.int32), 2**31 - 1),
                      (sid.astype(np.int32), 2**31 - 1), (gains, np.nan)):
        y = np.full(n, fill, x.dtype)
        y[:entries] = x
        dev.append(torch.from_numpy(y).cuda())
      results.append(fwd.tpu_sparse_dense_matmul_csr_primitive.bind(
          *dev, 1, table, device_batch_size=batch, max_ids_per_partition=n,
          max_unique_ids_per_partition=n, num_sc_per_device=1,
          csr_num_entries=count))
    for k, other in enumerate(results[1:]):
      assert torch.equal(results[0], other), (entries, k)
    # A sum of m products: pieces of at most 16 entries (one rounding each,
    # the products being fused), at most 16 pieces, and one addition per
    # doubling or block after that.
    e, s = torch.from_numpy(eid).long(), torch.from_numpy(sid).long()
    w = torch.from_numpy(gains).double()[:, None]
    t = table.cpu().double()
    exact = torch.zeros(batch, dim, dtype=torch.float64)
    size = torch.zeros(batch, dim, dtype=torch.float64)
    exact.index_add_(0, s, t[e] * w)
    size.index_add_(0, s, (t[e] * w).abs())
    bound = (16 + 16 + 32) * 2.0**-24 * size
    assert bool(((results[0].cpu().double() - exact).abs() <= bound).all())
