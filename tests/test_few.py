"""The vector form for few elements (``emit.small``): its geometry on the CPU, the chains that get
it, and its results on both sides of every edge of a launch."""
from dataclasses import replace

import numpy as np
import pytest
import torch

from tensorforge_amd import catalog
from tensorforge_amd import workloads as W
from tensorforge_amd.common.basic_types import FloatingPointType
from tensorforge_amd.emit import small, stream
from tensorforge_amd.emit.tuned import Schedule

from harness import (TOL, gpu_run, key_of, make_inputs, normwise_error, oracle_outputs,
                     outputs_of)


def _emitted(name):
  e = catalog.get(name)
  e.generator.generate()
  return e, e.generator.get_emitted()


@pytest.mark.parametrize('name', [f't_few_{t}_auto' for t in catalog.FEW_EDGES] +
                         ['ader_f64_tuned', 'ader_f32_tuned'])
def test_regions_and_rows(name):
  e, em = _emitted(name)
  assert em.few is not None and 0 < em.few_limit
  program = e.generator.get_program()
  pl, _ = stream.plan(program)
  pl = replace(pl, terms=[replace(t, L=t.L or pl.L, l_cols=t.l_cols or pl.l_cols)
                          for t in pl.terms])
  k = small._Small(program, e.generator._context, 'x', Schedule(k_block=8), pl)
  assert k.prepare()
  # the parts' rows are the destination's, their entries all stored ones
  assert [r for p in k.parts for r in range(*p.pl.rows)] == list(range(*pl.rows))
  assert sum(p.nu for p in k.parts) == em.schedule['shared_entries']
  assert len(k.parts) <= small.WAVES
  # rows a wavefront forms temporaries of: every row, none past the last
  rows = -(-k.K // small.WAVES)
  starts = [min(w * rows, k.K - rows) for w in range(small.WAVES)]
  assert min(starts) == 0
  assert {s + j for s in starts for j in range(rows)} == set(range(k.K))
  # pieces: inside the element's window, each entry once, regions apart
  regions = []
  for p in k.xstage + [k.out] + [p for _, st in k.wstage for _, _, _, p in st]:
    seen = set()
    for t in range(small.THREADS):
      run, piece, e0 = t % p.per_element // p.runs, t % p.runs * p.per, t // p.per_element
      if e0 >= p.step:
        continue
      h = max(0, piece - (p.rows - p.per)) if p.moved else 0
      for el in range(e0, k.elements, p.step):
        g = p.first + run * p.col_stride + piece - h
        start = p.first + run * p.col_stride
        assert start <= g and g + p.per <= start + p.rows and g + p.per <= p.arg.element_stride
        at = p.lds_base + el * p.lds_elem + run * p.lds_run + piece
        assert not seen & set(range(at, at + p.per))
        seen |= set(range(at, at + p.per))
    assert len(seen) == k.elements * p.per_element * p.per
    regions.append((min(seen), max(seen) + 1))
  (x0, x1), (d0, d1), *weights = regions
  assert k.total <= x0 == d0 and max(x1, d1) <= k.wbase0
  assert all(k.wbase0 <= a and b <= k.tbase for a, b in weights)
  # the shared operands as stored, and the order's table
  assert k.tbase + k.raw_total <= k.lds_bytes // k.size
  for p in k.parts:
    for _, ti, entry in p.seq:
      lo, n, off = k.raw[ti]
      assert 0 <= entry[2] - lo < n and off + n <= k.raw_total


def test_chains_without_the_form():
  def few(name):
    return _emitted(name)[1].few
  assert few('ader_dense_f64_tuned') is None and few('deriv_f64_tuned') is None
  w = W.ader_volume(FloatingPointType.DOUBLE, b=84)      # temporaries and entries exceed LDS
  catalog._REGISTRY['_few_84'] = lambda: catalog._wl_entry(w, 'tuned')
  catalog._REGISTRY['_few_explicit'] = lambda: catalog._wl_entry(
    W.ader_volume(FloatingPointType.DOUBLE), 'tuned', Schedule())
  try:
    assert few('_few_84') is None and few('_few_explicit') is None
  finally:
    del catalog._REGISTRY['_few_84'], catalog._REGISTRY['_few_explicit']


@pytest.mark.gpu
@pytest.mark.parametrize('tag', list(catalog.FEW_EDGES))
def test_both_sides_of_the_limit(tag):
  e, k = catalog.load(f't_few_{tag}_auto')
  _, em = _emitted(f't_few_{tag}_auto')
  group = em.few.elements_per_block
  dev = torch.device('cuda:0')
  for n in (1, group - 1 or 1, group, group + 1, em.few_limit, em.few_limit + 1):
    some = n <= group + 1
    offsets = {key_of(t): 1 + 2 * i for i, t in enumerate(e.generator._global_tensors)
               if t.addressing.name == 'STRIDED'} if some else None
    flags = (np.arange(n) % 4 != 1).astype(np.uint32) if some else None
    host = make_inputs(e, n, seed=n, offsets=offsets)
    ref = oracle_outputs(e, host, n, offsets=offsets, flags=flags)
    got = gpu_run(k, e, host, n, dev, offsets=offsets, flags=flags)
    for key in outputs_of(e):
      err = normwise_error(got[key], ref[key], e.tensors[key].get_real_volume(),
                           (offsets or {}).get(key, 0))
      assert err <= TOL[e.fp_type], (n, key, err)
