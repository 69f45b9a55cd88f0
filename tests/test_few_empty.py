"""The form for few elements where a shared operand stores no entry: nothing of it is read (its
buffer may be empty)."""
from dataclasses import replace

import pytest

from tensorforge_amd import catalog
from tensorforge_amd.emit import small, stream
from tensorforge_amd.emit.tuned import Schedule

from harness import TOL, gpu_run, make_inputs, normwise_error, oracle_outputs


def _small(stored):
  """Geometry of the chain with only the terms ``stored``, and whether it has the form."""
  e = catalog.get('few_empty_term')
  e.generator.generate()
  program = e.generator.get_program()
  pl, _ = stream.plan(program)
  terms = [replace(t, L=t.L or pl.L, l_cols=t.l_cols or pl.l_cols) for t in pl.terms]
  pl = replace(pl, terms=[terms[i] for i in stored])
  k = small._Small(program, e.generator._context, 'x', Schedule(k_block=8), pl)
  return k, k.prepare()


@pytest.mark.parametrize('stored', [(0, 1, 2, 3), (1, 0), (0, 1), (2, 1, 3)])
def test_entries_read_are_stored_ones(stored):
  k, fits = _small(stored)
  assert fits
  for t, (first, cnt, off) in zip(k.pl.terms, k.raw):
    assert first + cnt <= len(t.U.packed) and off + cnt <= k.raw_total
  assert k.raw_total == sum(len(t.U.packed) for t in k.pl.terms)


def test_nothing_stored_at_all():
  assert not _small((1, 2))[1]


@pytest.mark.gpu
@pytest.mark.parametrize('n', [1, 200, 3000, 6000])
def test_against_the_oracle(n, device):
  e, k = catalog.load('few_empty_term')
  host = make_inputs(e, n, seed=n)
  ref = oracle_outputs(e, host, n)
  got = gpu_run(k, e, host, n, device)
  assert normwise_error(got['D'], ref['D'], 12 * 9) <= TOL[e.fp_type]
