"""Chains that read the tensor they write: no form divides their destination into row bands (a later
band would read what an earlier one wrote), and the results agree with the oracle, which reads every
operand of a product before it writes."""
import numpy as np
import pytest

from tensorforge_amd import catalog
from tensorforge_amd.emit import stream

from harness import (TOL, gpu_run, key_of, make_inputs, normwise_error, oracle_outputs, outputs_of)


@pytest.mark.parametrize('tag', list(catalog.IN_PLACE))
def test_one_band(tag):
  e = catalog.get(f'inplace_{tag}')
  e.generator.generate()
  em = e.generator.get_emitted()
  pl, _ = stream.plan(e.generator.get_program())
  assert stream.in_place(pl)
  assert em.schedule.get('row_passes', 1) == 1


def test_bands_where_nothing_is_read_back():
  e = catalog.get('ader7_f64_tuned')
  e.generator.generate()
  pl, _ = stream.plan(e.generator.get_program())
  assert not stream.in_place(pl)
  assert e.generator.get_emitted().schedule['row_passes'] == 2


@pytest.mark.gpu
@pytest.mark.parametrize('tag', list(catalog.IN_PLACE))
def test_against_the_oracle(tag, device):
  e, k = catalog.load(f'inplace_{tag}')
  for n, masked in ((1, False), (203, True), (3000, False)):
    offsets = {key_of(t): 1 + 2 * i for i, t in enumerate(e.generator._global_tensors)
               if t.addressing.name == 'STRIDED'} if masked else None
    flags = (np.arange(n) % 4 != 1).astype(np.uint32) if masked else None
    host = make_inputs(e, n, seed=n, offsets=offsets)
    ref = oracle_outputs(e, host, n, offsets=offsets, flags=flags)
    got = gpu_run(k, e, host, n, device, offsets=offsets, flags=flags)
    for key in outputs_of(e):
      err = normwise_error(got[key], ref[key], e.tensors[key].get_real_volume(),
                           (offsets or {}).get(key, 0))
      print(f'{tag} n={n}: {err:.2e}', flush=True)
      assert err <= TOL[e.fp_type], (n, key, err)
