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


def test_matrix_core_forms_by_name_refuse_a_second_product_in_place():
  """Its right operand is what the first product wrote."""
  from tensorforge_amd.common.aux import generate_tmp_tensor
  from tensorforge_amd.common.basic_types import Addressing, FloatingPointType
  from tensorforge_amd.common.context import Context
  from tensorforge_amd.common.exceptions import GenerationError
  from tensorforge_amd.common.matrix.tensor import SubTensor, Tensor
  from tensorforge_amd.generators.descriptions import MultilinearDescr
  from tensorforge_amd.generators.generator import Generator
  pair, ident = [[0, -1], [-1, 1]], [[0, 1], [0, 1]]
  D = Tensor([20, 9], Addressing.STRIDED, alias='D')
  descrs = []
  for i in range(2):
    S = Tensor([9, 9], Addressing.STRIDED, alias=f'S{i}')
    K = Tensor([20, 20], Addressing.NONE, alias=f'K{i}')
    T = generate_tmp_tensor([SubTensor(D), SubTensor(S)], pair)
    descrs += [MultilinearDescr(SubTensor(T), [SubTensor(D), SubTensor(S)], pair, ident),
               MultilinearDescr(SubTensor(D), [SubTensor(K), SubTensor(T)], pair, ident, add=i > 0)]
  for emitter in ('mfma_fp64', 'mfma_fp32', 'mfma_bf16x3'):
    g = Generator(descrs, Context('gfx950', 'hip', FloatingPointType.DOUBLE), emitter=emitter)
    with pytest.raises(GenerationError, match='read after the chain writes it'):
      g.generate()
    Generator(descrs[:2], Context('gfx950', 'hip', FloatingPointType.DOUBLE),
              emitter=emitter).generate()


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
