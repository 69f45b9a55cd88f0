"""Generation-time features do not depend on how a floating type spells its FMA: the cost model was
trained on sources in which both types counted alike."""
import pytest

from tensorforge_amd import catalog
from tensorforge_amd import workloads as W
from tensorforge_amd.common.basic_types import FloatingPointType
from tensorforge_amd.emit.tuned import Schedule
from tensorforge_amd.tune import features


@pytest.mark.parametrize('knobs', [{}, {'stream': False}, {'dpp': 'builtin'}])
def test_fma_sites_of_both_types(knobs):
  class Candidate:
    emitter = 'tuned'

    @staticmethod
    def knobs():
      return knobs
  sites = []
  for fp in (FloatingPointType.DOUBLE, FloatingPointType.FLOAT):
    catalog._REGISTRY['_sites'] = lambda fp=fp: catalog._wl_entry(
      W.ader_volume(fp, b=10), 'tuned', Schedule(**knobs))
    try:
      e = catalog.get('_sites')
    finally:
      del catalog._REGISTRY['_sites']
    e.generator.generate()
    f = features.features(e.generator, Candidate, 1000, {'kind': 'fused'})
    sites.append(f[features.NAMES.index('log2_fma_sites')])
  assert sites[0] == sites[1]
