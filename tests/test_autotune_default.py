"""The autotuner's timed methods time the kernel the library takes without a schedule."""
import pytest

from tensorforge_amd import workloads as W
from tensorforge_amd.common.basic_types import FloatingPointType
from tensorforge_amd.tune import autotune as at

F64, F32 = FloatingPointType.DOUBLE, FloatingPointType.FLOAT


@pytest.mark.parametrize('fp, sparse, what', [
  (F64, False, 'matrix'), (F32, False, 'matrix'), (F64, True, 'few'), (F32, True, 'few')])
def test_default_of_a_volume_chain(fp, sparse, what):
  w = W.ader_volume(fp, b=20, sparse_k=sparse)
  cands, _ = at.candidates(w.descrs, fp, 4096, 'atd')
  cand, g = at.default_form(w.descrs, fp, cands, 'atd')
  assert cand.label == 'default' and all(g is not other for _, other in cands)
  em = g.get_emitted()
  assert em.schedule.get('matrix') == 'mfma' if what == 'matrix' else em.few is not None
  # one object holds them all, each under its own name
  every = at._with_default(cands, (cand, g))
  names = [x.get_base_name() for _, x in every]
  assert len(set(names)) == len(names) == len(cands) + 1


@pytest.mark.parametrize('name', ['t_gemm_ptr_auto', 't_gemm_NT_auto', 't_three_index_auto'])
def test_default_among_the_candidates(name):
  from tensorforge_amd import catalog
  e = catalog.get(name)
  cands, _ = at.candidates(e.descrs, e.fp_type, 4096, 'atd')
  cand, g = at.default_form(e.descrs, e.fp_type, cands, 'atd')
  assert any(g is other for _, other in cands) and cand.label != 'default'
  assert at._with_default(cands, (cand, g)) is cands


@pytest.mark.parametrize('k', [1, 2, 3, 50])
@pytest.mark.parametrize('method', ['pruned', 'exhaustive'])
def test_what_is_timed(monkeypatch, method, k):
  w = W.ader_volume(F64, b=20, sparse_k=False)

  class Net:
    def predict(self, features):
      return [float(i) for i in range(len(features))]
  monkeypatch.setattr(at, 'cost_model', lambda device: Net())
  monkeypatch.setattr(at.M, 'feature_matrix', lambda recs: recs)
  seen = []

  def time(cands, idx, *a):
    seen.extend(idx)
    return {cands[i][0].label: 2.0 - (cands[i][0].label == 'default') for i in idx}
  monkeypatch.setattr(at, '_time', time)
  choice = at.autotune(w.descrs, F64, 4096, method=method, k=k, build_dir='unused')
  assert choice.label == 'default' and choice.generator.get_emitted().schedule['matrix'] == 'mfma'
  assert len(set(seen)) == len(seen) and 'mfma_fp64' in choice.timed
  predicted = [x for x in choice.timed if x in choice.predicted]
  if method == 'pruned':
    assert len(predicted) == max(2, min(k, len(choice.predicted)))
  else:
    assert set(choice.predicted) <= set(choice.timed)
