"""Masked launches and extra offsets through the matrix-core and vector forms of both types.

20,011 elements (more than one round of a workgroup, a partial last set), every per-element operand behind
an odd number of unused entries, masks that skip single elements, whole sets of 16 and everything;
every element is compared with the plain launcher of the same chain. Normwise per element 1e-12
FP64, 1e-5 FP32.
"""
import numpy as np
import pytest

from tensorforge_amd import catalog

from harness import TOL, gpu_run, key_of, make_inputs, normwise_error, outputs_of

pytestmark = pytest.mark.gpu

N = 20011
MASKS = {
  'all': np.ones(N, bool),
  'single': np.arange(N) % 5 != 3,
  'runs': np.arange(N) // 37 % 3 == 1,
  'few': np.arange(N) % 1013 == 7,
  'none': np.zeros(N, bool),
}
ENTRIES = ['ader_f32_tuned', 'ader_dense_f64_tuned', 'ader_dense_f32_tuned', 'ader7_f64_tuned',
           'gemm_f64_tuned', 'gemm_f32_tuned', 'flux_local_mod_f64_tuned',
           'flux_neigh_mod_f64_tuned', 'deriv_f64_tuned', 'deriv_na_f64_tuned']
PLAIN = {name: name.rsplit('_', 1)[0] + '_plain' for name in ENTRIES}
PLAIN.update({f'matrix_{form}_{t}': f't_matrix_{t}_plain' for form in ('staged', 'direct')
              for t in catalog.MATRIX_EDGES})


@pytest.mark.parametrize('name', list(PLAIN))
def test_masked_with_offsets(name, device):
  et, kt = catalog.load(name)
  ep, kp = catalog.load(PLAIN[name])
  keys = [key_of(t) for t in ep.generator._global_tensors if t.addressing.name == 'STRIDED']
  offsets = {k: 3 + 2 * i for i, k in enumerate(keys)}
  host = make_inputs(ep, N, seed=29, offsets=offsets)
  for tag, mask in MASKS.items():
    flags = mask.astype(np.uint32)
    print(f'{name}: mask {tag}', flush=True)
    a = gpu_run(kp, ep, host, N, device, offsets=offsets, flags=flags)
    b = gpu_run(kt, et, host, N, device, offsets=offsets, flags=flags)
    for t in ep.generator._global_tensors:
      key = key_of(t)
      if key not in outputs_of(ep):
        continue
      off, vol = offsets.get(key, 0), t.get_real_volume()
      np.testing.assert_array_equal(b[key][:off], host[key][:off])
      rows = lambda x: x[off:off + N * vol].reshape(N, vol)
      np.testing.assert_array_equal(rows(b[key])[~mask], rows(host[key])[~mask])
      assert normwise_error(b[key], a[key], vol, off) <= TOL[et.fp_type]


@pytest.mark.parametrize('tag', ['gemm_16x16_q1', 'gemm_18x21_q8', 'gemm_7x5_f32', 'chain_13x6x29_q4'])
def test_more_sets_than_a_list_holds(tag, device):
  """A workgroup lists the active elements of 32 sets at a time."""
  n = 500003
  et, kt = catalog.load(f'matrix_staged_{tag}')
  ep, kp = catalog.load(f't_matrix_{tag}_plain')
  host = make_inputs(ep, n, seed=31)
  for mask in (np.arange(n) % 3 != 1, np.arange(n) // 5000 % 7 == 2, np.arange(n) == n - 1):
    flags = mask.astype(np.uint32)
    a = gpu_run(kp, ep, host, n, device, flags=flags)
    b = gpu_run(kt, et, host, n, device, flags=flags)
    for t in ep.generator._global_tensors:
      key = key_of(t)
      if key not in outputs_of(ep):
        continue
      rows = lambda x: x.reshape(n, t.get_real_volume())
      np.testing.assert_array_equal(rows(b[key])[~mask], rows(host[key])[~mask])
      assert normwise_error(b[key], a[key], t.get_real_volume()) <= TOL[et.fp_type]
