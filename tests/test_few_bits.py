"""Chains that overwrite their destination have the same results to the last bit in the form for few
elements and in the vector stream."""
import numpy as np
import pytest

from tensorforge_amd import catalog

from harness import gpu_run, make_inputs, outputs_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('name', ['t_few_gemm_41x38_auto', 't_few_volume_10_auto',
                                  't_few_volume_83x84_f32_auto', 'ader_f64_tuned',
                                  'ader_f32_tuned'])
def test_same_bits_on_both_sides_of_the_line(name, device):
  e, k = catalog.load(name)
  em = e.generator.get_emitted()
  n = em.few_limit
  host = make_inputs(e, n + 1, seed=7)
  key, = outputs_of(e)
  vol = e.tensors[key].get_real_volume()
  few, many = gpu_run(k, e, host, n, device), gpu_run(k, e, host, n + 1, device)
  np.testing.assert_array_equal(few[key][:n * vol], many[key][:n * vol])
