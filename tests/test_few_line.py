"""Launches of few elements: the line is drawn by the device's compute units, not by a fixed number."""
import re

import pytest

from tensorforge_amd import catalog


@pytest.mark.parametrize('name, groups', [('ader_f64_tuned', 3), ('t_few_volume_10_auto', 2)])
def test_line_by_compute_units(name, groups):
  e = catalog.get(name)
  e.generator.generate()
  em = e.generator.get_emitted()
  src = e.generator.get_launcher()
  assert f'if (numElements <= {groups * em.few.elements_per_block}ull * tf_cus)' in src
  assert 'hipDeviceAttributeMultiprocessorCount' in src[:src.index('numElements <=')]
  assert em.few_limit == groups * 256 * em.few.elements_per_block
