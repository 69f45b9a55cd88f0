"""The staged form's kernel for launches with flags: its list in LDS, where the launcher takes it, and
its first launch inside a graph capture."""
import re
import shutil

import numpy as np
import pytest

from tensorforge_amd import catalog
from tensorforge_amd.emit import staged, tile

from harness import TOL, gpu_run, key_of, make_inputs, normwise_error, outputs_of

STAGED = ['gemm_f64_tuned', 'gemm_f32_tuned', 'flux_local_mod_f64_tuned', 'flux_neigh_mod_f64_tuned',
          'deriv_f64_tuned', 'deriv_na_f64_tuned']


@pytest.mark.parametrize('name', STAGED)
def test_list_lies_behind_the_form_s_regions(name):
  e = catalog.get(name)
  e.generator.generate()
  em = e.generator.get_emitted()
  assert em.schedule['staged'] and em.masked is not None
  base, m = em.lds_bytes, em.masked.lds_bytes
  assert m == base + 2 * staged.THREADS + 4 * tile.WAVES <= tile.LDS_LIMIT and base % 4 == 0
  src = em.masked.kernel_src
  assert f'reinterpret_cast<unsigned short*>(lds) + {base // 2};' in src
  assert f'reinterpret_cast<int*>(lds) + {(base + 2 * staged.THREADS) // 4};' in src
  # nothing is read at a distance of whole elements: they come from the list
  assert 'set * 16 + lane' not in src
  assert f'flags != nullptr && numElements > {3 * tile.SET}ull * tf_cus' in e.generator.get_launcher()


def test_places_of_a_list():
  """Threads' places of a scan cover 32 sets of a workgroup, the sets those of the other kernel."""
  grid, first, sets = 7, 3, staged.THREADS // tile.SET
  assert sets == 32
  elements = [((first + (t >> 4) * grid) * tile.SET + (t & 15)) for t in range(staged.THREADS)]
  assert elements == [(first + grid * s) * 16 + i for s in range(sets) for i in range(16)]
  assert max(range(staged.THREADS)) < 1 << 16


def test_forms_without_it():
  for name in ('ader_dense_f64_tuned', 'ader_f64_tuned', 'pw_update_f64'):
    e = catalog.get(name)
    e.generator.generate()
    assert getattr(e.generator.get_emitted(), 'masked', None) is None


def _compare(e, got, ref, mask, host):
  n = len(mask)
  for t in e.generator._global_tensors:
    key = key_of(t)
    if key in outputs_of(e):
      vol = t.get_real_volume()
      rows = lambda x: x.reshape(n, vol)
      np.testing.assert_array_equal(rows(got[key])[~mask], rows(host[key])[~mask])
      assert normwise_error(got[key], ref[key], vol) <= TOL[e.fp_type]


@pytest.mark.gpu
@pytest.mark.parametrize('name', ['gemm_f64_tuned', 'deriv_f64_tuned'])
def test_both_sides_of_the_line(name, device):
  import torch
  e, k = catalog.load(name)
  ep, kp = catalog.load(name.replace('_tuned', '_plain'))
  line = 3 * tile.SET * torch.cuda.get_device_properties(device).multi_processor_count
  for n in (line, line + 1):
    mask = np.arange(n) % 7 < 3
    host = make_inputs(ep, n, seed=3)
    flags = mask.astype(np.uint32)
    _compare(e, gpu_run(k, e, host, n, device, flags=flags),
             gpu_run(kp, ep, host, n, device, flags=flags), mask, host)


@pytest.mark.gpu
def test_first_masked_launch_inside_a_capture(device, tmp_path):
  """Launches without flags do the other kernel's one-time setup, not this one's."""
  import torch
  from tensorforge_amd.device import launch
  from tensorforge_amd.graph import Graph
  from tensorforge_amd.runtime.loader import load_kernels
  e = catalog.get('gemm_f32_tuned')
  e.generator.generate()
  so = str(tmp_path / 'libfresh.so')
  shutil.copy(catalog.so_path('gemm_f32_tuned'), so)
  k = load_kernels(so, [e.generator])[0]
  n = 20001
  mask = np.arange(n) % 4 != 1
  flags = torch.from_numpy(mask.astype(np.int32)).to(device)
  host = make_inputs(e, n, seed=5)
  fresh = lambda: {key: torch.from_numpy(v.copy()).to(device) for key, v in host.items()}
  work, eager = fresh(), fresh()
  launch(k, fresh(), n)
  torch.cuda.synchronize()
  stream = torch.cuda.Stream(device)
  graph = Graph(stream)
  graph.capture(lambda: launch(k, work, n, flags=flags, stream=stream))
  for _ in range(3):
    graph.launch()
    launch(k, eager, n, flags=flags)
    torch.cuda.synchronize()
    assert torch.equal(work['C'], eager['C'])
  graph.close()
