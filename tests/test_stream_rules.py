"""Where the vector stream's wavefronts take their groups as they get to them and where the next
group's weights are loaded early: by work per entry moved, type and weights held."""
import pytest

from tensorforge_amd import catalog
from tensorforge_amd import workloads as W
from tensorforge_amd.common.basic_types import FloatingPointType
from tensorforge_amd.common.context import Context
from tensorforge_amd.emit import stream
from tensorforge_amd.generators.generator import Generator

F64, F32 = FloatingPointType.DOUBLE, FloatingPointType.FLOAT


def _rules(g):
  g.generate()
  src, lds = g.get_emitted().kernel_src, g.get_emitted().lds_bytes
  assert lds <= stream.LDS_LIMIT
  return 'fetch_add(claim' in src, 'const size_t ew =' in src


@pytest.mark.parametrize('fp, b, claims, early', [
  (F64, 10, False, False), (F64, 35, False, False), (F64, 56, True, True), (F64, 84, True, True),
  (F32, 10, True, False), (F32, 35, True, False), (F32, 56, True, True)])
def test_volume(fp, b, claims, early):
  g = Generator(W.ader_volume(fp, b=b).descrs, Context('gfx950', 'hip', fp))
  assert _rules(g) == (claims, early)


@pytest.mark.parametrize('fp, m, claims, early', [
  (F64, 57, False, False), (F32, 20, True, False)])
def test_one_term(fp, m, claims, early):
  for dense in (False, True):
    e = catalog._matrix_entry('volume', m=m, k=m, q=9, fp=fp, dense_star=dense, sparse=True)
    assert _rules(Generator(e.descrs, Context('gfx950', 'hip', fp))) == (claims, early)


def test_gemm_with_statements():
  e = catalog.get('t_fused_gemm_pw')
  assert _rules(e.generator) == (False, False)


def test_both_ways_in_one_grouped_launch():
  """Members whose wavefronts take their groups and members with fixed shares."""
  from tensorforge_amd.grouped import GroupedGenerator
  members = [Generator(W.ader_volume(F64, b=b).descrs, Context('gfx950', 'hip', F64))
             for b in (20, 56, 10)]
  for m in members:
    m.generate()
  g = GroupedGenerator(members)
  g.generate()
  assert g.get_kernel().count('fetch_add(claim') == 1
