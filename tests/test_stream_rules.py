"""Where the vector stream's wavefronts take their groups as they get to them: by work per entry
moved and type."""
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
  return 'fetch_add(claim' in src


@pytest.mark.parametrize('fp, b, claims', [
  (F64, 10, False), (F64, 35, False), (F64, 56, True), (F64, 84, True),
  (F32, 10, True), (F32, 35, True), (F32, 56, True)])
def test_volume(fp, b, claims):
  g = Generator(W.ader_volume(fp, b=b).descrs, Context('gfx950', 'hip', fp))
  assert _rules(g) == claims


@pytest.mark.parametrize('fp, m, claims', [
  (F64, 57, False), (F32, 20, True)])
def test_one_term(fp, m, claims):
  for dense in (False, True):
    e = catalog._matrix_entry('volume', m=m, k=m, q=9, fp=fp, dense_star=dense, sparse=True)
    assert _rules(Generator(e.descrs, Context('gfx950', 'hip', fp))) == claims


def test_gemm_with_statements():
  e = catalog.get('t_fused_gemm_pw')
  assert not _rules(e.generator)


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
