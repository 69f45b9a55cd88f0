"""Which form a chain with dense shared operands gets by its sizes: chains too small for the
matrix-core forms stay in the vector stream, and a form named by the schedule is taken at any size."""
import pytest

from tensorforge_amd import catalog
from tensorforge_amd import workloads as W
from tensorforge_amd.common.basic_types import FloatingPointType
from tensorforge_amd.common.context import Context
from tensorforge_amd.generators.generator import Generator

from test_staged_refused import REFUSED

F64, F32 = FloatingPointType.DOUBLE, FloatingPointType.FLOAT


def _form(descrs, fp, **kw):
  g = Generator(descrs, Context('gfx950', 'hip', fp), **kw)
  g.generate()
  s = g.get_emitted().schedule
  return 'staged' if s.get('staged') else 'direct' if s.get('matrix') else 'vector'


@pytest.mark.parametrize('fp, m, k, q, form', [
  (F64, 2, 2, 9, 'vector'), (F32, 9, 4, 9, 'vector'), (F32, 8, 8, 1, 'vector'),
  (F64, 12, 12, 3, 'vector'), (F64, 14, 14, 3, 'staged'),       # columns of about a line
  (F32, 14, 14, 12, 'vector'), (F32, 18, 18, 6, 'staged'),
  (F64, 8, 8, 4, 'vector'), (F64, 8, 8, 9, 'staged'),
  (F64, 16, 16, 1, 'direct'), (F32, 16, 16, 1, 'vector'), (F32, 32, 32, 1, 'direct'),
  (F64, 56, 56, 9, 'staged'), (F32, 56, 56, 9, 'staged'), (F64, 48, 48, 16, 'direct')])
def test_gemm(fp, m, k, q, form):
  e = catalog._matrix_entry('gemm', m=m, k=k, q=q, fp=fp, beta=1.0)
  assert _form(e.descrs, fp) == form


@pytest.mark.parametrize('fp, b, form', [
  (F64, 4, 'direct'), (F64, 10, 'direct'), (F64, 28, 'direct'), (F64, 56, 'direct'),
  (F32, 4, 'vector'), (F32, 10, 'vector'), (F32, 20, 'direct'), (F32, 56, 'direct')])
def test_volume(fp, b, form):
  w = W.ader_volume(fp, b=b, sparse_k=False)
  assert _form(w.descrs, fp) == form


@pytest.mark.parametrize('fp, b, q, dense, form', [
  (F64, 4, 9, False, 'vector'), (F64, 4, 16, False, 'direct'), (F64, 6, 9, False, 'direct'),
  (F32, 8, 9, False, 'vector'), (F32, 8, 16, False, 'direct'), (F32, 10, 12, False, 'vector'),
  (F32, 10, 13, False, 'direct'), (F32, 4, 9, True, 'direct'), (F32, 10, 9, True, 'vector'),
  (F32, 16, 9, False, 'direct'), (F64, 10, 16, False, 'direct'), (F64, 40, 9, False, 'direct'),
  (F64, 35, 9, True, 'staged')])
def test_volume_by_weights(fp, b, q, dense, form):
  """Three terms whose columns have the same number of weights."""
  from tensorforge_amd.common.aux import generate_tmp_tensor
  from tensorforge_amd.common.basic_types import Addressing
  from tensorforge_amd.common.matrix.spp import ListSPP
  from tensorforge_amd.common.matrix.tensor import SubTensor, Tensor
  from tensorforge_amd.generators.descriptions import MultilinearDescr
  pair, ident = [[0, -1], [-1, 1]], [[0, 1], [0, 1]]
  Q, D = (Tensor([b, q], Addressing.STRIDED, alias=x) for x in 'QD')
  star = None if dense else ListSPP([(r, c) for c in range(q) for r in range(q)
                                     if (r + 2 * c) % 3 == 0], (q, q))
  descrs = []
  for i in range(3):
    S = Tensor([q, q], Addressing.STRIDED, spp=star, alias=f'S{i}')
    K = Tensor([b, b], Addressing.NONE, alias=f'K{i}')
    T = generate_tmp_tensor([SubTensor(Q), SubTensor(S)], pair)
    descrs += [MultilinearDescr(SubTensor(T), [SubTensor(Q), SubTensor(S)], pair, ident),
               MultilinearDescr(SubTensor(D), [SubTensor(K), SubTensor(T)], pair, ident, add=i > 0)]
  assert _form(descrs, fp) == form


@pytest.mark.parametrize('fp, m, mid, q, dense, form', [
  (F64, 56, 21, 9, True, 'staged'), (F32, 10, 6, 3, False, 'vector'),
  (F32, 10, 6, 9, True, 'staged'), (F64, 56, 21, 13, False, 'vector'),
  (F64, 10, 6, 3, False, 'direct'), (F64, 10, 6, 9, True, 'direct')])
def test_flux(fp, m, mid, q, dense, form):
  e = catalog._matrix_entry('chain', m=m, mid=mid, k=m, q=q, fp=fp, beta=1.0, dense_star=dense)
  assert _form(e.descrs, fp) == form


@pytest.mark.parametrize('tag', list(catalog.MATRIX_EDGES))
@pytest.mark.parametrize('form', ['staged', 'direct'])
def test_form_by_name(tag, form):
  e = catalog.get(f'matrix_{form}_{tag}')
  want = 'vector' if form == 'staged' and tag in REFUSED else form
  assert _form(e.descrs, e.fp_type, emitter='tuned', schedule=e.schedule) == want
