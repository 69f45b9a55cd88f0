"""The matrix-core forms of the streaming schedule, on the CPU: row orders, the pieces in which a
set crosses memory, LDS regions, and which calls take the forms.

The index arithmetic of the generated kernels is restated here from the same geometry objects the
emitter prints, and checked over every chain of ``catalog.MATRIX_EDGES``: each entry the chain needs
is moved exactly once, nothing outside its window is read, written or multiplied.
"""
import pytest

from tensorforge_amd import catalog
from tensorforge_amd import workloads as W
from tensorforge_amd.common.basic_types import Addressing, FloatingPointType
from tensorforge_amd.common.context import Context
from tensorforge_amd.common.exceptions import GenerationError
from tensorforge_amd.emit import staged, stream, tile
from tensorforge_amd.emit.tuned import Schedule
from tensorforge_amd.generators.generator import Generator

F64, F32 = FloatingPointType.DOUBLE, FloatingPointType.FLOAT


def _form(name):
  e = catalog.get(name)
  e.generator.generate()
  program = e.generator.get_program()
  pl, why = stream.plan(program)
  assert pl is not None, why
  from dataclasses import replace
  pl = replace(pl, terms=[replace(t, L=t.L or pl.L, l_cols=t.l_cols or pl.l_cols)
                          for t in pl.terms])
  return e, program, pl


@pytest.mark.parametrize('nb', [2, 4])
@pytest.mark.parametrize('n', list(range(1, 70)) + [83, 84, 120, 128])
def test_row_order_covers_every_row_once(n, nb):
  r = tile.Rows(n, nb)
  rows = [r.row(s, g) for s in range(r.steps) for g in range(4)]
  assert sorted(x for x in rows if x < n) == list(range(n))
  assert len(set(rows)) == len(rows) and max(rows) < 4 * r.steps
  # the C expression agrees, blocks partition the steps, a block's lanes hold adjacent rows
  for s in range(r.steps):
    for g in range(4):
      c = r.row_expr(str(s), str(g)).replace('?', ' and ').replace('/', '//')
      if '<' in c:
        cond, rest = c[1:-1].split(' and ', 1)
        a, b = rest.split(' : ')
        c = a if eval(cond) else b
      assert eval(c) == r.row(s, g)
  assert [s for st, _, k in r.blocks() for s in range(st, st + k)] == list(range(r.steps))


def _pieces(p):
  """[(element, first storage offset, LDS offset, entries moved down)] of every thread's pieces."""
  out = []
  for t in range(staged.THREADS):
    pr = t % p.per_element
    pm, pp = pr // p.runs, pr % p.runs * p.per
    e0 = t // p.per_element
    if e0 >= p.step:
      continue
    h = max(0, pp - (p.rows - p.per)) if p.moved else 0
    for j in range(p.count):
      e = e0 + j * p.step
      if e < staged.SET:
        out.append((e, p.first + pm * p.col_stride + pp - h,
                    p.lds_base + e * p.lds_elem + pm * p.lds_run + pp, h, pm, pp))
  return out


@pytest.mark.parametrize('tag', list(catalog.MATRIX_EDGES))
def test_staged_pieces_cover_the_set(tag):
  e, program, pl = _form(f't_matrix_{tag}_auto')
  k = staged._Staged(program, e.generator._context, 'x', pl)
  if not k.prepare():
    return
  regions = []
  for p in k.xstage + [k.out] + [p for _, st in k.wstage for _, _, _, p in st]:
    got = _pieces(p)
    seen = {}
    for el, g, l, h, pm, pp in got:
      # 16 bytes inside the run, and inside the element's slot
      run = p.first + pm * p.col_stride
      assert run <= g and g + p.per <= run + p.rows
      assert 0 <= g and g + p.per <= p.arg.element_stride
      assert l % p.per == 0
      for x in range(p.per):
        key = (el, pm, pp + x)
        assert key not in seen
        seen[key] = g + x + h if pp + x < p.rows else None
    cols = p.per_element // p.runs
    for el in range(staged.SET):
      for m in range(cols):
        for r in range(p.rows):
          assert seen[(el, m, r)] == p.first + m * p.col_stride + r
    regions.append((p, min(l for _, _, l, *_ in got), max(l for _, _, l, *_ in got) + p.per))
  # LDS: shared entries, then the streamed operand or the results, then the weights
  shared = sum(s.kr.steps * k.fragment(s.dr) for s in k.stages + k.post)
  for p, lo, hi in regions:
    top = k.lds_bytes // k.size if p.lds_base >= k.wbase0 else k.wbase0
    assert shared <= lo and hi <= top
  # operand reads and result writes stay inside an element's rows
  for x, ph in zip(k.xstage, k.phases):
    assert x.lds_run == 4 * ph.kr.steps and x.lds_run * (x.per_element // x.runs) <= x.lds_elem
  assert k.out_lds_rows * k.q <= k.out.lds_elem
  assert k.lds_bytes <= tile.LDS_LIMIT


@pytest.mark.parametrize('tag', list(catalog.MATRIX_EDGES))
def test_direct_blocks_read_inside_the_range(tag):
  e, program, pl = _form(f't_matrix_{tag}_auto')
  k = tile._Tile(program, e.generator._context, 'x', pl)
  chosen = k.choose()
  assert chosen is not None
  for stages, post, phases, off, wregion in chosen[1]:
    for ph in phases:
      n = ph.kr.n
      for st, base, b in ph.kr.blocks():
        for g in range(4):
          sh = max(0, base + b * g - (n - b)) if base + 4 * b > n else 0
          assert 0 <= base + b * g - sh and base + b * g - sh + b <= n
          for j in range(b):
            want = ph.kr.row(st + j, g)
            assert want == base + b * g + j
            # the value moved down to step j, or zero past the range
            assert (want < n) == (sh + j < b)
    assert off * k.size + tile.WAVES * wregion * k.size <= tile.LDS_LIMIT
  assert sum(len(h) for h in k.halves) == pl.q


def test_forms_by_chain():
  """Dense shared operands and strided per-element ones take the matrix cores by default; an
  explicit schedule, sparse or pointer-based operands and fused statements keep their kernels."""
  def kind(w, fp=F64, **kw):
    g = Generator(w.descrs, Context('gfx950', 'hip', fp), **kw)
    g.generate()
    em = g.get_emitted()
    return em.schedule.get('matrix'), em.schedule.get('staged', False)
  assert kind(W.gemm()) == ('mfma', True) == kind(W.gemm(F32), F32)
  assert kind(W.ader_volume(sparse_k=False)) == ('mfma', False)
  assert kind(W.ader_volume(F32, sparse_k=False), F32) == ('mfma', False)
  assert kind(W.flux_local()) == kind(W.flux_neigh()) == ('mfma', True)
  assert kind(W.ader_derivative(aligned=False)) == ('mfma', True)
  assert kind(W.gemm(), schedule=Schedule()) == (None, False)
  assert kind(W.gemm(), schedule=Schedule(stream_matrix='auto')) == ('mfma', True)
  assert kind(W.ader_volume())[0] is None
  for name in ('t_gemm_ptr_auto', 't_ab_transb_auto', 't_fused_gemm_pw', 't_five_multiplies_auto'):
    e = catalog.get(name)
    e.generator.generate()
    assert e.generator.get_emitted().schedule.get('matrix') is None


def test_in_place_volume_chain_keeps_the_vector_form():
  """Both quantities' shares of a set are written by different wavefronts: a chain whose
  destination is its own streamed operand or weight stays on the form that has one."""
  from tensorforge_amd.common.aux import generate_tmp_tensor
  from tensorforge_amd.common.matrix.tensor import SubTensor, Tensor
  from tensorforge_amd.generators.descriptions import MultilinearDescr
  Q = Tensor([20, 9], Addressing.STRIDED, alias='Q')
  S = Tensor([9, 9], Addressing.STRIDED, alias='S')
  K = Tensor([20, 20], Addressing.NONE, alias='K')
  pair, ident = [[0, -1], [-1, 1]], [[0, 1], [0, 1]]
  T = generate_tmp_tensor([SubTensor(Q), SubTensor(S)], pair)
  d = [MultilinearDescr(SubTensor(T), [SubTensor(Q), SubTensor(S)], pair, ident),
       MultilinearDescr(SubTensor(Q), [SubTensor(K), SubTensor(T)], pair, ident)]
  g = Generator(d, Context('gfx950', 'hip', F64))
  g.generate()
  assert g.get_emitted().schedule.get('matrix') is None


def test_grouped_launch_takes_both_forms():
  """Members in the vector and in the matrix-core form share a workgroup size."""
  from tensorforge_amd.grouped import GroupedGenerator
  members = []
  for w in (W.ader_volume(), W.ader_volume(b=20, sparse_k=False), W.gemm()):
    g = Generator(w.descrs, Context('gfx950', 'hip', F64))
    g.generate()
    members.append(g)
  grouped = GroupedGenerator(members)
  try:
    grouped.generate()
  except GenerationError as err:
    pytest.fail(str(err))
  assert grouped.block == (512, 1, 1)


@pytest.mark.parametrize('tag', list(catalog.MATRIX_EDGES))
def test_shares_of_a_ninth_quantity(tag):
  e, program, pl = _form(f't_matrix_{tag}_auto')
  k = staged._Staged(program, e.generator._context, 'x', pl)
  if not k.prepare() or not k.shared_last:
    return
  for ph in k.phases:
    # every block of the contraction belongs to one wavefront
    full = [b for w in range(staged.SHARES) for b in range(w, ph.kr.full, staged.SHARES)]
    assert sorted(full) == list(range(ph.kr.full))
  # the other shares lie behind the results and inside the workgroup's LDS, a row run per element
  assert k.share_base >= k.out.lds_base + tile.SET * k.out.lds_elem
  end = k.share_base + (staged.SHARES - 1) * tile.SET * k.share_elem
  assert k.share_elem >= k.out.lds_run and end <= k.lds_bytes // k.size
  assert k.share_elem % k.per == 0 and k.share_base % k.per == 0


@pytest.mark.parametrize('n', [1, 2])
def test_lane_group_sums_are_dealt_out(n):
  """The exchanges of ``finish`` on four lane groups, ``[register][group]``."""
  import numpy as np
  part = np.random.default_rng(n).integers(-9, 9, (4 * n, 4))

  def swap(a, b, rows):
    """Odd ``rows``-groups of a against even ones of b (halves: 2 groups, neighbours: 1)."""
    a2, b2 = a.copy(), b.copy()
    for g in range(0, 4, 2 * rows):
      a2[g + rows:g + 2 * rows], b2[g:g + rows] = b[g:g + rows], a[g + rows:g + 2 * rows]
    return a2, b2
  x = list(part)
  for rows, count in ((2, 2 * n), (1, n)):
    x = [sum(swap(x[r], x[r + count], rows)) for r in range(count)]
  for g in range(4):
    for j in range(n):
      assert x[j][g] == part[n * g + j].sum()
