"""Which chains the staged matrix-core form refuses (too many pieces a thread) and which it takes."""
import pytest

from tensorforge_amd import catalog
from tensorforge_amd.emit import staged

from test_matrix_forms import _form

REFUSED = ('gemm_57x60', 'gemm_84x83', 'volume_84x84')


@pytest.mark.parametrize('tag', list(catalog.MATRIX_EDGES))
def test_staged_form_by_chain(tag):
  e, program, pl = _form(f't_matrix_{tag}_auto')
  k = staged._Staged(program, e.generator._context, 'x', pl)
  assert k.prepare() == (tag not in REFUSED)
