"""Register stages of the vector stream (a shared operand applied to the streamed product's rows)."""
import re

from tensorforge_amd import catalog
from tensorforge_amd.emit import stream


def test_every_row_of_the_streamed_product_reaches_the_stage():
  e = catalog.get('opt_t_matrix_chain_20x70x20_vector')
  e.generator.generate()
  pl, _ = stream.plan(e.generator.get_program())
  assert pl.post and pl.rows == (0, 70)
  assert e.generator.get_emitted().schedule.get('row_passes', 1) == 1
  # the accumulator the stage reads has a register per row
  src = e.generator.get_kernel()
  assert 'double acc[70];' in src
  assert max(int(i) for i in re.findall(r'\bacc\[(\d+)\]', src.replace('acc[70]', ''))) == 69
