"""Matrix-core form of the streaming schedule: 16 elements side by side, one MFMA column tile per
quantity, for chains with dense shared operands (FP64 and FP32, the chain's own type throughout).

Applies to the chains the streaming plan recognises (:func:`stream.plan`)::

    D_e = [beta D_e] + sum_t U_t · (L_t,e · W_t,e)         volume chain, time-derivative step
    D_e = [beta D_e] + sum_t U_t · B_t,e                   batched GEMM
    D_e = [beta D_e] + U_n · (... (U_1 · (L_e · W_e)))     flux integrals

Mapping. A wavefront owns 16 elements and half of the output columns. Column ``n`` of every MFMA
operand is an element, so each quantity has tiles of its own and lane ``l`` only ever holds entries
of element ``l % 16``:

* B operand (4 contraction rows x 16 elements): lane group ``g = l / 16`` holds one row. The order
  of the contraction rows is free, so group ``g`` takes rows that lie next to each other in memory
  (``base + n g + j`` for step ``j`` of a block of ``n`` steps): one 16-byte load per quantity feeds
  ``n`` steps, and 4 groups read whole 64-byte runs.
* ``L_e · W_e`` mixes the quantities of one element at one row, i.e. values of one lane: it is
  formed in registers with no cross-lane traffic, one FMA per stored entry of ``W``.
* D operand: register ``j`` of group ``g`` holds row ``4 j + g`` (FP64) or ``4 g + j`` (FP32) of
  the tile. The rows of the A operand are permuted so that this is row ``base + n g + j`` of the
  destination: stores are 16 bytes per lane, and a result register is the B operand of the next
  product of a flux chain as it stands.

The shared operands are staged once per workgroup into LDS in A-operand order (one fragment read
feeds the MFMAs of all of the wavefront's quantities), the weights of a wavefront's 16 elements once
per element set. Eight wavefronts per workgroup (two per SIMD) form four element sets; the two
wavefronts of a set split its quantities.

What bounds it: FP64 matrix instructions and FP64 FMAs share one unit (measured apart and together:
1.09 + 1.31 ms, 2.46 ms), 70-75 TF for either; the vector form's DPP-broadcast FMA reaches 49-58 TF
at its two wavefronts per SIMD and pays for the address of every lane's own cache line. FP32 matrix
instructions run at 125-150 TF beside the vector unit. Measured on MI355X, vector form before / this
form: order-6 volume chain with dense K_d, 65,536 elements FP64 335 / 206 us (57 TF), 100,003
elements FP32 409 / 177 us (100 TF); order 7, 30,000 elements FP64 432 / 235 us. Matrix instructions
are issued 62 % of the cycles there, the FP64 FMAs of the temporaries take another 5 %; fragments
read further ahead, the next term's temporaries formed among the matrix instructions, or rows
shared through LDS (a barrier per block) did not change or lost time.
"""
from dataclasses import dataclass, replace
from typing import List, Optional

from ..common.basic_types import Addressing, FloatingPointType
from . import ir
from .launcher import Emitted, Writer, fill_shared, kernel_params, persistent_grid
from .stream import in_place
from .traffic import element_traffic

WAVE = 64
WAVES = 8
SET = 16                     # elements per wavefront: the columns of an MFMA tile
LDS_LIMIT = 160 * 1024
# accumulator registers (32-bit) per lane: 140 of the 256 a lane has at two wavefronts per SIMD;
# the rest holds two blocks of streamed rows (72 for 9 quantities), temporaries and addresses
ACC_LIMIT = 144


def _ceil(a, b):
  return (a + b - 1) // b


@dataclass
class Rows:
  """Row order of ``n`` rows in steps of four: blocks of ``nb`` steps, group g's rows adjacent."""
  n: int
  nb: int

  @property
  def full(self):
    return self.n // (4 * self.nb)

  @property
  def tail(self):
    """Steps of the last, partial block."""
    return _ceil(self.n - self.full * 4 * self.nb, 4)

  @property
  def steps(self):
    return self.full * self.nb + self.tail

  def blocks(self):
    """[(first step, base row, steps)]"""
    out = [(b * self.nb, b * 4 * self.nb, self.nb) for b in range(self.full)]
    if self.tail:
      out.append((self.full * self.nb, self.full * 4 * self.nb, self.tail))
    return out

  def row(self, step, g):
    b = step // self.nb
    n = self.nb if b < self.full else self.tail
    return b * 4 * self.nb + n * g + step % self.nb

  def exact(self, step):
    """Every lane group's row of this step lies inside the range."""
    return self.row(step, 3) < self.n

  def row_expr(self, step, g):
    """C expression of :meth:`row` for run-time ``step`` and ``g``."""
    if not self.full:
      return f'({self.tail} * ({g}) + ({step}))'
    body = f'(({step}) / {self.nb} * {4 * self.nb} + {self.nb} * ({g}) + ({step}) % {self.nb})'
    if not self.tail:
      return body
    f = self.full * self.nb
    return (f'(({step}) < {f} ? {body} : {self.full * 4 * self.nb} + {self.tail} * ({g}) + '
            f'({step}) - {f})')

  def row_sum(self, step, g):
    """:meth:`row_expr` with one choice between constants, for code that must not branch."""
    n = self.nb if not self.tail else \
        f'({step} < {self.full * self.nb} ? {self.nb} : {self.tail})'
    return f'{step} / {self.nb} * {4 * self.nb} + {n} * {g} + {step} % {self.nb}'


@dataclass
class Stage:
  """One shared operand and where its fragments sit in LDS."""
  U: ir.Factor
  u_dims: tuple
  rows: tuple                 # destination rows
  k0: int                     # contraction index of relative row 0
  krange: tuple               # the operand's contraction range
  kr: Rows                    # contraction steps
  dr: Rows                    # destination row steps
  base: int = 0               # LDS offset (entries)


@dataclass
class Phase:
  """Terms that contract rows of one streamed operand (``X``), block by block."""
  X: ir.Factor
  row0: int                   # storage row of contraction index 0
  cols: List[int]             # columns of X that are loaded
  terms: List[int]
  kr: Rows


def set_unsupported_reason(program, pl):
  """Why whole elements of a chain cannot be staged in LDS, or None."""
  if program.epilogue is not None:
    return 'pointwise statements fused into the chain'
  kinds = {t.kind for t in pl.terms}
  if len(kinds) != 1:
    return 'temporaries beside a per-element right operand'
  if any(a.per_element and a.addressing != Addressing.STRIDED for a in program.args):
    return 'a per-element operand is not strided'
  if any(a.kind != ir.SRC_GLOBAL or a.dtype != program.fp_type for a in program.args):
    return 'an operand by value or of another type'
  if pl.dest_product.dest_strides[0] != 1:
    return 'destination rows are not contiguous'
  final = pl.post[-1].product if pl.post else pl.dest_product
  if final.dest_strides[0] != 1:
    return 'destination rows are not contiguous'
  if kinds == {'fused'} and pl.cols[0] != 0:
    return 'temporary with offset columns'
  for t in pl.terms:
    if t.kind == 'fused':
      if t.L.arg is pl.dest:
        return 'the destination is also the streamed operand'
      if t.L.strides[0] != 1:
        return 'streamed operand layout'
      if t.W.arg is pl.dest:
        return 'the destination is also a weight'
    else:
      if t.B.strides[t.b_dims[0]] != 1:
        return 'right operand rows are not contiguous'
      if t.B.arg is pl.dest and len(pl.terms) > 1:
        return 'the destination is also an operand'
  return None


def unsupported_reason(program, pl):
  if pl.q > 16 or any(t.kind == 'fused' and t.l_cols[1] - t.l_cols[0] > 16 for t in pl.terms):
    return 'more than 16 columns'
  if any(t.U.is_sparse() for t in pl.terms) or any(s.U.is_sparse() for s in pl.post):
    return 'sparse shared operand'
  return set_unsupported_reason(program, pl)


def term_weights(t, columns):
  """[(column, [(m, position)])] of term t's stored weights in the columns."""
  prod = t.producer
  mlo, mhi = prod.k_ranges[0]
  c_lo = prod.n_ranges[1][0]
  rk, rn = t.w_dims
  out = []
  for c in columns:
    ms = []
    for m in range(mlo, mhi):
      idx = [0, 0]
      idx[rk], idx[rn] = m, c_lo + c
      pos = t.W.packed.get(tuple(idx)) if t.W.is_sparse() else t.W.offset(idx)
      if pos is not None:
        ms.append((m, pos))
    out.append((c, ms))
  return out


class _Tile:
  def __init__(self, program, context, base_name, pl):
    self.prog, self.ctx, self.pl = program, context, pl
    self.base_name = base_name
    self.kname = f'kernel_{base_name}'
    self.fp = program.fp_type
    self.f64 = self.fp == FloatingPointType.DOUBLE
    self.real = FloatingPointType.as_str(self.fp)
    self.size = self.fp.size()
    self.nb = 2 if self.f64 else 4
    self.w = Writer()
    self.q = pl.q
    self.fused = pl.terms[0].kind == 'fused'
    self.n = 0

  def split(self, parts):
    """Divide the quantities among ``parts`` wavefronts of a set, the larger shares first."""
    self.parts = parts
    self.sets = WAVES // parts
    lo, self.halves = 0, []
    for i in range(parts):
      n = self.q // parts + (1 if i < self.q % parts else 0)
      self.halves.append(list(range(lo, lo + n)))
      lo += n

  def fresh(self, p):
    self.n += 1
    return f'{p}{self.n}'

  # ------------------------------------------------------------------ geometry
  def tiles(self, dr: Rows):
    """(16-row tiles, 4-row tiles) of a destination row range. The FP64 matrix core runs a 4-row
    tile of four column blocks (v_mfma_f64_4x4x4_4b, 16 cycles) at the 16-row tile's rate (64
    cycles) with the same B and D registers. The FP32 one (v_mfma_f32_4x4x1_16b, 8 cycles against
    32) multiplies each lane group's contraction row into sums of its own: four registers, added
    over the lane groups when the contraction ends (:meth:`finish`). Three of them take more
    registers than they save (dense volume chains FP32, last rows in 16-row / 4-row tiles: 10 rows,
    3 tiles 50 / 54 us; 20 rows, 1 tile 123 / 110; 35 rows, 1 tile 330 / 311; 56 rows, 2 tiles 180 /
    178; 84 rows, 1 tile 419 / 389)."""
    big, small = dr.steps // 4, dr.steps % 4
    return (big, small) if self.f64 or small < 3 else (big + 1, 0)

  def fragment(self, dr):
    """LDS entries of one contraction step's A operand."""
    big, small = self.tiles(dr)
    return 64 * big + 16 * small

  def acc_registers(self, dr):
    big, small = self.tiles(dr)
    return (4 * big + small * (1 if self.f64 else 5)) * (self.size // 4) * len(self.halves[0])

  def weights(self, t, half):
    return term_weights(t, half)

  def weight_span(self, t, half):
    ps = [p for _, ms in self.weights(t, half) for _, p in ms]
    return (min(ps), max(ps) + 1) if ps else (0, 0)

  def plan(self, rows, split_terms):
    """Stages, phases and LDS use of one band of destination rows."""
    pl = self.pl
    stages = []
    for t in pl.terms:
      k0, k1 = t.product.k_ranges[0]
      top = pl.khi if self.fused and not split_terms else k1
      stages.append(Stage(t.U, t.u_dims, rows, pl.klo, (k0, k1), Rows(top - pl.klo, self.nb),
                          Rows(rows[1] - rows[0], self.nb)))
    prev = stages[-1]
    post = []
    for s in pl.post:
      post.append(Stage(s.U, s.u_dims, s.rows, s.prev_lo, tuple(s.product.k_ranges[0]), prev.dr,
                        Rows(s.rows[1] - s.rows[0], self.nb)))
      prev = post[-1]
    off = 0
    for s in stages + post:
      s.base = off
      off += s.kr.steps * self.fragment(s.dr)
    phases = []
    if self.fused and not split_terms:
      t = pl.terms[0]
      phases.append(Phase(t.L, pl.klo + t.l_shift - t.L.origin[0], list(range(*t.l_cols)),
                          list(range(len(pl.terms))), stages[0].kr))
    else:
      for ti, t in enumerate(pl.terms):
        if self.fused:
          phases.append(Phase(t.L, pl.klo + t.l_shift - t.L.origin[0], list(range(*t.l_cols)),
                              [ti], stages[ti].kr))
        else:
          phases.append(Phase(t.B, pl.klo - t.B.origin[t.b_dims[0]], None, [ti], stages[ti].kr))
    wregion = 0
    if self.fused:
      for ph in phases:
        for half in self.halves:
          spans = [self.weight_span(pl.terms[ti], half) for ti in ph.terms]
          wregion = max(wregion, sum(b - a for a, b in spans) * SET)
    return stages, post, phases, off, wregion

  # ------------------------------------------------------------------ emission
  def choose(self):
    """Row bands, wavefronts per set and term order that fit the registers and LDS, or None. Two
    wavefronts per set where the weights of every term fit in LDS beside the shared operands; four
    per set (half as many sets, so half the weights) where they do not (three dense 9x9 weights);
    as the last resort the terms one after the other, reading the streamed rows once per term."""
    pl = self.pl
    n = pl.rows[1] - pl.rows[0]
    # (a second band of a product in place would read what the first one wrote)
    max_bands = 1 if pl.post or in_place(pl) else 4
    for bands in range(1, max_bands + 1):
      step = _ceil(_ceil(n, bands), 4) * 4
      windows = [(r, min(r + step, pl.rows[1])) for r in range(pl.rows[0], pl.rows[1], step)]
      in_turn = pl.stacked or not self.fused
      for parts, turn in ((2, in_turn), (4, in_turn), (2, True)):
        if self.q < parts and parts > 1:
          parts = 1
        self.split(parts)
        plans = [self.plan(w, turn) for w in windows]
        lds = max((off + WAVES * wr) * self.size for _, _, _, off, wr in plans)
        acc = max(self.acc_registers(s.dr) for st, post, _, _, _ in plans
                  for s in st + post[:-1])
        if lds <= LDS_LIMIT and acc <= ACC_LIMIT:
          return windows, plans, lds, turn
    return None

  def matrix_bound(self):
    memory, matrix = set_times(self.prog, self.pl)
    return matrix > memory

  def depth(self, stages, phases):
    """Blocks of streamed rows held in registers: as many as fit beside the accumulators of the
    streamed product, at most three. More of them keep more bytes in flight; a lane has 256
    registers, about 60 of them go to temporaries, weights, fragments and addresses."""
    acc = self.acc_registers(stages[0].dr)
    if self.pl.post:
      # beside them the previous product's and a tile of the last one's
      acc += 4 * (self.size // 4) * len(self.halves[0])
    cols = max(len(self.ph_cols(ph, self.halves[0])) for ph in phases)
    rows = cols * self.nb * self.size // 4
    blocks = sum(len(ph.kr.blocks()) for ph in phases)
    return max(1, min(3, (256 - 60 - acc) // rows, blocks))

  def emit(self) -> Optional[Emitted]:
    chosen = self.choose()
    if chosen is None:
      return None
    windows, plans, lds_bytes, split = chosen
    w = self.w
    pl = self.pl
    real = self.real
    threads = WAVE * WAVES
    self.typedefs()
    params = ', '.join(kernel_params(self.prog, self.ctx))
    w(f'extern "C" __global__ void __launch_bounds__({threads}, 2) {self.kname}({params})')
    w('{')
    w._depth += 1
    for i, (window, plan) in enumerate(zip(windows, plans)):
      w(f'// matrix-core streaming: rows [{window[0]}, {window[1]}), {self.sets} sets of {SET} '
        f'elements per workgroup, {plan[3]} shared entries in LDS')
      w('{')
      w._depth += 1
      self.band(window, plan)
      w._depth -= 1
      w('}')
      if i + 1 < len(windows):
        w('__syncthreads();')
    w._depth -= 1
    w('}')
    traffic = element_traffic(self.prog)
    sched = {'kind': 'stream', 'matrix': 'mfma', 'waves_per_block': WAVES, 'elements_per_wave': SET,
             'columns': self.q, 'column_parts': self.parts, 'shared_entries': self.entry_count(),
             'lds_bytes': lds_bytes, 'terms_in_turn': split, 'row_passes': len(windows)}
    return Emitted(kernel_name=self.kname, kernel_src=w.src(), block=(threads, 1, 1),
                   elements_per_block=SET, lds_bytes=lds_bytes, emitter='tuned', schedule=sched,
                   bytes_per_element=traffic.per_element, shared_bytes=traffic.shared,
                   grid_override='tf_grid',
                   extra_launch_setup=persistent_grid(self.kname, lds_bytes, threads, SET,
                                                      f'launcher_{self.base_name}'))

  def typedefs(self):
    w = self.w
    real = self.real
    tag = 'D' if self.f64 else 'F'
    w(f'#ifndef TF_TILE_{tag}')
    w(f'#define TF_TILE_{tag}')
    w(f'typedef {real} tf_t{tag} __attribute__((ext_vector_type(4)));')
    # rows of one lane in memory: aligned as single entries are (odd offsets and row counts)
    for n in (2,) if self.f64 else (2, 4):
      w(f'typedef {real} tf_v{tag}{n} __attribute__((ext_vector_type({n}), '
        f'aligned({self.size})));')
    # the same in LDS, where they are aligned
    w(f'typedef {real} tf_x{tag} __attribute__((ext_vector_type({16 // self.size})));')
    w('#endif')
    self.acc_t = f'tf_t{tag}'
    self.lds_t = f'tf_x{tag}'
    self.vec_t = {2: f'tf_v{tag}2', 4: f'tf_v{tag}4'}

  def entry_count(self):
    """Entries of the shared operands inside the products' ranges."""
    pl = self.pl
    entries = sum((t.product.k_ranges[0][1] - t.product.k_ranges[0][0]) * (pl.rows[1] - pl.rows[0])
                  for t in pl.terms)
    entries += sum((s.product.k_ranges[0][1] - s.product.k_ranges[0][0]) *
                   (s.rows[1] - s.rows[0]) for s in pl.post)
    return entries

  def stage_shared(self, s: Stage):
    """A fragments of one shared operand: entry ``e`` is step ``e / F``, then the 16-row tiles' 64
    lanes, then the 4-row tiles' 16 entries; rows and contraction indices outside the operand's
    ranges are zero."""
    w = self.w
    F = self.fragment(s.dr)
    big, small = self.tiles(s.dr)
    nrows = s.rows[1] - s.rows[0]
    nd, kd = s.u_dims
    total = s.kr.steps * F
    if total == 0:
      return
    # every value on a line of its own: a conditional expression of such terms becomes a branch,
    # and a branch between two entries keeps their loads apart
    lines = [f'const int st = e / {F};', f'const int f = e - st * {F};']
    # 16-row tiles, then 4-row tiles
    if self.f64:
      lines += ['const int j1 = f / 64 * 4 + f % 16 / 4;', 'const int g1 = f % 4;',
                f'const int j2 = {4 * big} + (f - {64 * big}) / 16;', 'const int g2 = g1;']
    else:
      # (a 4-row tile's rows follow each other: entry x of the last block's 4 n rows)
      n = max(1, small)
      lines += ['const int j1 = f / 64 * 4 + f % 4;', 'const int g1 = f % 16 / 4;',
                f'const int x = (f - {64 * big}) / 16 * 4 + f % 4;',
                f'const int j2 = {4 * big} + x % {n};', f'const int g2 = x / {n};']
    lines += ['const int kg1 = f % 64 / 16;', f'const int kg2 = (f - {64 * big}) % 16 / 4;',
              f'const int j = f < {64 * big} ? j1 : j2;', f'const int g = f < {64 * big} ? g1 : g2;',
              f'const int kg = f < {64 * big} ? kg1 : kg2;']
    lines += [f'const int row = {s.dr.row_sum("j", "g")};',
              f'const int k = {s.kr.row_sum("st", "kg")} + {s.k0};',
              f'const bool in = (j < {s.dr.steps}) & (row < {nrows}) & (k >= {s.krange[0]}) & '
              f'(k < {s.krange[1]});',
              f'const int pos = (row + {s.rows[0] - s.U.origin[nd]}) * {s.U.strides[nd]} + '
              f'(k - {s.U.origin[kd]}) * {s.U.strides[kd]};',
              f'const {self.real} u = {s.U.arg.name}[in ? pos : 0];']
    fill_shared(w, total, WAVE * WAVES,
                [(self.real, 'uv', lines, f'in ? u : ({self.real})0')],
                lambda e, v: f'ubuf[{s.base} + {e}] = {v}')

  def band(self, window, plan):
    w = self.w
    stages, post, phases, koff, wregion = plan
    real = self.real
    w(f'extern __shared__ __align__(16) {real} lds[];')
    w(f'{real}* __restrict__ ubuf = lds;')
    for s in stages + post:
      self.stage_shared(s)
    w('__syncthreads();')
    w(f'const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / {WAVE});')
    w(f'const int lane = threadIdx.x % {WAVE};')
    w('const int el = lane % 16;')
    w('const int g = lane / 16;')
    w(f'{real}* __restrict__ wbuf = lds + {koff} + wave * {wregion};')
    w(f'const {real}* __restrict__ ka = ubuf + lane;')
    w(f'const {real}* __restrict__ ks = ubuf + (lane % 4 + 4 * g);')
    w(f'const size_t nsets = (numElements + {SET - 1}) / {SET};')
    # waves w and w + 4 share a SIMD: they take unequal shares of the quantities
    w(f'const int part = (wave + wave / 4) % {self.parts};')
    w(f'const size_t set0 = (size_t)(wave / {self.parts}) * gridDim.x + blockIdx.x;')
    w(f'const size_t sstep = (size_t)gridDim.x * {self.sets};')
    for h, half in enumerate(self.halves):
      with w.block(f'{"else " if h else ""}if (part == {h})'):
        self.sets_loop(half, window, plan)

  # ------------------------------------------------------------------ streamed rows
  def ph_cols(self, ph, half):
    """Columns of the phase's streamed operand this half reads."""
    if ph.cols is not None:
      return ph.cols
    t = self.pl.terms[ph.terms[0]]
    return [self.pl.cols[0] + c for c in half]

  def col_off(self, ph, m):
    if ph.cols is not None:
      return (m - ph.X.origin[1]) * ph.X.strides[1]
    nd = self.pl.terms[ph.terms[0]].b_dims[1]
    return (m - ph.X.origin[nd]) * ph.X.strides[nd]

  def pointer(self, ph, eexpr):
    a = ph.X.arg
    return (f'{a.name} + {eexpr} * {a.element_stride}ull + {a.name}_extraOffset + '
            f'{ph.row0} + {self.nb} * g')

  def load_block(self, ph, half, block, elem, name, off='0'):
    """``{name}{i}`` <- the block's rows of every column of element ``elem``."""
    w = self.w
    st, base, n = block
    ptr = 'lp'
    w(f'const {self.real}* __restrict__ lp = {self.pointer(ph, elem)};')
    whole = base + 4 * n <= ph.kr.n
    # partial block: group g's n rows start at n g. Where they would pass the end of the range the
    # last n rows are read, moved down by the distance and filled up with zeros (nothing outside the
    # range is read, and nothing in the padding reaches a product)
    if not whole:
      w(f'const int sh = {base} + {n} * g - {ph.kr.n - n} > 0 ? {base} + {n} * g - '
        f'{ph.kr.n - n} : 0;')
    shift = ('' if n == self.nb else f' + ({n - self.nb}) * g') + ('' if whole else ' - sh')
    for i, m in enumerate(self.ph_cols(ph, half)):
      at = f'{ptr} + {off} + {self.col_off(ph, m) + base}{shift}'
      if whole and n == self.nb:
        w(f'{name}{i} = *reinterpret_cast<const {self.vec_t[n]}*>({at});')
        continue
      v = [self.fresh('xr') for _ in range(n)]
      if n in self.vec_t:
        x = self.fresh('xr')
        w(f'const {self.vec_t[n]} {x} = *reinterpret_cast<const {self.vec_t[n]}*>({at});')
        v = [f'{x}[{j}]' for j in range(n)]
      else:
        for j in range(n):
          w(f'const {self.real} {v[j]} = ({at})[{j}];')
      for j in range(n):
        e = v[j]
        if not whole:
          e = f'({self.real})0'
          for d in range(n - 1 - j, -1, -1):
            e = f'(sh == {d} ? {v[j + d]} : {e})'
        w(f'{name}{i}[{j}] = {e};')

  # ------------------------------------------------------------------ one part's loop over sets
  def sets_loop(self, half, window, plan):
    w = self.w
    pl = self.pl
    stages, post, phases, koff, wregion = plan
    D = self.D = self.depth(stages, phases)
    # all blocks of a set in order; block i's rows sit in register set (rot + i) % D
    self.seq = [(pi, b) for pi, ph in enumerate(phases) for b in range(len(ph.kr.blocks()))]
    self.rot = 0
    cols = max(len(self.ph_cols(ph, half)) for ph in phases)
    for d in range(D):
      names = ', '.join(f'q{d}_{i}' for i in range(cols))
      w(f'{self.vec_t[self.nb]} {names};')
    w('size_t set = set0;')
    w('size_t eg = set * 16 + el;')
    w('size_t eS = eg < numElements ? eg : numElements - 1;')
    for d in range(D):
      pi, b = self.seq[d]
      with w.block(''):
        self.load_block(phases[pi], half, phases[pi].kr.blocks()[b], 'eS', f'q{d}_')
    # every wavefront of the workgroup runs the same number of rounds
    w('const size_t rounds = (nsets + sstep - 1) / sstep;')
    with w.block('for (size_t r = 0; r < rounds; ++r, set += sstep)'):
      if self.fused and self.parts > 1 and not self.matrix_bound():
        # the wavefronts of a set read the same rows: kept together, one of them finds the other's
        # lines in the caches (left alone they drift apart by whole sets)
        w('__builtin_amdgcn_s_barrier();')
      w('if (set >= nsets) continue;')
      w('eg = set * 16 + el;')
      w('eS = eg < numElements ? eg : numElements - 1;')
      w('const size_t egn = (set + sstep) * 16 + el;')
      w('const size_t eSn = egn < numElements ? egn : numElements - 1;')
      w('const bool act = eg < numElements && (flags == nullptr || flags[eg] != 0u);')
      if not post:
        self.declare_acc('acc', stages[0].dr, half)
        if pl.init == 'load':
          self.dest_rows('acc', stages[0].dr, half, window, 'load', pl.beta)
      else:
        # the last product of a flux chain runs tile by tile: its accumulators need not all be
        # live beside the previous product's, and the old destination is loaded a tile ahead
        last = post[-1]
        chunks = self.row_chunks(last.dr)
        self.open_chunk('out', last, chunks[0], half)
        self.declare_acc('acc', stages[0].dr, half)
      for pi in range(len(phases)):
        self.phase(pi, half, plan, 'acc')
      self.finish('acc', stages[-1].dr, half)
      prev, prev_stage = 'acc', stages[-1]
      for si, s in enumerate(post[:-1]):
        name = f'acp{si}'
        self.declare_acc(name, s.dr, half)
        ops = self.post_operands(s, prev, prev_stage, half)
        for j in range(s.kr.steps):
          self.mfma(name, s, f'{s.base + j * self.fragment(s.dr)}', ops[j])
        self.finish(name, s.dr, half)
        prev, prev_stage = name, s
      if not post:
        with w.block('if (act)'):
          self.dest_rows('acc', stages[0].dr, half, window, 'store')
      else:
        ops = self.post_operands(last, prev, prev_stage, half)
        for ci, chunk in enumerate(chunks):
          if ci + 1 < len(chunks):
            self.open_chunk('out', last, chunks[ci + 1], half)
          w('__builtin_amdgcn_sched_barrier(0);')
          for j in range(last.kr.steps):
            self.mfma('out', last, f'{last.base + j * self.fragment(last.dr)}', ops[j], chunk)
          self.finish('out', last.dr, half, chunk)
          with w.block('if (act)'):
            self.dest_rows('out', last.dr, half, last.rows, 'store', 1.0, chunk)
          w('__builtin_amdgcn_sched_barrier(0);')
      # the pending blocks move to the register sets the loop starts with
      if self.rot % D:
        with w.block(''):
          for d in range(D):
            for i in range(cols):
              w(f'const {self.vec_t[self.nb]} y{d}_{i} = q{(self.rot + d) % D}_{i};')
          for d in range(D):
            for i in range(cols):
              w(f'q{d}_{i} = y{d}_{i};')

  # ------------------------------------------------------------------ accumulators
  def acc_ref(self, name, c, j):
    """Result register j of quantity c."""
    big = self.acc_big[name]
    return f'{name}_{c}_{j // 4}[{j % 4}]' if j < 4 * big else f'{name}_{c}s{j - 4 * big}'

  def row_chunks(self, dr):
    """Row tiles one at a time: [(16-row tiles, 4-row tiles)]; the 4-row tiles together."""
    big, small = self.tiles(dr)
    return [((t,), ()) for t in range(big)] + ([((), tuple(range(small)))] if small else [])

  def all_tiles(self, dr):
    big, small = self.tiles(dr)
    return tuple(range(big)), tuple(range(small))

  def declare_acc(self, name, dr, half, chunk=None):
    w = self.w
    self.acc_big = getattr(self, 'acc_big', {})
    self.acc_big[name] = self.tiles(dr)[0]
    big, small = chunk or self.all_tiles(dr)
    zero = f'({self.real})0'
    for c in half:
      for t in big:
        w(f'{self.acc_t} {name}_{c}_{t} = {{{zero}, {zero}, {zero}, {zero}}};')
      for s in small:
        w(f'{self.real} {name}_{c}s{s} = {zero};')
        if not self.f64:
          w(f'{self.acc_t} {name}_{c}q{s} = {{{zero}, {zero}, {zero}, {zero}}};')

  def open_chunk(self, name, s, chunk, half):
    self.declare_acc(name, s.dr, half, chunk)
    if self.pl.final_init == 'load':
      self.dest_rows(name, s.dr, half, s.rows, 'load', self.pl.final_beta, chunk)

  def dest_pointer(self):
    d = self.pl.dest
    final = self.pl.post[-1].product if self.pl.post else self.pl.dest_product
    return d, final.dest_origin, final.dest_strides

  def dest_rows(self, name, dr, half, rows, what, beta=1.0, chunk=None):
    """Load the old destination into the accumulators (of the chunk's tiles), or store them."""
    w = self.w
    d, (o0, o1), (s0, s1) = self.dest_pointer()
    const = 'const ' if what == 'load' else ''
    w('{')
    w._depth += 1
    w(f'{const}{self.real}* __restrict__ dp = {d.name} + eS * {d.element_stride}ull + '
      f'{d.name}_extraOffset + {rows[0] - o0};')
    scale = '' if beta == 1.0 else f'{self.fp.literal(beta)} * '
    big, small = chunk or self.all_tiles(dr)
    held = [4 * t + x for t in big for x in range(4)]
    held += [4 * self.tiles(dr)[0] + x for x in small]
    for st, base, n in dr.blocks():
      if st not in held:
        continue
      whole = base + 4 * n <= dr.n
      for c in half:
        co = (c + self.pl.cols[0] - o1) * s1
        refs = [self.acc_ref(name, c, st + j) for j in range(n)]
        if n == self.nb and whole:
          vt = self.vec_t[n]
          p = f'dp + {co + base} + {n} * g'
          if what == 'load':
            v = self.fresh('xo')
            w(f'const {vt} {v} = *reinterpret_cast<const {vt}*>({p});')
            for j, r in enumerate(refs):
              w(f'{r} = {scale}{v}[{j}];')
          else:
            w(f'*reinterpret_cast<{vt}*>({p}) = {vt}{{{", ".join(refs)}}};')
        elif what == 'load':
          # rows past the range are never stored: the last row stands in for them
          for j, r in enumerate(refs):
            row = f'{base + j} + {n} * g'
            if not dr.exact(st + j):
              row = f'({row} < {dr.n} ? {row} : {dr.n - 1})'
            w(f'{r} = {scale}dp[{co} + {row}];')
      if what == 'store' and not (n == self.nb and whole):
        for j in range(n):
          head = '' if dr.exact(st + j) else f'if ({base + j} + {n} * g < {dr.n})'
          with w.block(head):
            for c in half:
              co = (c + self.pl.cols[0] - o1) * s1
              w(f'dp[{co + base + j} + {n} * g] = {self.acc_ref(name, c, st + j)};')
    w._depth -= 1
    w('}')

  # ------------------------------------------------------------------ products
  def mfma(self, name, s: Stage, step_off, operands, chunk=None):
    """One contraction step: ``operands`` {quantity: B register expression}; ``step_off`` the LDS
    offset (C expression) of the step's fragment."""
    w = self.w
    big, small = chunk or self.all_tiles(s.dr)
    for t in big:
      a = self.fresh('xa')
      w(f'const {self.real} {a} = ka[{step_off} + {64 * t}];')
      for c, b in operands.items():
        fn = '__builtin_amdgcn_mfma_f64_16x16x4f64' if self.f64 else \
            '__builtin_amdgcn_mfma_f32_16x16x4f32'
        w(f'{name}_{c}_{t} = {fn}({a}, {b}, {name}_{c}_{t}, 0, 0, 0);')
    for i in small:
      a = self.fresh('xa')
      w(f'const {self.real} {a} = ks[{step_off} + {64 * self.tiles(s.dr)[0] + 16 * i}];')
      for c, b in operands.items():
        self.mfma_small(f'{name}_{c}', i, a, b)

  def mfma_small(self, name, i, a, b):
    if self.f64:
      self.w(f'{name}s{i} = __builtin_amdgcn_mfma_f64_4x4x4f64({a}, {b}, {name}s{i}, 0, 0, 0);')
    else:
      self.w(f'{name}q{i} = __builtin_amdgcn_mfma_f32_4x4x1f32({a}, {b}, {name}q{i}, 0, 0, 0);')

  def finish(self, name, dr, half, chunk=None):
    """The lane groups' sums of the FP32 4-row tiles, added up and dealt out: entry x of the 4 n rows
    of the last block ends in group x / n. Two exchanges, of half the wavefront and of neighbouring
    groups, each halving the number of registers."""
    w = self.w
    small = (chunk or self.all_tiles(dr))[1]
    n = len(small)
    if self.f64 or not n:
      return
    for c in half:
      x = [f'{name}_{c}q{t}[{i}]' for t in small for i in range(4)]
      for swap, count in (('32', 2 * n), ('16', n)):
        y = []
        for r in range(count):
          p, v = self.fresh('xe'), self.fresh('xf')
          w(f'const auto {p} = __builtin_amdgcn_permlane{swap}_swap(__float_as_uint({x[r]}), '
            f'__float_as_uint({x[r + count]}), false, false);')
          w(f'const float {v} = __uint_as_float({p}[0]) + __uint_as_float({p}[1]);')
          y.append(v)
        x = y
      for j in range(n):
        w(f'{name}_{c}s{j} += {x[j]};')

  def stage_weights(self, ph, half):
    """The wavefront's weights of the phase's terms into its LDS region, [position][element]."""
    w = self.w
    off = 0
    self.wbase = {}
    loads = []
    for ti in ph.terms:
      t = self.pl.terms[ti]
      lo, hi = self.weight_span(t, half)
      self.wbase[ti] = off - lo
      loads.append((t, lo, hi - lo, off))
      off += hi - lo
    self.fence()
    # group g of an element's four lanes reads neighbouring positions: 16-byte loads again
    for t, lo, cnt, o in loads:
      if cnt == 0:
        continue
      a = t.W.arg
      p = self.fresh('xp')
      w(f'const {self.real}* __restrict__ {p} = {a.name} + eS * {a.element_stride}ull + '
        f'{a.name}_extraOffset + {lo} + {self.nb} * g;')
      full = cnt // (4 * self.nb)
      vals = []
      for b in range(full):
        v = self.fresh('xw')
        w(f'const {self.vec_t[self.nb]} {v} = *reinterpret_cast<const {self.vec_t[self.nb]}*>('
          f'{p} + {b * 4 * self.nb});')
        vals += [(f'{v}[{j}]', f'({o + b * 4 * self.nb + j} + {self.nb} * g)')
                 for j in range(self.nb)]
      base = full * 4 * self.nb
      for j in range(_ceil(cnt - base, 4)):
        # the last positions one by one, past the end the last one again
        v = self.fresh('xw')
        r = f'{base + 4 * j} + g' if base + 4 * j + 3 < cnt else \
            f'({base + 4 * j} + g < {cnt} ? {base + 4 * j} + g : {cnt - 1})'
        w(f'const int {v}r = {r};')
        w(f'const {self.real} {v} = {p}[{v}r - {self.nb} * g];')
        vals.append((v, f'({o} + {v}r)'))
      for v, at in vals:
        w(f'wbuf[{at} * {SET} + el] = {v};')
    self.fence()

  def fence(self):
    w = self.w
    w('__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");')
    w('__builtin_amdgcn_wave_barrier();')
    w('__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");')

  def phase(self, pi, half, plan, acc):
    w = self.w
    stages, post, phases, _, _ = plan
    ph = phases[pi]
    D = self.D
    blocks = ph.kr.blocks()
    first = self.seq.index((pi, 0))
    w('{')
    w._depth += 1
    w(f'// contraction of {ph.X.arg.name}, terms {ph.terms}')
    if self.fused:
      self.stage_weights(ph, half)
      w('int wl = el;')
    # full blocks whose successor D blocks on is full too run as a loop over D blocks at a time
    groups = max(0, ph.kr.full - D) // D
    if groups > 1:
      w('#pragma unroll 1')
      with w.block(f'for (int kb = 0; kb < {groups}; ++kb)'):
        w(f'const int ro = kb * {4 * self.nb * D};')
        for d in range(D):
          with w.block(''):
            nxt = (0, (d + D) * 4 * self.nb, self.nb)
            self.block(ph, half, stages, blocks[d], d, acc, groups,
                       lambda name: self.load_block(ph, half, nxt, 'eS', name, 'ro'))
      done = groups * D
    else:
      done = 0
    for bi in range(done, len(blocks)):
      t = first + bi + D
      tp, tb = self.seq[t % len(self.seq)]
      elem = 'eS' if t < len(self.seq) else 'eSn'
      with w.block(''):
        self.block(ph, half, stages, blocks[bi], bi, acc, 0,
                   lambda name: self.load_block(phases[tp], half, phases[tp].kr.blocks()[tb],
                                                elem, name))
    self.rot = (self.rot + len(blocks)) % D
    w._depth -= 1
    w('}')

  def block(self, ph, half, stages, block, bi, acc, groups, load_next):
    """The products of block ``bi`` of the phase (in a loop of ``groups`` rounds over D blocks when
    that is not 0). ``load_next(name)`` emits the loads of the block D blocks on into the same
    registers: as soon as the last term's temporary rows are formed; for a GEMM, whose rows are
    operands themselves, after the products."""
    w = self.w
    st, base, n = block
    q = f'q{(self.rot + bi) % self.D}_'
    for ti in ph.terms:
      s = stages[ti]
      F = self.fragment(s.dr)
      if self.fused:
        ops = self.temporary_rows(ph, half, ti, s, block, q, groups)
        if ti == ph.terms[-1]:
          load_next(q)
      else:
        ops = [{c: f'{q}{i}[{j}]' for i, c in enumerate(half)} for j in range(n)]
      w('__builtin_amdgcn_sched_barrier(0);')
      for j in range(n):
        off = f'{s.base + (st + j) * F}'
        if groups:
          off += f' + kb * {self.nb * F * self.D}'
        self.mfma(acc, s, off, ops[j])
      if not self.fused:
        load_next(q)
      w('__builtin_amdgcn_sched_barrier(0);')

  def temporary_rows(self, ph, half, ti, s, block, q, groups):
    """Term t's temporary in the block's rows: [{quantity: register}] per step. The weights are
    read through an offset the compiler takes as new each time: they must not all sit in registers
    across the blocks."""
    w = self.w
    t = self.pl.terms[ti]
    st, base, n = block
    ops = [dict() for _ in range(n)]
    cols = {m: i for i, m in enumerate(ph.cols)}
    w('asm volatile("" : "+v"(wl));')
    # the weights of about nine products are read ahead of the ones that use them
    chunks = [[]]
    for c, ms in self.weights(t, half):
      if not ms:
        continue
      if chunks[-1] and sum(len(x) for _, x in chunks[-1]) + len(ms) > 9:
        chunks.append([])
      chunks[-1].append((c, ms))
    names = {}

    def read(group):
      for c, ms in group:
        for m, p in ms:
          names[(c, m)] = self.fresh('xs')
          w(f'const {self.real} {names[(c, m)]} = wbuf[{(self.wbase[ti] + p) * SET} + wl];')

    read(chunks[0])
    for gi, group in enumerate(chunks):
      if gi + 1 < len(chunks):
        read(chunks[gi + 1])
        w('__builtin_amdgcn_sched_barrier(0);')
      for c, ms in group:
        self.temporary_column(s, block, q, groups, c, ms, names, cols, ops)
    return ops

  def temporary_column(self, s, block, q, groups, c, ms, weights, cols, ops):
    w = self.w
    st, base, n = block
    names = [self.fresh('xt') for _ in range(n)]
    for x, (m, p) in enumerate(ms):
      for j in range(n):
        qv, sv = f'{q}{cols[m]}[{j}]', weights[(c, m)]
        if x == 0:
          w(f'{self.real} {names[j]} = {qv} * {sv};')
        else:
          w(f'{names[j]} = {self.fp.fma()}({qv}, {sv}, {names[j]});')
    for j in range(n):
      # rows past this term's own range (a wider term's rows) must not reach the product
      lim = s.krange[1] - s.k0
      top = s.kr.row(st + j, 3) + max(0, groups - 1) * 4 * self.nb * self.D
      if top >= lim:
        at = f'{base + j} + {n} * g' + (' + ro' if groups else '')
        w(f'{names[j]} = {at} < {lim} ? {names[j]} : ({self.real})0;')
      ops[j][c] = names[j]

  def post_operands(self, s: Stage, prev, prev_stage, half):
    """B operands of the next shared operand of a flux chain, per step: the previous product's
    result registers, cleared where they hold no row of its range."""
    w = self.w
    nprev = prev_stage.rows[1] - prev_stage.rows[0]
    lo, hi = max(0, s.krange[0] - s.k0), min(nprev, s.krange[1] - s.k0)
    out = []
    for j in range(s.kr.steps):
      ops = {}
      inside = all(lo <= s.kr.row(j, gg) < hi for gg in range(4))
      for c in half:
        v = self.acc_ref(prev, c, j)
        if not inside:
          x = self.fresh('xm')
          r = s.kr.row_expr(str(j), 'g')
          w(f'const {self.real} {x} = {r} >= {lo} && {r} < {hi} ? {v} : ({self.real})0;')
          v = x
        ops[c] = v
      out.append(ops)
    return out


def set_times(program, pl):
  """Microseconds a compute unit needs for a set of 16 elements: its share of the memory rate
  (5.9 TB/s measured over 256 units) for the compulsory bytes, and the matrix instructions on four
  SIMDs at 2.2 GHz (the clock under this load)."""
  f64 = program.fp_type == FloatingPointType.DOUBLE
  nb = 2 if f64 else 4

  def cycles(k, rows):
    steps = Rows(rows, nb).steps
    per = 64 * (steps // 4) + 16 * (steps % 4) if f64 else \
        32 * (steps // 4) + (8 * (steps % 4) if steps % 4 < 3 else 32)
    return Rows(k, nb).steps * per
  rows = pl.rows[1] - pl.rows[0]
  total = sum(cycles(t.product.k_ranges[0][1] - t.product.k_ranges[0][0], rows) for t in pl.terms)
  prev = rows
  for s in pl.post:
    total += cycles(prev, s.rows[1] - s.rows[0])
    prev = s.rows[1] - s.rows[0]
  memory = element_traffic(program).per_element * SET / 23000.0
  return memory, total * pl.q / 4 / 2200.0


def forms(program, pl):
  """The matrix-core forms that are faster than the vector stream, the fastest first: of 'staged'
  and 'direct'. Measured on 400 MB of operands, times in us.

  The staged form moves whole lines, but a set's steps are separated by barriers: it needs enough
  bytes per set of 16 elements, the more the better the vector stream's lanes use the lines of
  their columns. C += A B (vector / staged), columns of 112 bytes and more: 16 KB sets 97 / 95, 18 KB
  102 / 89, 9 KB 103 / 124; of 64 to 96 bytes: 18 KB 91 / 88, 12 KB 86 / 104; below: 36 KB 84 / 80,
  30 KB 84 / 94, 9 KB 80 / 122. Where a set is smaller the direct form is faster for columns of
  whole lines (16 x 16 FP64, one column: 99 / 84; 32 x 32 FP32, two columns: 100 / 86), but not for
  shorter ones (4 to 12 rows, two columns: 77-91 / 90-105).

  Flux chains FP32: 22 KB sets 99 vector / 91 staged, 16 KB 98 / 99; FP64 from 64 KB (44 KB 87 direct /
  86 staged, but 22 / 26 at 30,000 elements, where the direct form has four sets per workgroup). A
  chain of one shared operand per term is staged where memory time is as long as matrix time (35
  rows 171 direct / 160 staged, 40 rows 156 / 158), a set has 64 KB (55 KB 113 / 116) and its
  wavefronts form little more than the stored products: one quantity each and a share of a ninth
  (16 columns, 10 rows: 138 vector / 123 direct / 194 staged), with about as many weights in every
  column (28 rows, at most 5 weights in a column, 2.7 on average: 136 / 114 / 158; 3 in every
  column: 137 / 131 / 116).

  The direct form of a chain needs blocks of rows to work on. FP32 blocks have 16 rows (14 rows 127
  vector / 134 direct, 16 rows 129 / 111, flux chain 10 x 6 rows, three columns 87 / 141); with whole
  steps of 4 rows it is also faster than a vector form that selects many weights per lane (4 rows, 27
  weights 117 / 105, 9 weights 143 / 172), and from 13 columns on, where a wavefront of the vector form
  has four elements or fewer (8 rows, 16 columns 154 / 117, 14 rows, 13 columns 139 / 124 and with 100
  elements 14.7 / 10.8; 10 rows, 16 columns 152 / 187 and 16.9 / 12.3, 12 columns 107 / 199). FP64 blocks have 8 (6 rows
  117 / 109; 4 rows, 27 weights 119 / 87, 15 116 / 118, 12 92 / 100, 3 79 / 98). Of flux chains it
  holds two products' accumulators (56 x 21 rows FP64, 10 columns 111 / 109, 13 columns 118 / 129,
  16 columns 127 / 193)."""
  per_set = element_traffic(program).per_element * SET
  size = program.fp_type.size()
  stages = [t.product for t in pl.terms] + [s.product for s in pl.post]
  extents = [hi - lo for p in stages for lo, hi in (p.n_ranges[0], p.k_ranges[0])]
  few = min(extents)
  if pl.terms[0].kind == 'global':
    column = max(extents) * size
    if per_set >= (13.5 if column >= 112 else 17 if column >= 64 else 32) * 1024:
      return ['staged', 'direct']
    return ['direct'] if few * size >= 128 else []
  if pl.post:
    staged = per_set >= (20 if size == 4 else 64) * 1024
    whole = few >= 16 if size == 4 else few >= 6 or per_set >= 16 * 1024
    return ['staged'] * staged + ['direct'] * (whole and pl.q <= WAVES + 1)
  memory, matrix = set_times(program, pl)
  stored = [[len(ms) for _, ms in term_weights(t, range(pl.q))] for t in pl.terms]
  held = sum(map(max, stored))
  staged = memory >= 0.95 * matrix and per_set >= 64 * 1024 and pl.q <= WAVES + 1 and \
      held * pl.q <= 1.2 * sum(map(sum, stored))
  if size == 4:
    whole = few >= 16 or pl.q >= 13 or (held >= 16 and few % 4 == 0)
  else:
    whole = few >= 6 or held >= 15
  return ['staged'] * staged + ['direct'] * whole


def emit(program, context, base_name, pl, matrix='auto'):
  """(Emitted, None) or (None, reason). ``matrix``: 'auto', or the form to take."""
  # a flux chain's plan names its streamed operand once
  pl = replace(pl, terms=[replace(t, L=t.L or pl.L, l_cols=t.l_cols or pl.l_cols)
                          for t in pl.terms])
  reason = unsupported_reason(program, pl)
  if reason is not None:
    return None, reason
  from .staged import _Staged
  chosen = forms(program, pl) if matrix == 'auto' else [matrix]
  if not chosen:
    return None, 'the vector stream is faster'
  for form in chosen:
    em = (_Staged if form == 'staged' else _Tile)(program, context, base_name, pl).emit()
    if em is not None:
      if form == 'staged':
        em.masked = _Staged(program, context, base_name, pl, masked=True).emit()
        # with fewer sets there is little to save, and listing them takes 0.5-0.8 us of 9-60 (a
        # quarter masked, 4,096 elements: C += A B 11.4 without / 12.1 with lists, derivative step
        # 23.5 / 23.5, 10,000 elements 27.7 / 28.2 and 56.9 / 58.6)
        em.masked_from = 3 * SET
      return em, None
  return None, 'accumulators or shared operands do not fit'
