"""Vector form for few elements: chains with sparse shared operands whose launch does not fill the
GPU (small time clusters), where the time is that of one wavefront's instructions.

The streaming form (:mod:`stream`) gives a wavefront the whole work of its ``64 // q`` elements:
5,400 instructions for the order-6 volume chain, at two wavefronts per SIMD 18 us whatever the number
of elements. Here a workgroup of four wavefronts shares one such group. Its operands come through LDS
as in the staged matrix-core form (:mod:`staged`); then

1. each wavefront forms the temporaries ``L_t,e W_t,e`` of a quarter of the contraction rows and
   leaves them in LDS, one entry per lane;
2. each wavefront computes a quarter of the destination's rows from all temporaries, one
   DPP-broadcast FMA per stored entry, in the streaming form's order: the results of chains that
   overwrite their destination are the same to the last bit. (One that accumulates adds the old
   destination at the end here, the streaming form starts from it.)

Order-6 volume chain, streaming form / this one: 100 elements FP64 30.3 / 10.3 us, FP32 25.7 / 8.7;
1,792 elements (one group on each CU) 32.0 / 12.4 and 26.3 / 9.6. What is left is a chain of
latencies: the arguments, the loads (one latency for the operands, the shared entries and their
order), five barriers with an LDS latency each, 1,300 instructions of a wavefront's products at one
wavefront per SIMD. Eight wavefronts were tried: they read every temporary twice as often, which
the LDS bounds (14,336 elements 76 us against 58), and 100 elements take the same time.
"""
from dataclasses import replace
from typing import Optional

from ..common.basic_types import FloatingPointType
from .launcher import Emitted, Writer, fill_shared, kernel_params, persistent_grid
from .staged import _Pieces, _SetKernel
from .stream import CHUNK, _Stream
from .tile import LDS_LIMIT, WAVE, _ceil, set_unsupported_reason
from .traffic import element_traffic

WAVES = 4
THREADS = WAVE * WAVES


class _Part(_Stream):
  """A wavefront's share of the destination's rows; its shared entries sit in LDS from chunk
  ``chunk0`` on."""
  chunk0 = 0

  def chunk_ref(self, c):
    return f'ubuf[{(self.chunk0 + c) * CHUNK} + lane15]'


class _Phase:
  def __init__(self, terms):
    self.terms = terms


class _Small(_SetKernel):
  shared_last = False

  def __init__(self, program, context, base_name, schedule, pl):
    self.prog, self.ctx, self.pl = program, context, pl
    self.base_name = base_name
    self.kname = f'kernel_{base_name}_few'
    self.fp = program.fp_type
    self.real = FloatingPointType.as_str(self.fp)
    self.size = self.fp.size()
    self.per = 16 // self.size
    self.w = Writer()
    self.q = pl.q
    self.elements = WAVE // pl.q
    self.sched = schedule
    self.fused = pl.terms[0].kind == 'fused'
    self.n = 0

  def fresh(self, p):
    self.n += 1
    return f'{p}{self.n}'

  def beta_load(self):
    return self.pl.beta if self.pl.init == 'load' else None

  # ------------------------------------------------------------------ geometry
  def prepare(self):
    """Geometry; False when the chain does not fit this form."""
    pl, per = self.pl, self.per
    lo, hi = pl.rows
    part = _ceil(hi - lo, WAVES)
    self.parts, chunk = [], 0
    for r0 in range(lo, hi, part):
      sub = replace(pl, rows=(r0, min(hi, r0 + part)),
                    terms=[replace(t, entries=[]) for t in pl.terms])
      p = _Part(self.prog, self.ctx, self.base_name, self.sched, sub)
      p.w = self.w
      p.order_entries()
      p.pair = p.dma = False
      p.chunk0 = chunk
      chunk += p.nu_pad // CHUNK
      self.parts.append(p)
    t = pl.terms[0]
    if self.fused:
      X, row0, cols = t.L, pl.klo - t.L.origin[0], t.l_cols
      c0, step, ncols = (cols[0] - X.origin[1]) * X.strides[1], X.strides[1], cols[1] - cols[0]
    else:
      X, (kd, nd) = t.B, t.b_dims
      row0 = pl.klo - X.origin[kd]
      c0, step, ncols = (pl.cols[0] - X.origin[nd]) * X.strides[nd], X.strides[nd], self.q
    rows, nrows = pl.khi - pl.klo, hi - lo
    if min(rows, nrows) < per:
      return False
    # columns an odd number of entries apart: lanes reading one row of different columns meet no
    # bank conflict
    up = lambda n: _ceil(n, per) * per
    self.run, self.out_run = up(rows) | 1, up(nrows) | 1
    elem, out_elem = ncols * self.run, self.q * self.out_run
    base = chunk * CHUNK
    x = _Pieces('x', X.arg, rows, ncols, row0 + c0, step, up(rows), elem, base, per, self.run,
                self.elements, THREADS)
    dp = pl.dest_product
    (o0, o1), (_, s1) = dp.dest_origin, dp.dest_strides
    self.dest = pl.dest
    self.out = _Pieces('d', pl.dest, nrows, self.q, (pl.cols[0] - o1) * s1 + lo - o0, s1,
                       up(nrows), out_elem, base, per, self.out_run, self.elements, THREADS)
    base += up(self.elements * max(elem, out_elem))
    # weights of all terms
    items, off = [], 0
    for ti, t in enumerate(pl.terms) if self.fused else ():
      ps = [p for ms in self.columns(t) for _, p in ms]
      if not ps or max(ps) + 1 - min(ps) < per:
        return False
      items.append((ti, min(ps), max(ps) + 1 - min(ps), off))
      off += up(max(ps) + 1 - min(ps))
    self.wbase0, welem = base, off | 1
    stage = [(ti, first, o, _Pieces(f'w{ti}_', pl.terms[ti].W.arg, cnt, 1, first, 0, up(cnt), welem,
                                    base + o, per, None, self.elements, THREADS))
             for ti, first, cnt, o in items]
    self.xstage, self.wstage = [x], [(welem, stage)]
    self.old_early = True
    # temporaries: one entry per lane, contraction row and term
    self.tbase = base + up(self.elements * welem)
    self.K = rows
    # the shared operands as they are stored, until the temporaries take their place:
    # per term (first position, entries, offset)
    self.raw, n = [], 0
    for ti in range(len(pl.terms)):
      ps = [s[2][2] for p in self.parts for s in p.seq if s[1] == ti]
      first, cnt = (min(ps), max(ps) + 1 - min(ps)) if ps else (0, 0)
      self.raw.append((first, cnt, n))
      n += cnt
    self.raw_total, self.total = n, chunk * CHUNK
    if n == 0:
      return False
    words = self.tbase + max(n, len(pl.terms) * rows * WAVE if self.fused else 0)
    if _ceil(self.total, THREADS) > 64:
      return False
    self.lds_bytes = words * self.size
    pieces = [x, self.out] + [p for _, _, _, p in stage]
    return self.lds_bytes <= LDS_LIMIT and all(p.fits and p.count <= 8 for p in pieces)

  def columns(self, t):
    """Per output column: [(streamed column, position)] of term t's stored weights."""
    prod = t.producer
    mlo, mhi = prod.k_ranges[0]
    c_lo = prod.n_ranges[1][0]
    rk, rn = t.w_dims
    out = []
    for c in range(self.q):
      ms = []
      for m in range(mlo, mhi):
        idx = [0, 0]
        idx[rk], idx[rn] = m, c_lo + c
        pos = t.W.packed.get(tuple(idx)) if t.W.is_sparse() else t.W.offset(idx)
        if pos is not None:
          ms.append((m, pos))
      out.append(ms)
    return out

  # ------------------------------------------------------------------ emission
  def emit(self) -> Optional[Emitted]:
    if not self.prepare():
      return None
    w = self.w
    self.phases = [_Phase(list(range(len(self.pl.terms))))]
    entries = []
    for p in self.parts:
      tab = [e[2] - self.raw[ti][0] + self.raw[ti][2] for _, ti, e in p.seq]
      entries += tab + [0] * (p.nu_pad - len(tab))
    self.utab = self.table('utab', 'unsigned short' if self.raw_total < 65536 else 'unsigned',
                           entries)
    self.lane_values = []
    if self.fused:
      self.lane_slots()
      self.ltab = self.table('ltab', 'int', [x for vs in self.lane_values for x in vs])
    self.typedefs()
    params = ', '.join(kernel_params(self.prog, self.ctx))
    w(f'extern "C" __global__ void __launch_bounds__({THREADS}, 1) {self.kname}({params})')
    w('{')
    w._depth += 1
    w(f'// few elements: {self.elements} elements x {self.q} columns per workgroup, rows divided '
      f'among its {WAVES} wavefronts')
    self.body()
    w._depth -= 1
    w('}')
    traffic = element_traffic(self.prog)
    sched = {'kind': 'stream', 'few': True, 'waves_per_block': WAVES,
             'elements_per_wave': self.elements, 'columns': self.q,
             'shared_entries': sum(p.nu for p in self.parts), 'lds_bytes': self.lds_bytes,
             'dpp': self.sched.dpp}
    return Emitted(kernel_name=self.kname, kernel_src=w.src(), block=(THREADS, 1, 1),
                   elements_per_block=self.elements, lds_bytes=self.lds_bytes, emitter='tuned',
                   schedule=sched, bytes_per_element=traffic.per_element,
                   shared_bytes=traffic.shared, grid_override='tf_grid',
                   extra_launch_setup=persistent_grid(self.kname, self.lds_bytes, THREADS,
                                                      self.elements,
                                                      f'launcher_{self.base_name}'))

  def table(self, name, ctype, entries):
    w = self.w
    name = f'{self.kname}_{name}'
    w(f'#ifndef TF_{name}')
    w(f'#define TF_{name}')
    w(f'static __device__ const {ctype} {name}[{max(1, len(entries))}] = '
      f'{{{", ".join(map(str, entries)) or "0"}}};')
    w('#endif')
    return name

  def lane_slots(self):
    """Per term and weight slot: the streamed column (its offset in LDS) and the weight's position
    of the lane's column, as rows of a table (-1: no weight)."""
    lo = self.pl.terms[0].l_cols[0]
    self.slots, offsets = {}, {}
    for ti, t in enumerate(self.pl.terms):
      cols = self.columns(t)
      first = {ti: f for ti, f, _, _ in self.wstage[0][1]}[ti]
      self.slots[ti] = []
      for s in range(max(len(c) for c in cols)):
        ms = tuple(c[s][0] if s < len(c) else (c[0][0] if c else lo) for c in cols)
        if ms not in offsets:
          offsets[ms] = len(self.lane_values)
          self.lane_values.append([(m - lo) * self.run for m in ms])
        self.slots[ti].append((offsets[ms], len(self.lane_values)))
        self.lane_values.append([c[s][1] - first if s < len(c) else -1 for c in cols])
    self.offsets = list(offsets.values())

  def typedefs(self):
    w = self.w
    tag = 'D' if self.size == 8 else 'F'
    n = self.per
    w(f'#ifndef TF_PIECE_{tag}')
    w(f'#define TF_PIECE_{tag}')
    w(f'typedef {self.real} tf_p{tag} __attribute__((ext_vector_type({n})));')
    # in memory aligned as single entries are (odd offsets and row counts)
    w(f'typedef {self.real} tf_q{tag} __attribute__((ext_vector_type({n}), '
      f'aligned({self.size})));')
    w('#endif')
    self.lds_t = f'tf_p{tag}'
    self.vec_t = {n: f'tf_q{tag}'}

  def place(self):
    w, real, q, G = self.w, self.real, self.q, self.elements
    w(f'extern __shared__ __align__(16) {real} lds[];')
    w(f'{real}* __restrict__ ubuf = lds;')
    w(f'const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / {WAVE});')
    w(f'const int lane = threadIdx.x % {WAVE};')
    # lanes past the last element work on a copy of its first column
    w(f'const int slot = lane / {q} < {G} ? lane / {q} : {G - 1};')
    w(f'const int col = lane / {q} < {G} ? lane - slot * {q} : 0;')
    w(f'const bool own = lane < {G * q};')
    w('int lane15 = lane & 15;')
    x = self.xstage[0]
    w(f'const {real}* xs = lds + {x.lds_base} + slot * {x.lds_elem};')
    if not self.fused:
      w(f'int xoff = col * {self.run};')
    for i in range(len(self.lane_values)):
      w(f'const int lv{i} = {self.ltab}[{i * q} + col];')

  def shared(self):
    """The shared entries: as they are stored into LDS, beside the table of their order, then into
    that order. Reading them from memory in that order would take two latencies, one for the
    table."""
    w, real = self.w, self.real
    n = _ceil(self.total, THREADS)
    w(f'unsigned tv[{n}];')
    at = f'(int)threadIdx.x + i * {THREADS}'
    last = f'const int e = {at} < {self.total} ? {at} : {self.total - 1};'
    w('#pragma unroll')
    with w.block(f'for (int i = 0; i < {n}; ++i)'):
      w(last)
      w(f'tv[i] = {self.utab}[e];')
    ptr = lambda ti: f'{self.pl.terms[ti].U.arg.name} + {self.raw[ti][0] - self.raw[ti][2]}'
    pick = ptr(len(self.raw) - 1)
    for ti in range(len(self.raw) - 2, -1, -1):
      pick = f'(e < {self.raw[ti + 1][2]} ? {ptr(ti)} : {pick})'
    fill_shared(w, self.raw_total, THREADS,
                [(real, 'uv', [f'const {real}* up = {pick};'], 'up[e]')],
                lambda e, v: f'lds[{self.tbase} + {e}] = {v}')
    self.barrier()
    w('#pragma unroll')
    with w.block(f'for (int i = 0; i < {n}; ++i)'):
      w(last)
      w(f'ubuf[e] = lds[{self.tbase} + tv[i]];')

  def each_part(self, body):
    w = self.w
    for i, p in enumerate(self.parts):
      with w.block(f'{"else " if i else ""}if (wave == {i})'):
        body(p)

  def acc_declare(self):
    rows = self.parts[0].pl.rows
    self.w(f'{self.real} acc[{rows[1] - rows[0]}];')
    for i in range(rows[1] - rows[0]):
      self.w(f'acc[{i}] = ({self.real})0;')

  def compute(self, pi):
    if self.fused:
      with self.w.block(''):
        self.temporaries()
      self.barrier()
    self.each_part(self.products)

  def temporaries(self):
    w, real = self.w, self.real
    welem, stage = self.wstage[0]
    w(f'const {real}* wl = lds + {self.wbase0} + slot * {welem};')
    for ti, _, off, _ in stage:
      for _, i in self.slots[ti]:
        w(f'const {real} x{i} = wl[{off} + (lv{i} < 0 ? 0 : lv{i})];')
        w(f'const {real} v{i} = lv{i} < 0 ? ({real})0 : x{i};')
    rows = _ceil(self.K, WAVES)
    # the last wavefronts may repeat rows of the one before
    w(f'const int k0 = wave * {rows} < {self.K - rows} ? wave * {rows} : {self.K - rows};')
    for o in self.offsets:
      w(f'const int x{o} = lv{o} + k0;')
    for ti in self.slots:
      w(f'const int to{ti} = {self.tbase + ti * self.K * WAVE} + k0 * {WAVE} + lane;')
    for j in range(rows):
      with w.block(''):
        for o in self.offsets:
          w(f'const {real} q{o} = xs[x{o} + {j}];')
        for ti in self.slots:
          (o0, i0), *rest = self.slots[ti]
          w(f'{real} t{ti} = q{o0} * v{i0};')
          for o, i in rest:
            w(f't{ti} = {self.fp.fma()}(q{o}, v{i}, t{ti});')
          w(f'lds[to{ti} + {j * WAVE}] = t{ti};')

  def products(self, p):
    """All blocks of a part; the right operand's rows of a block are requested before the products
    of the block before."""
    w, real = self.w, self.real
    p.global_rows = {}
    terms = [replace(t, kind='global') for t in p.pl.terms]
    p.pl = replace(p.pl, terms=terms)

    if self.fused:
      # a base per term: the offsets of its rows fit the read instructions
      for ti in range(len(p.pl.terms)):
        w(f'int tb{ti} = {self.tbase + ti * self.K * WAVE} + lane;')
        w(f'asm("" : "+v"(tb{ti}));')

    def read(bi):
      p.global_rows[bi] = {}
      for ti, k in sorted({(s[1], s[2][1]) for s in p.seq if s[0] == bi}):
        v = p.fresh('gr')
        at = f'lds[tb{ti} + {(k - p.pl.klo) * WAVE}]' if self.fused else \
            f'xs[xoff + {k - p.pl.klo}]'
        w(f'const {real} {v} = {at};')
        p.global_rows[bi][(ti, k)] = v
    read(0)
    for bi, (b0, b1, _) in enumerate(p.blocks):
      w(f'// contraction rows [{b0}, {b1})')
      if bi + 1 < len(p.blocks):
        read(bi + 1)
      p.compute_block_pipelined(bi, b0, 'acc')

  def results(self):
    w, o = self.w, self.out

    def write(p):
      lo = p.pl.rows[0] - self.pl.rows[0]
      with w.block('if (own)'):
        w(f'{self.real}* __restrict__ ob = lds + {o.lds_base} + slot * {o.lds_elem} + '
          f'col * {self.out_run};')
        for i in range(p.pl.rows[1] - p.pl.rows[0]):
          w(f'ob[{lo + i}] = acc[{i}];')
    self.each_part(write)


def groups(em):
  """Most groups per CU of the launches the form is used for. Above one per CU its groups run one
  after the other, while the streaming form takes eight per CU at once: it is faster up to 3 for
  chains of some hundred shared entries, up to 2 for smaller ones (streaming /
  this form, volume chains FP64, 9 columns, 2, 3 and 4 rounds: 10 rows, 127 entries 7.0 / 6.3,
  7.6 / 8.0, 8.2 / 9.0 us; 20 rows, 481 entries 11.0 / 8.1, 12.0 / 10.1, 13.0 / 12.0; 35 rows, 1,489
  entries 20.2 / 13.7, 21.3 / 18.7, 22.5 / 23.5; 56 rows, 3,715 entries 33.6 / 19.3, 34.9 / 26.2,
  36.6 / 33.1; FP32, 84 rows, 8,522 entries 52.2 / 25.9, 54.6 / 35.8, 55.1 / 45.3)."""
  return 3 if em.schedule['shared_entries'] >= 400 else 2


def emit(program, context, base_name, schedule, pl):
  """Emitted, or None where the chain does not have the form."""
  if pl.stacked or pl.post or not any(t.U.is_sparse() for t in pl.terms):
    return None
  if pl.terms[0].kind == 'global' and len(pl.terms) > 1:
    return None
  pl = replace(pl, terms=[replace(t, L=t.L or pl.L, l_cols=t.l_cols or pl.l_cols)
                          for t in pl.terms])
  if set_unsupported_reason(program, pl) is not None:
    return None
  return _Small(program, context, base_name, schedule, pl).emit()
