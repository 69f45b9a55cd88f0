"""Matrix-core streaming form whose operands cross memory as whole runs (see :mod:`tile` for the
operand orders it shares).

Memory on this GPU wants whole 128-byte lines touched at once: reading and writing 16 elements in
64-byte pieces at a column's stride runs at 3.4-3.7 TB/s whatever the lane order, the same bytes as
one linear run of non-temporal 16-byte accesses at 5.9 TB/s (C += B over 65,536 elements of 56 x 9
doubles, buffers larger than the last-level cache). So a workgroup works on one set of 16 elements
at a time:

1. the set's streamed operand and weights, loaded one set ahead into registers as linear runs, go
   into LDS;
2. the old destination of this set and the operands of the next one are requested; they arrive
   while the matrix cores work;
3. each of the eight wavefronts forms the products of its own quantity (B operands are one 16-byte
   LDS read per streamed column and block; elements are 16 bytes off a multiple of the bank period,
   so 16 lanes reading the same row of 16 elements meet no conflict). A ninth quantity is divided
   so that every SIMD does the same work: its contraction among four wavefronts, each forming the
   temporaries of its own blocks only (derivative step, 131,071 elements: 549 us; divided by row
   tiles, with the temporaries of all rows in each of three wavefronts, 576). Further quantities go
   to one wavefront each;
4. the results replace the streamed operand in LDS and leave as a linear run, with the old
   destination added.

Loads are issued without branches around them and waited for before the results are stored: a
register written on two paths is copied where they meet, and the memory counter is in order, so
either mistake turns the requests of the next set into waits (flux integral 428 us with both, 337
without; derivative step 659 us with 21 spilled registers, 576 with none). Measured, vector form
before / this form: C += A B, 56 x 56 by 56 x 9, 65,536 elements FP64 208 / 138-142 us (5.6-5.7 TB/s);
local flux integral, 131,072 elements 468 / 331 us (5.0 TB/s, which is what a plain copy of 56 of
every 64 rows reaches); neighbour flux integral, 40,001 elements, every fourth masked 124 / 99-102 us
(116 with the masked ones moved and multiplied); time-derivative step, 131,071 elements
618 / 541-553 us, three arrays, 50,000 elements 293 / 250-254 us (both bound by the steps between the
barriers of a set: two wavefronts per SIMD do not cover their LDS latencies).
"""
from typing import Optional

from .launcher import Emitted, kernel_params, persistent_grid
from .tile import LDS_LIMIT, SET, WAVE, WAVES, _ceil, _Tile
from .traffic import element_traffic

THREADS = WAVE * WAVES
SHARES = 4                    # wavefronts that divide a ninth quantity, one on each SIMD


class _Pieces:
  """16-byte pieces of one per-element array, ``rows`` entries in each of ``cols`` runs. A thread
  moves the same piece of elements e0, e0 + step, ...: one offset per thread serves all of them."""

  def __init__(self, tag, arg, rows, cols, first, col_stride, lds_rows, lds_elem, lds_base, per,
               lds_run=None, elements=SET, threads=THREADS):
    self.tag, self.arg, self.rows, self.elements = tag, arg, rows, elements
    self.listed = False          # the set's elements come from a list: no distance between them
    self.first, self.col_stride = first, col_stride      # storage offset of run 0, of the next run
    self.lds_elem, self.lds_base = lds_elem, lds_base
    self.lds_run = lds_run or lds_rows                   # distance of two runs in LDS
    self.per = per
    # pieces lie on 16 bytes in LDS
    self.aligned = self.lds_run % per == 0 and lds_elem % per == 0
    self.runs = lds_rows // per                          # pieces of one run
    self.per_element = self.runs * cols
    self.fits = self.per_element <= threads
    self.count = _ceil(elements, min(elements, max(1, threads // self.per_element)))
    self.step = _ceil(elements, self.count)
    # offsets kept in registers over the loop, or formed anew at every use
    self.held, self.uses = True, 0
    # pieces that pass the end of the run start earlier and are moved down
    self.moved = lds_rows > rows

  def declare(self, w):
    """Before the loop: the thread's offsets where they are held, else its element, run and piece
    in one register."""
    t = self.tag
    w(f'int {t}k;' if not self.held else self.names())
    with w.block(''):
      w(f'const int pr = (int)threadIdx.x % {self.per_element};')
      w(f'const int pm = pr / {self.runs};')
      # threads without a piece: an element past the set (they read the last one's)
      w(f'const int pt = (int)threadIdx.x / {self.per_element};')
      w(f'const int pe = pt < {self.step} ? pt : {self.elements};')
      if self.held:
        w(f'const int pp = (pr - pm * {self.runs}) * {self.per};')
        self.offsets(w)
      else:
        w(f'{t}k = pe << 20 | pm << 12 | (pr - pm * {self.runs});')

  def setup(self, w):
    """The offsets, at a use."""
    if self.held:
      return
    t = self.tag
    w(self.names())
    with w.block(''):
      w(f'int pk = {t}k;')
      # may be scheduled freely, but neither leaves the loop nor serves another use as well
      self.uses += 1
      w(f'asm("; {t} {self.uses}" : "+v"(pk) : "s"((unsigned)set));')
      w('const int pe = pk >> 20;')
      w('const int pm = pk >> 12 & 255;')
      w(f'const int pp = (pk & 4095) * {self.per};')
      self.offsets(w)

  def names(self):
    t = self.tag
    return f'int {t}e, {t}g, {t}l{f", {t}h" if self.moved else ""};'

  def offsets(self, w):
    t = self.tag
    w(f'{t}e = pe;')
    sh = ''
    if self.moved:
      w(f'{t}h = pp > {self.rows - self.per} ? pp - {self.rows - self.per} : 0;')
      sh = f' - {t}h'
    e = '' if self.listed else f'{t}e * {self.arg.element_stride} + '
    w(f'{t}g = {e}{self.first} + pm * {self.col_stride} + pp{sh};')
    w(f'{t}l = {self.lds_base} + {t}e * {self.lds_elem} + pm * {self.lds_run} + pp;')

  def each(self, w, body):
    """``body(j)`` for every piece of the thread that exists."""
    even = self.step * self.count == self.elements
    n = self.count if even else self.count - 1
    with w.block(f'if ({self.tag}e < {self.elements})'):
      for j in range(n):
        body(j)
    if not even:
      with w.block(f'if ({self.tag}e + {n * self.step} < {self.elements})'):
        body(n)

  def at(self, j, bp='bp'):
    step = 0 if self.listed else j * self.step * self.arg.element_stride
    return f'{bp} + {step} + {self.tag}g'

  def lds(self, j):
    return f'lds + {self.tag}l + {j * self.step * self.lds_elem}'

  def element(self, j):
    return f'({self.tag}e + {j * self.step})'


class _SetKernel:
  """A workgroup's loop over sets of ``elements`` elements: the way of the operands and results
  between memory, registers and LDS. A form supplies its geometry (``xstage`` and ``wstage`` per
  phase, ``out``, ``dest``, ``old_early``) and ``place``, ``shared``, ``acc_declare``, ``compute``,
  ``results``.

  ``masked``: the kernel for launches with flags. It takes the same sets, 32 at a time, lists their
  active elements in LDS and forms sets of 16 from the list: masked elements are neither moved nor
  multiplied (an element's run is some KB, so whole lines remain). Vector form / sets of masked and
  active elements / this one: neighbour flux integral, 40,001 elements, every fourth masked 126 / 121
  / 102 us, nine tenths masked 86 / 114 / 29; C += A B, 65,536 elements 186 / 142 / 117 and 109 / 123 /
  32; derivative step, 131,071 elements 613 / 549 / 437 and 517 / 537 / 99. Where flags mask nothing the
  list costs 2-4 % (558 / 580 us)."""
  masked = False

  def barrier(self):
    # this wavefront's LDS accesses done, every wavefront here; memory accesses stay in flight
    self.w('asm volatile("s_waitcnt lgkmcnt(0)\\n\\ts_barrier" ::: "memory");')

  def body(self):
    w = self.w
    self.place()
    for x in self.xstage:
      x.declare(w)
    for _, stage in self.wstage:
      for _, _, _, p in stage:
        p.declare(w)
    self.out.declare(w)
    beta = self.beta_load()
    vt = self.lds_t
    n = max(x.count for x in self.xstage)
    w(f'{vt} {", ".join(f"xv{j}" for j in range(n))};')
    nw = max((sum(p.count for _, _, _, p in st) for _, st in self.wstage), default=0)
    if nw:
      w(f'{vt} {", ".join(f"wv{j}" for j in range(nw))};')
    if beta is not None:
      w(f'{vt} {", ".join(f"dv{j}" for j in range(self.out.count))};')
    touches = []
    if beta is not None and not self.old_early:
      touches = [f'touched{j}' for j in range(self.touches())]
      w(f'unsigned {", ".join(touches)};')
    if self.masked:
      self.shared()
      w(f'const size_t every = (numElements + {SET - 1}) / {SET};')
      with w.block(f'for (size_t first = blockIdx.x; first < every; '
                   f'first += {THREADS // SET}ull * gridDim.x)'):
        self.scan()
        w('if (nsets == 0) continue;')
        w('int set = 0;')
        self.fetch(0, 'set')
        self.arrived()
        with w.block('for (; set < nsets; ++set)'):
          self.one_set(beta, touches, 'set + 1')
      return
    w(f'const size_t nsets = (numElements + {self.elements - 1}) / {self.elements};')
    w('size_t set = blockIdx.x;')
    # the first set's operands are on their way while the shared ones are staged
    self.fetch(0, 'set')
    self.shared()
    self.arrived()
    with w.block('for (; set < nsets; set += gridDim.x)'):
      self.one_set(beta, touches, 'set + gridDim.x')

  def one_set(self, beta, touches, following):
    w = self.w
    self.acc_declare()
    for pi, ph in enumerate(self.phases):
      self.put(pi)
      self.barrier()
      last = pi == len(self.phases) - 1
      if last:
        if not self.masked:
          self.mask_load()
        if beta is not None and self.old_early:
          self.move(self.out, 'dv', 'set')
        elif beta is not None:
          self.touch()
        with w.block(f'if ({following} < nsets)'):
          self.fetch(0, f'({following})')
      else:
        self.fetch(pi + 1, 'set')
      self.compute(pi)
      self.barrier()
    self.results()
    self.barrier()
    if touches:
      w(f'asm volatile("" :: {", ".join(f"{chr(34)}v{chr(34)}({t})" for t in touches)});')
      self.move(self.out, 'dv', 'set')
    # the next set's operands have arrived before the results are stored: waiting for them
    # afterwards would wait for the stores as well
    self.arrived()
    self.leave(beta)
    self.barrier()

  # ------------------------------------------------------------------ active elements
  def list_bytes(self):
    return 2 * THREADS + 4 * WAVES

  def scan(self):
    """Lists the active elements of sets ``first``, ``first + gridDim.x``, ... in LDS: a thread's
    number is its place in these sets."""
    w = self.w
    w('{')
    w._depth += 1
    w(f'const size_t e = (first + threadIdx.x / {SET} * (size_t)gridDim.x) * {SET} + '
      f'threadIdx.x % {SET};')
    w('const bool on = e < numElements && flags[e] != 0u;')
    w('const unsigned long long ons = __ballot(on);')
    w('if (lane == 0) counts[wave] = __popcll(ons);')
    self.barrier()
    w('int at = __popcll(ons & ((1ull << lane) - 1ull));')
    w('listed = 0;')
    with w.block(f'for (int i = 0; i < {WAVES}; ++i)'):
      w('at += i < wave ? counts[i] : 0;')
      w('listed += counts[i];')
    w('if (on) list[at] = (unsigned short)threadIdx.x;')
    self.barrier()
    w('listed = __builtin_amdgcn_readfirstlane(listed);')
    w._depth -= 1
    w('}')
    w(f'const int nsets = (listed + {SET - 1}) / {SET};')

  def list_declare(self, base):
    """``base``: byte offset of the list in LDS."""
    w = self.w
    w(f'unsigned short* list = reinterpret_cast<unsigned short*>(lds) + {base // 2};')
    w(f'int* counts = reinterpret_cast<int*>(lds) + {(base + 2 * THREADS) // 4};')
    w('int listed;')

  def element_place(self, name, setexpr, slot):
    """``name``: the list's entry of a set's ``slot``, past the end its last one. The entries of all
    pieces are read before the first is used: one LDS latency for all of them."""
    at = f'{setexpr} * {SET} + {slot}'
    self.w(f'const int {name} = list[{at} < listed ? {at} : listed - 1];')

  def element_pointer(self, name, arg, place, const=''):
    self.w(f'{const}{self.real}* __restrict__ {name} = {arg.name} + ((first + ({place} >> 4) * '
           f'(size_t)gridDim.x) * {SET} + ({place} & 15)) * {arg.element_stride}ull + '
           f'{arg.name}_extraOffset;')

  # ------------------------------------------------------------------ memory <-> registers <-> LDS
  def arrived(self):
    """Waits for the registers of the first phase's operands."""
    held = [f'xv{j}' for j in range(self.xstage[0].count)]
    held += [f'wv{j}' for j in range(sum(p.count for _, _, _, p in self.wstage[0][1]))]
    for j in range(0, len(held), 8):
      self.w(f'asm volatile("" : {", ".join(f"{chr(34)}+v{chr(34)}({v})" for v in held[j:j + 8])});')

  def touch(self):
    """One load per 128-byte line of the old destination: the lines come into the L2 while the
    products run."""
    w = self.w
    o = self.out
    per = 128 // self.size
    end = o.first + (self.q - 1) * o.col_stride + o.rows        # of an element's window
    w('{')
    w._depth += 1
    if self.masked:
      lines = self.element_lines()
      for j in range(self.touches()):
        w(f'const int slot{j} = ((int)threadIdx.x + {j * THREADS}) / {lines};')
        w(f'const int line{j} = {o.first} + ((int)threadIdx.x + {j * THREADS} - slot{j} * {lines}) '
          f'* {per};')
        self.element_place(f'tc{j}', 'set', f'slot{j}')
        self.element_pointer(f'tp{j}', o.arg, f'tc{j}', 'const ')
        w(f'touched{j} = *reinterpret_cast<const unsigned*>(tp{j} + (line{j} < {end - 1} ? '
          f'line{j} : {end - 1}));')
      w._depth -= 1
      w('}')
      return
    w(f'const size_t left = numElements - set * {self.elements};')
    w(f'const int last = ((left < {self.elements} ? (int)left : {self.elements}) - 1) * '
      f'{o.arg.element_stride} + {end - 1};')
    w(f'const {self.real}* __restrict__ bp = {o.arg.name} + set * '
      f'{self.elements * o.arg.element_stride}ull + {o.arg.name}_extraOffset;')
    for j in range(self.touches()):
      w(f'const int line{j} = {o.first} + ((int)threadIdx.x + {j * THREADS}) * {per};')
      w(f'touched{j} = *reinterpret_cast<const unsigned*>(bp + (line{j} < last ? line{j} : last));')
    w._depth -= 1
    w('}')

  def element_lines(self):
    o = self.out
    return _ceil((self.q - 1) * o.col_stride + o.rows, 128 // self.size) + 1

  def touches(self):
    if self.masked:
      return _ceil(self.elements * self.element_lines(), THREADS)
    return _ceil(self.elements * self.dest.element_stride, 128 // self.size * THREADS)

  def mask_load(self):
    """The element's flag, requested early. Without flags the load reads the destination."""
    w = self.w
    e = f'set * {self.elements} + lane'
    w(f'const size_t ef = {e} < numElements ? {e} : numElements - 1;')
    w(f'const unsigned fv = *(flags != nullptr ? flags + ef : reinterpret_cast<const unsigned*>('
      f'{self.dest.name} + ef * {self.dest.element_stride}ull + {self.dest.name}_extraOffset));')

  def mask(self):
    """Bit e: element e of the set is to be stored."""
    if self.masked:
      self.w(f'const unsigned live = listed - set * {SET} >= {SET} ? {(1 << SET) - 1}u : '
             f'(1u << (listed - set * {SET})) - 1u;')
      return
    self.w(f'const unsigned long long live = __ballot(lane < {self.elements} && '
           f'set * {self.elements} + lane < numElements && (flags == nullptr || fv != 0u));')

  def move(self, x, name, setexpr, first=0, bp='bp'):
    """Registers ``{name}{first + j}`` <- the thread's pieces of array ``x`` of the set. Elements
    past the end of the batch are read as the last one."""
    w = self.w
    vt = self.vec_t[self.per]
    w('{')
    w._depth += 1
    if self.masked:
      x.setup(w)
      for j in range(x.count):
        self.element_place(f'c{j}', setexpr, x.element(j))
      for j in range(x.count):
        with w.block(''):
          self.element_pointer(bp, x.arg, f'c{j}', 'const ')
          w(f'{name}{first + j} = __builtin_nontemporal_load(reinterpret_cast<const {vt}*>('
            f'{x.at(j, bp)}));')
      w._depth -= 1
      w('}')
      return
    w(f'const {self.real}* __restrict__ {bp} = {x.arg.name} + {setexpr} * '
      f'{self.elements * x.arg.element_stride}ull + {x.arg.name}_extraOffset;')
    w(f'const size_t left = numElements - {setexpr} * {self.elements};')
    w(f'const int last = left < {self.elements} ? (int)left - 1 : {self.elements - 1};')
    x.setup(w)
    # no branch around a load: its register would be copied where the paths meet, and the copy
    # would wait for the load
    for j in range(x.count):
      with w.block(''):
        w(f'const int past = {x.element(j)} - last;')
        w(f'{name}{first + j} = __builtin_nontemporal_load(reinterpret_cast<const {vt}*>('
          f'{x.at(j, bp)} - (past > 0 ? past : 0) * {x.arg.element_stride}));')
    w._depth -= 1
    w('}')

  def moved_down(self, v, h):
    """Entries of a piece that was read ``h`` entries early, zeros past the end."""
    w = self.w
    for x in range(self.per):
      e = f'({self.real})0'
      for d in range(self.per - 1 - x, -1, -1):
        e = f'({h} == {d} ? {v}[{x + d}] : {e})'
      w(f'{v}[{x}] = {e};')

  def fetch(self, pi, setexpr):
    terms = self.phases[pi].terms
    self.w(f'// rows of term{"" if len(terms) == 1 else "s"} {", ".join(map(str, terms))}')
    self.move(self.xstage[pi], 'xv', setexpr, bp=f'lp_cur{pi or ""}')
    at = 0
    for _, _, _, p in self.wstage[pi][1]:
      self.move(p, 'wv', setexpr, at)
      at += p.count

  def put(self, pi):
    """The phase's operands from registers into LDS."""
    w = self.w
    at = 0
    for p, name in [(self.xstage[pi], 'xv')] + [(p, 'wv') for _, _, _, p in self.wstage[pi][1]]:
      first = at if name == 'wv' else 0

      def store(j):
        v = f'{name}{first + j}'
        if p.moved:
          self.moved_down(v, f'{p.tag}h')
        if p.aligned:
          w(f'*reinterpret_cast<{self.lds_t}*>({p.lds(j)}) = {v};')
        else:
          for x in range(self.per):
            w(f'({p.lds(j)})[{x}] = {v}[{x}];')
      with w.block(''):
        p.setup(w)
        p.each(w, store)
      at += p.count if name == 'wv' else 0

  def leave(self, beta):
    """The results from LDS into the destination, the old one added; whole sets without a mask
    take the first branch."""
    w = self.w
    o = self.out
    vt = self.vec_t[self.per]
    o.setup(w)
    scale = '' if beta in (None, 1.0) else f'{self.fp.literal(beta)} * '
    if not self.masked:
      w(f'{self.real}* __restrict__ bp = {o.arg.name} + set * '
        f'{self.elements * o.arg.element_stride}ull + {o.arg.name}_extraOffset;')

    if self.shared_last:
      # the thread's place in the other shares of the last quantity
      w(f'const int sl = dl - {o.lds_base + (self.q - 1) * o.lds_run} - de * {o.lds_elem};')
      w(f'const {self.real}* sp = lds + {self.share_base} + de * {self.share_elem} + sl;')

    def write(j):
      if self.masked:
        self.element_pointer('bp', o.arg, f'c{j}')
      if o.aligned:
        w(f'{self.lds_t} rv = *reinterpret_cast<const {self.lds_t}*>({o.lds(j)});')
      else:
        w(f'{self.lds_t} rv = {{{", ".join(f"({o.lds(j)})[{x}]" for x in range(self.per))}}};')
      if self.shared_last:
        # (all of them before the first is added: 29 spilled registers, 582 us against 549)
        with w.block('if (sl >= 0)'):
          for i in range(SHARES - 1):
            w(f'rv += *reinterpret_cast<const {self.lds_t}*>(sp + '
              f'{(j * o.step + i * SET) * self.share_elem});')
      if beta is not None:
        if o.moved:
          self.moved_down(f'dv{j}', 'dh')
        w(f'rv = {scale}dv{j} + rv;')
      full = f'__builtin_nontemporal_store(({vt})rv, reinterpret_cast<{vt}*>({o.at(j)}));'
      if not o.moved:
        w(full)
        return
      with w.block('if (dh == 0)'):
        w(full)
      with w.block('else'):
        for x in range(o.rows % o.per):
          w(f'({o.at(j)})[dh + {x}] = rv[{x}];')

    def masked(j):
      with w.block(f'if (live >> {o.element(j)} & 1ull)'):
        write(j)

    def scoped(body):
      def run(j):
        with w.block(''):
          body(j)
      return run

    self.mask()
    if self.masked:
      for j in range(o.count):
        self.element_place(f'c{j}', 'set', o.element(j))
    with w.block(f'if (live == {(1 << self.elements) - 1}ull)'):
      o.each(w, scoped(write))
    with w.block('else'):
      o.each(w, scoped(masked))


class _Staged(_SetKernel, _Tile):
  elements = SET

  def __init__(self, program, context, base_name, pl, masked=False):
    super().__init__(program, context, base_name, pl)
    self.masked = masked
    if masked:
      self.kname += '_m'

  def prepare(self):
    """Geometry; False when the chain does not fit this form."""
    pl = self.pl
    self.parts, self.sets = 1, 1
    self.halves = [list(range(self.q))]
    self.per = 16 // self.size
    per = self.per
    in_turn = pl.stacked or not self.fused
    self.stages, self.post, self.phases, koff, _ = self.plan(pl.rows, in_turn)
    self.last = self.post[-1] if self.post else self.stages[0]
    self.dest, (o0, o1), (s0, s1) = self.dest_pointer()
    # streamed operand, then the results, in the same region
    skew = lambda n, mod: n + (per - n) % mod
    self.xstage, region = [], 0
    for ph in self.phases:
      cols = ph.cols if ph.cols is not None else [pl.cols[0] + c for c in range(self.q)]
      rows, lds_rows = ph.kr.n, 4 * ph.kr.steps
      if rows < per or lds_rows % per:
        return False
      elem = skew(lds_rows * len(cols), 256 // self.size)
      step = self.col_off(ph, cols[-1]) - self.col_off(ph, cols[0])
      step = step // (len(cols) - 1) if len(cols) > 1 else 0
      self.xstage.append(_Pieces(f'x{len(self.xstage)}', ph.X.arg, rows, len(cols),
                                 ph.row0 + self.col_off(ph, cols[0]), step, lds_rows, elem, koff,
                                 per))
      region = max(region, SET * elem)
    dr = self.last.dr
    nrows = self.last.rows[1] - self.last.rows[0]
    lds_rows = 4 * dr.steps
    if nrows < per or lds_rows % per:
      return False
    elem = skew(lds_rows * self.q, 256 // self.size)
    region = max(region, SET * elem)
    out_rows = _ceil(nrows, per) * per
    self.out = _Pieces('d', self.dest, nrows, self.q,
                       (pl.cols[0] - o1) * s1 + self.last.rows[0] - o0, s1, out_rows, elem, koff,
                       per, lds_rows)
    self.out_lds_rows = lds_rows
    # weights: the span of stored positions of every term of a phase
    wbase = koff + region
    self.wstage, wsize = [], 0
    for ph in self.phases:
      items, off = [], 0
      for ti in ph.terms if self.fused else ():
        t = pl.terms[ti]
        lo, hi = self.weight_span(t, self.halves[0])
        if hi - lo < per:
          return False
        items.append((ti, lo, hi - lo, off))
        off += _ceil(hi - lo, per) * per
      elem = off + (per - off) % (2 * per) if off else 0
      stage = []
      for ti, lo, cnt, o in items:
        stage.append((ti, lo, o, _Pieces(f'w{ti}_', pl.terms[ti].W.arg, cnt, 1, lo, 0,
                                         _ceil(cnt, per) * per, elem, wbase + o, per)))
      self.wstage.append((elem, stage))
      wsize = max(wsize, SET * elem)
    self.wbase0 = wbase
    self.lds_bytes = (wbase + wsize) * self.size
    pieces = self.xstage + [self.out] + [p for _, st in self.wstage for _, _, _, p in st]
    # more than eight pieces a thread leave too few registers (84 rows x 9 columns, 16 pieces: 356 us
    # against 295 in the direct form; 56 x 13: 319 against 268)
    if self.lds_bytes > LDS_LIMIT or not all(p.fits and p.count <= 8 for p in pieces):
      return False
    # a wavefront's quantities: its own and one more, or a share of the ninth: SHARES wavefronts
    # divide its contraction, their sums meet in LDS in place of the weights or behind them
    self.extra = max(0, self.q - WAVES)
    self.share_base, self.share_elem = wbase, skew(lds_rows, 256 // self.size)
    end = max(wbase + wsize, wbase + (SHARES - 1) * SET * self.share_elem) * self.size
    self.shared_last = self.extra == 1 and not self.post and self.fused and end <= LDS_LIMIT
    # a bare product waits for memory: its ninth quantity is divided by row tiles, which adds
    # nothing to the way of the results (138 us; in shares of the contraction 142)
    self.tiled_last = self.extra == 1 and not self.post and not self.fused
    if self.shared_last:
      self.lds_bytes = max(self.lds_bytes, end)
    self.list_base = self.lds_bytes
    if self.masked:
      self.lds_bytes += self.list_bytes()
      if self.lds_bytes > LDS_LIMIT:
        return False
    cols = 1 if self.extra == 0 or self.shared_last or self.tiled_last else 2
    acc = max((4 * self.tiles(s.dr)[0] + self.tiles(s.dr)[1] * (1 if self.f64 else 5))
              for s in self.stages + self.post)
    # the share's accumulators beside the own ones only over several phases
    acc = acc * (2 if self.shared_last and len(self.phases) > 1 else cols) + 4 * self.tiled_last
    # registers (32-bit): accumulators, operands on the way, streamed rows, weights
    words = self.size // 4
    held = 4 * (max(x.count for x in self.xstage) +
                max((sum(p.count for _, _, _, p in st) for _, st in self.wstage), default=0))
    reads = max(sum(4 if len(set(k)) == 1 else 4 * cols + 4 * self.tiled_last
                    for k in self.keys(ph)) for ph in self.phases)
    slots = max(sum(len(self.slots(ti)) for ti in ph.terms) for ph in self.phases) * words \
        if self.fused else 0
    use = acc * words + held + reads + slots + 3 * len(pieces) + 48
    # the old destination waits in registers of its own, or where they do not suffice its lines are
    # requested into the L2 early and read when they are needed
    old = 4 * self.out.count if self.beta_load() is not None else 0
    self.old_early = use + old <= 256
    if self.old_early:
      use += old
    # three or four registers per array: with up to three arrays all offsets stay, with more of them
    # those of the destination (they are needed at once, between two barriers) unless several
    # streamed operands take turns. What does not fit is spilled, and a spilled register's reload
    # waits for every load in flight (derivative step 131,071 elements, all held 659 us, none 606,
    # the destination's 578; three arrays, 50,000 elements, 278 / 252 / 259 us; flux integral, three
    # arrays here, all 331 us, none 345)
    for p in pieces:
      p.listed = self.masked
      p.held = len(pieces) <= 3 or (p is self.out and len(self.phases) == 1)
    self.weights_held = 2 if use + slots <= 256 else 1
    return use <= 256

  def beta_load(self):
    """Factor of the old destination, or None."""
    pl = self.pl
    init, beta = (pl.final_init, pl.final_beta) if pl.post else (pl.init, pl.beta)
    return beta if init == 'load' else None

  # ------------------------------------------------------------------ weights of a column
  def slots(self, ti):
    """Weight slots of term ``ti``: per slot ([streamed column per quantity], [position or -1])."""
    cols = [ms for _, ms in self.weights(self.pl.terms[ti], range(self.q))]
    n = max(len(c) for c in cols)
    lo = self.pl.terms[ti].l_cols[0]
    out = []
    for s in range(n):
      m = [c[s][0] if s < len(c) else (c[0][0] if c else lo) for c in cols]
      p = [c[s][1] if s < len(c) else -1 for c in cols]
      out.append((tuple(m), tuple(p)))
    return out

  def keys(self, ph):
    """The distinct streamed columns (as functions of the quantity) a phase's terms read."""
    if not self.fused:
      return [tuple(range(self.q))]
    out = []
    for ti in ph.terms:
      for m, _ in self.slots(ti):
        if m not in out:
          out.append(m)
    return out

  @staticmethod
  def select(values, c):
    d = values[1] - values[0] if len(values) > 1 else 0
    if all(v == values[0] + i * d for i, v in enumerate(values)):
      return str(values[0]) if d == 0 else f'({values[0]} + {c} * {d})'
    expr = str(values[-1])
    for i in range(len(values) - 2, -1, -1):
      expr = f'({c} == {i} ? {values[i]} : {expr})'
    return expr

  # ------------------------------------------------------------------ emission
  def emit(self) -> Optional[Emitted]:
    if not self.prepare():
      return None
    w = self.w
    pl = self.pl
    self.typedefs()
    params = ', '.join(kernel_params(self.prog, self.ctx))
    w(f'extern "C" __global__ void __launch_bounds__({THREADS}, 2) {self.kname}({params})')
    w('{')
    w._depth += 1
    w(f'// matrix-core streaming, one set of {SET} elements per workgroup at a time')
    self.body()
    w._depth -= 1
    w('}')
    traffic = element_traffic(self.prog)
    sched = {'kind': 'stream', 'matrix': 'mfma', 'staged': True, 'waves_per_block': WAVES,
             'elements_per_wave': SET, 'columns': self.q,
             'shared_entries': self.entry_count(), 'lds_bytes': self.lds_bytes}
    return Emitted(kernel_name=self.kname, kernel_src=w.src(), block=(THREADS, 1, 1),
                   elements_per_block=SET, lds_bytes=self.lds_bytes, emitter='tuned',
                   schedule=sched, bytes_per_element=traffic.per_element,
                   shared_bytes=traffic.shared, grid_override='tf_grid',
                   extra_launch_setup=persistent_grid(self.kname, self.lds_bytes, THREADS, SET,
                                                      f'launcher_{self.base_name}'))

  def place(self):
    w = self.w
    real = self.real
    w(f'extern __shared__ __align__(16) {real} lds[];')
    w(f'{real}* __restrict__ ubuf = lds;')
    w(f'const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / {WAVE});')
    w(f'const int lane = threadIdx.x % {WAVE};')
    w('const int el = lane % 16;')
    w('const int g = lane / 16;')
    w(f'const {real}* __restrict__ ka = ubuf + lane;')
    w(f'const {real}* __restrict__ ks = ubuf + (lane % 4 + 4 * g);')
    if self.masked:
      self.list_declare(self.list_base)

  def shared(self):
    for s in self.stages + self.post:
      self.stage_shared(s)

  # ------------------------------------------------------------------ products
  def columns(self):
    """Variants of the wavefronts' work: [(condition, [(acc name, quantity, tiles)])]. ``tiles``
    None: all; ('u',): 16-row tile number ``wave``; ('r', big, small): the remaining tiles."""
    own = ('acc', 'wave', None)
    if self.q < WAVES:
      return [(f'wave < {self.q}', [own])]
    if not self.extra or self.shared_last:
      return [('', [own])]
    if not self.tiled_last:
      return [(f'wave < {self.extra}', [own, ('acx', f'(wave + {WAVES})', None)]), ('', [own])]
    big, small = self.tiles(self.last.dr)
    # 16-row tiles made of whole blocks are alike: tile ``wave``; the others together
    uniform = big if self.f64 else self.last.dr.full
    out = []
    if uniform:
      out.append((f'wave < {uniform}', [own, ('acu', str(WAVES), ('u',))]))
    rest = (tuple(range(uniform, big)), tuple(range(small)))
    if rest[0] or rest[1]:
      out.append((f'wave == {uniform}', [own, ('acr', str(WAVES), ('r',) + rest)]))
    out.append(('', [own]))
    return out

  def acc_declare(self):
    """Accumulators of every variant (a wavefront uses its own), cleared."""
    first = self.stages[0].dr
    names = {n for _, cols in self.columns() for n, _, _ in cols}
    if self.shared_last:
      names.add('acx')
    for n in ('acc', 'acx'):
      if n in names:
        self.declare_acc(n, first, [0])
        for i, s in enumerate(self.post):
          self.declare_acc(f'{n}p{i}', s.dr, [0])
    if 'acu' in names:
      self.declare_acc('acu', first, [0], ((0,), ()))
    if 'acr' in names:
      tiles = next(t for _, cols in self.columns() for n, _, t in cols if n == 'acr')
      self.declare_acc('acr', first, [0], tiles[1:])

  def variants(self, emit):
    w = self.w
    for i, (cond, cols) in enumerate(self.columns()):
      head = f'if ({cond})' if cond else ''
      with w.block(('else ' if i else '') + head):
        emit(cols)

  def compute(self, pi):
    self.variants(lambda cols: self.compute_columns(pi, cols))
    if self.shared_last:
      with self.w.block(f'if (wave < {SHARES})'):
        self.compute_share(pi)

  def compute_share(self, pi):
    """The wavefront's blocks of the last quantity's contraction, every fourth one (fused chains)."""
    w, real, ph = self.w, self.real, self.phases[pi]
    x, c = self.xstage[pi], self.q - 1
    welem, wst = self.wstage[pi]
    keys = self.keys(ph)
    col0 = ph.cols[0]
    w(f'const {real}* __restrict__ xb = lds + {x.lds_base} + el * {x.lds_elem};')
    w(f'const {real}* __restrict__ wb = lds + {self.wbase0} + el * {welem};')
    offs = {ti: off - lo for ti, lo, off, _ in wst}

    def block(st, base, n):
      for ki, m in enumerate(keys):
        at = f'xb + {(m[c] - col0) * x.lds_run} + {base} + {n} * g'
        if n == self.per:
          w(f'const {self.lds_t} u{ki} = *reinterpret_cast<const {self.lds_t}*>({at});')
        else:
          w(f'{self.lds_t} u{ki} = {{{", ".join(f"({at})[{j}]" for j in range(n))}}};')
      for ti in ph.terms:
        s = self.stages[ti]
        ops = []
        for j in range(n):
          t, first = self.fresh('xt'), True
          for m, p in self.slots(ti):
            if p[c] < 0:
              continue
            v, u = f'wb[{offs[ti] + p[c]}]', f'u{keys.index(m)}[{j}]'
            w(f'{real} {t} = {u} * {v};' if first else f'{t} = {self.fp.fma()}({u}, {v}, {t});')
            first = False
          if first:
            w(f'{real} {t} = ({real})0;')
          lim = s.krange[1] - s.k0
          if lim < 4 * ph.kr.steps:
            # rows past this term's own range must not reach the product
            w(f'{t} = {base} + {j} + {n} * g < {lim} ? {t} : ({real})0;')
          ops.append(t)
        for j in range(n):
          self.step(s, f'{s.base} + ({st} + {j}) * {self.fragment(s.dr)}', [('acx', str(c), None)], [ops[j]])

    if ph.kr.full:
      with w.block(f'for (int b = wave; b < {ph.kr.full}; b += {SHARES})'):
        block(f'b * {self.nb}', f'b * {4 * self.nb}', self.nb)
    if ph.kr.tail:
      with w.block(f'if (wave == {ph.kr.full % SHARES})'):
        block(ph.kr.full * self.nb, ph.kr.full * 4 * self.nb, ph.kr.tail)
    if pi == len(self.phases) - 1:
      self.finish('acx', self.stages[-1].dr, [0])

  def compute_columns(self, pi, cols):
    w = self.w
    ph = self.phases[pi]
    x = self.xstage[pi]
    real = self.real
    blocks = ph.kr.blocks()
    last = pi == len(self.phases) - 1
    w(f'const {real}* __restrict__ xb = lds + {x.lds_base} + el * {x.lds_elem};')
    welem, wst = self.wstage[pi]
    keys = self.keys(ph)
    col0 = ph.cols[0] if ph.cols is not None else 0
    wreg = {}
    for ci, (name, c, _) in enumerate(cols):
      for ki, m in enumerate(keys):
        w(f'const int mo{ci}_{ki} = {self.select([v - col0 for v in m], c)} * {x.lds_run};')
      for ti, lo, off, _ in wst:
        for si, (m, p) in enumerate(self.slots(ti)):
          v = f'wr{ci}_{ti}_{si}'
          w(f'const int {v}p = {self.select(p, c)};')
          at = f'lds[{self.wbase0 + off - lo} + el * {welem} + ({v}p < 0 ? {lo} : {v}p)]'
          value = f'{v}p < 0 ? ({real})0 : {v}x' if -1 in p else f'{v}x'
          if ci < self.weights_held:
            w(f'const {real} {v}x = {at};')
            w(f'const {real} {v} = {value};')
            wreg[(ci, ti, si)] = (v, None)
          else:
            wreg[(ci, ti, si)] = (v, (at.replace('el *', 'wl *'), value))
    if len(cols) > self.weights_held:
      w('int wl = el;')

    # a key that is the same streamed column for every quantity is read once
    same = lambda ki: len(set(keys[ki])) == 1
    uc = lambda ci, ki: f'u{0 if same(ki) else ci}_{ki}'

    def read(bi):
      """B pieces of block bi of every column's keys."""
      st, base, n = blocks[bi]
      for ci in range(len(cols)):
        for ki in range(len(keys)):
          if ci and same(ki):
            continue
          if n == self.per:
            w(f'u{ci}_{ki} = *reinterpret_cast<const {self.lds_t}*>(xb + mo{ci}_{ki} + '
              f'{base} + {n} * g);')
          else:
            for j in range(n):
              w(f'u{ci}_{ki}[{j}] = xb[mo{ci}_{ki} + {base + j} + {n} * g];')

    names = ', '.join(f'u{ci}_{ki}' for ci in range(len(cols)) for ki in range(len(keys)))
    w(f'{self.lds_t} {names};')
    read(0)
    for bi, (st, base, n) in enumerate(blocks):
      for ti in ph.terms:
        s = self.stages[ti]
        F = self.fragment(s.dr)
        ops = [[None] * len(cols) for _ in range(n)]
        for ci, (name, c, _) in enumerate(cols):
          if not self.fused:
            for j in range(n):
              ops[j][ci] = f'u{ci}_0[{j}]'
            continue
          t = [self.fresh('xt') for _ in range(n)]
          if ci >= self.weights_held:
            w('asm volatile("" : "+v"(wl));')
          for si, (m, _) in enumerate(self.slots(ti)):
            v, source = wreg[(ci, ti, si)]
            if source is not None:
              r = self.fresh('xs')
              w(f'const {real} {r}x = {source[0]};')
              w(f'const {real} {r} = {source[1].replace(v + "x", r + "x")};')
              v = r
            ki = keys.index(m)
            for j in range(n):
              if si == 0:
                w(f'{real} {t[j]} = {uc(ci, ki)}[{j}] * {v};')
              else:
                w(f'{t[j]} = {self.fp.fma()}({uc(ci, ki)}[{j}], {v}, {t[j]});')
          for j in range(n):
            lim = s.krange[1] - s.k0
            if s.kr.row(st + j, 3) >= lim:
              # rows past this term's own range must not reach the product
              w(f'{t[j]} = {base + j} + {n} * g < {lim} ? {t[j]} : ({real})0;')
            ops[j][ci] = t[j]
        copied = None
        if ti == ph.terms[-1] and bi + 1 < len(blocks):
          if not self.fused:
            # the rows are operands themselves: keep them while the next ones arrive
            for ci in range(len(cols)):
              for j in range(n):
                copied = self.fresh('xc')
                w(f'const {real} {copied} = {ops[j][ci]};')
                ops[j][ci] = copied
          read(bi + 1)
        # a fence behind the products of a term: with another before them the fragments are read
        # only once the temporaries are formed (derivative step 556 us, now 543), without any the
        # registers do not suffice (600)
        for j in range(n):
          self.step(s, f'{s.base + (st + j) * F}', cols, ops[j])
        w('__builtin_amdgcn_sched_barrier(0);')
    if last:
      for name, _, tiles in cols:
        self.finish(name, self.stages[-1].dr, [0],
                    None if tiles is None else ((), tiles[2] if tiles[0] == 'r' else ()))
    if last and self.post:
      prev_stage = self.stages[-1]
      for i, s in enumerate(self.post):
        per_col = []
        for name, c, _ in cols:
          per_col.append(self.post_operands(s, name if i == 0 else f'{name}p{i - 1}', prev_stage,
                                            [0]))
        for j in range(s.kr.steps):
          self.step(s, f'{s.base + j * self.fragment(s.dr)}',
                    [(f'{name}p{i}', c, t) for name, c, t in cols], [o[j][0] for o in per_col])
        for name, _, _ in cols:
          self.finish(f'{name}p{i}', s.dr, [0])
        prev_stage = s

  def step(self, s, off, cols, ops):
    """One contraction step of every column of the variant: a fragment read serves all of them."""
    w = self.w
    big, small = self.tiles(s.dr)
    whole = [(name, op) for (name, _, t), op in zip(cols, ops) if t is None]
    rest = [(name, t, op) for (name, _, t), op in zip(cols, ops) if t is not None]
    fn = '__builtin_amdgcn_mfma_f64_16x16x4f64' if self.f64 else '__builtin_amdgcn_mfma_f32_16x16x4f32'
    for t in range(big):
      a = self.fresh('xa')
      w(f'const {self.real} {a} = ka[{off} + {64 * t}];')
      for name, op in whole + [(nm, op) for nm, tiles, op in rest
                               if tiles[0] == 'r' and t in tiles[1]]:
        w(f'{name}_0_{t} = {fn}({a}, {op}, {name}_0_{t}, 0, 0, 0);')
    for i in range(small):
      a = self.fresh('xa')
      w(f'const {self.real} {a} = ks[{off} + {64 * big + 16 * i}];')
      for name, op in whole + [(nm, op) for nm, tiles, op in rest
                               if tiles[0] == 'r' and i in tiles[2]]:
        self.mfma_small(f'{name}_0', i, a, op)
    for name, tiles, op in rest:
      if tiles[0] == 'u':
        a = self.fresh('xa')
        w(f'const {self.real} {a} = ka[{off} + 64 * wave];')
        w(f'{name}_0_0 = {fn}({a}, {op}, {name}_0_0, 0, 0, 0);')

  # ------------------------------------------------------------------ results
  def results(self):
    w, o = self.w, self.out
    ob = f'{self.real}* __restrict__ ob = lds + {o.lds_base} + el * {o.lds_elem}'

    def columns(cols):
      w(f'{ob};')
      for name, c, tiles in cols:
        self.result_column(name, f'{c} * {self.out_lds_rows}', tiles)
    self.variants(columns)
    if self.shared_last:
      with w.block(f'if (wave < {SHARES})'):
        # the first share in its place, the others to be added to it
        w(f'{ob};')
        w(f'const int at = wave == 0 ? {(self.q - 1) * o.lds_run} : {self.share_base - o.lds_base} + '
          f'((wave - 1) * {SET} + el) * {self.share_elem} - el * {o.lds_elem};')
        self.result_column('acx', 'at')

  def result_column(self, name, at, tiles=None):
    w = self.w
    dr = self.last.dr
    if self.post:
      name = f'{name}p{len(self.post) - 1}'
    if tiles is not None and tiles[0] == 'u':
      # one 16-row tile, number ``wave``: whole blocks
      for b in range(4 // self.nb):
        vals = ', '.join(f'{name}_0_0[{b * self.nb + j}]' for j in range(self.nb))
        w(f'*reinterpret_cast<{self.lds_t}*>(ob + {at} + 16 * wave + {b * 4 * self.nb} + '
          f'{self.nb} * g) = {self.lds_t}{{{vals}}};')
      return
    held = None
    if tiles is not None:
      big = self.tiles(dr)[0]
      held = [4 * t + x for t in tiles[1] for x in range(4)] + [4 * big + x for x in tiles[2]]
    for st, base, n in dr.blocks():
      if held is not None and st not in held:
        continue
      refs = [self.acc_ref(name, 0, st + j) for j in range(n)]
      if n == self.per:
        w(f'*reinterpret_cast<{self.lds_t}*>(ob + {at} + {base} + {n} * g) = '
          f'{self.lds_t}{{{", ".join(refs)}}};')
      else:
        for j in range(n):
          w(f'ob[{at} + {base + j} + {n} * g] = {refs[j]};')
