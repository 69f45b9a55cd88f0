"""Timed cases: launches of the generated kernels as a solver's time loop makes them.

Every case is one launch through the public entry points (``catalog.load`` / ``load_group``, then
``device.launch`` or the grouped launcher) on operands that stay on the GPU:

* ``volume``: the ADER-DG volume chain ``Q' = sum_d K_d Q S_d`` (order 6: 56 basis functions,
  9 quantities; sparse or dense ``K_d``, FP64 or FP32; order 7: 84 basis functions, dense);
* ``mixed``: the same chain over elements of orders 2..7 in one grouped launch;
* ``flux``: the local / neighbour flux integrals, accumulated into the degrees of freedom;
* ``derivative``: one step of the time-derivative recursion, from one array or from three;
* ``gemm``: one batched product ``C += A B`` with a shared ``A``.

Element counts run from a small time cluster (launch latency) to a whole partition, odd counts
included. ``flags`` masks elements as local time stepping does (a quarter of them is skipped);
``offset`` shifts every per-element operand by that many entries (``extraOffset``).
"""
import math

import numpy as np
import torch

from tensorforge_amd import catalog
from tensorforge_amd import workloads as W
from tensorforge_amd.device import launch, launch_args

Q = 9                       # quantities
STAR_NNZ = len(W.STAR_PATTERN)
DTYPES = {'f64': torch.float64, 'f32': torch.float32}


def listed():
  return [
    # the headline workload: a whole partition's volume step
    dict(name='volume_f64', kind='volume', order=6, k='sparse', dtype='f64', n=262144,
         flags=False, offset=0),
    # a small time cluster: one launch's latency
    dict(name='volume_f64_small', kind='volume', order=6, k='sparse', dtype='f64', n=100,
         flags=False, offset=0),
    # a single-precision build of the same step
    dict(name='volume_f32', kind='volume', order=6, k='sparse', dtype='f32', n=200000,
         flags=False, offset=0),
    # dense stiffness matrices (bases without zero blocks)
    dict(name='volume_dense_f64', kind='volume', order=6, k='dense', dtype='f64', n=65536,
         flags=False, offset=0),
    dict(name='volume_dense_f32', kind='volume', order=6, k='dense', dtype='f32', n=100003,
         flags=False, offset=0),
    # a p-adaptive partition: orders 2..7 in one launch
    dict(name='mixed_orders', kind='mixed', n=500000),
    # the highest order of the repository's workloads
    dict(name='order7_f64', kind='volume', order=7, k='dense', dtype='f64', n=30000,
         flags=False, offset=0),
    # surface integral of an element's own faces
    dict(name='flux_local', kind='flux', side='local', n=131072, flags=False, offset=0),
    # neighbour contribution of one time cluster: the other clusters' elements are masked out
    dict(name='flux_neigh', kind='flux', side='neigh', n=40001, flags=True, offset=0),
    # time-derivative recursion, aligned arrays
    dict(name='derivative', kind='derivative', aligned=True, n=131071, flags=False, offset=0),
    # the same recursion on three arrays (bounding boxes from row 1), at an extra offset
    dict(name='derivative_na', kind='derivative', aligned=False, n=50000, flags=False, offset=64),
    # one batched product
    dict(name='gemm_f64', kind='gemm', dtype='f64', n=65536, flags=False, offset=0),
  ]


def _count(rng, hi, lo=1):
  """An element count, log-uniform over [lo, hi]."""
  return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
  kind = rng.choice(['volume', 'volume', 'volume', 'mixed', 'flux', 'flux', 'derivative',
                     'derivative', 'gemm'])
  if kind == 'mixed':
    return dict(kind='mixed', n=_count(rng, 500000, 100))
  case = dict(kind=kind, flags=rng.random() < 0.25,
              offset=rng.choice([0, 0, 0, 64, rng.randrange(1, 64)]))
  if kind == 'volume':
    case['order'] = rng.choice([6, 6, 6, 7])
    case['k'] = 'dense' if case['order'] == 7 else rng.choice(['sparse', 'dense'])
    case['dtype'] = 'f64' if case['order'] == 7 else rng.choice(['f64', 'f32'])
    case['n'] = _count(rng, 100000 if case['order'] == 7 else 262144)
  elif kind == 'flux':
    case['side'] = rng.choice(['local', 'neigh'])
    case['n'] = _count(rng, 262144)
  elif kind == 'derivative':
    case['aligned'] = rng.random() < 0.5
    case['n'] = _count(rng, 200000)
  else:
    case['dtype'] = rng.choice(['f64', 'f32'])
    case['n'] = _count(rng, 262144)
  return case


def _entry_name(case):
  if case['kind'] == 'volume':
    if case['order'] == 7:
      return 'ader7_f64_tuned'
    return f'ader_{"dense_" if case["k"] == "dense" else ""}{case["dtype"]}_tuned'
  if case['kind'] == 'flux':
    return f'flux_{case["side"]}_mod_f64_tuned'
  if case['kind'] == 'derivative':
    return 'deriv_f64_tuned' if case['aligned'] else 'deriv_na_f64_tuned'
  return f'gemm_{case["dtype"]}_tuned'


_LOADED = {}


def _load(name):
  """The launcher handle a program holds: loaded once per process."""
  if name not in _LOADED:
    _LOADED[name] = catalog.load_group('ader_mixed_f64') if name == 'mixed' else \
        catalog.load(name)
  return _LOADED[name]


# ---------------------------------------------------------------- operands

def _uniform(g, shape, lo, hi, dtype):
  return (torch.rand(shape, generator=g, device='cuda', dtype=torch.float64) * (hi - lo) + lo) \
      .to(dtype)


def _normal(g, shape, dtype):
  return torch.randn(shape, generator=g, device='cuda', dtype=torch.float64).to(dtype)


def _volume_arrays(g, n, b, sparse, dtype):
  """Degrees of freedom N(0, 1), star entries in [-2, 2] at the start of each element's 81-entry
  slot, stiffness values in [-1, 1]. Shapes are (elements, column, row)."""
  out = {'Q': _normal(g, (n, Q, b), dtype), 'Qp': torch.zeros(n, Q, b, device='cuda', dtype=dtype)}
  masks = W.k_patterns(b) if sparse else [None] * 3
  for d in range(3):
    s = torch.zeros(n, Q * Q, device='cuda', dtype=dtype)
    s[:, :STAR_NNZ] = _uniform(g, (n, STAR_NNZ), -2, 2, dtype)
    out[f'S{d + 1}'] = s
    nk = int(masks[d].sum()) if sparse else b * b
    out[f'K{d + 1}'] = _uniform(g, (nk,), -1, 1, dtype)
  return out


def _arrays(case, seed):
  g = torch.Generator(device='cuda')
  g.manual_seed(seed)
  n = case['n']
  f64 = torch.float64
  if case['kind'] == 'volume':
    return _volume_arrays(g, n, 56 if case['order'] == 6 else 84, case['k'] == 'sparse',
                          DTYPES[case['dtype']])
  if case['kind'] == 'mixed':
    counts = W.mixed_counts(n)
    return [_volume_arrays(g, c, b, False, f64) for b, c in zip(W.MIXED_BASES, counts)]
  if case['kind'] == 'flux':
    star = _uniform(g, (n, Q, Q), -2, 2, f64)
    if case['side'] == 'local':
      return {'i_surf': _normal(g, (n, Q, 64), f64), 'd_k': _normal(g, (n, Q, 64), f64),
              'a_plus': star, 'r_div_m': _uniform(g, (32, 64), -1, 1, f64),
              'f_mr_t': _uniform(g, (64, 32), -1, 1, f64)}
    return {'dofs': _normal(g, (n, Q, 64), f64), 'i_dofs': _normal(g, (n, Q, 64), f64),
            'a_plus': star, 'r_div_mat': _uniform(g, (21, 64), -1, 1, f64),
            'f_plus': _uniform(g, (21, 32), -1, 1, f64),
            'r_mat': _uniform(g, (56, 32), -1, 1, f64)}
  if case['kind'] == 'derivative':
    out = {'D': _normal(g, (n, Q, 48), f64)}
    for name in (['A'] if case['aligned'] else ['A1', 'A2', 'A3']):
      out[name] = _normal(g, (n, Q, 64), f64)
    for d, kc in enumerate((53, 54, 55)):
      out[f'S{d + 1}'] = _uniform(g, (n, Q, Q), -2, 2, f64)
      out[f'K{d + 1}'] = _uniform(g, (kc, 48), -1, 1, f64)
    return out
  dt = DTYPES[case['dtype']]
  return {'A': _uniform(g, (56, 56), -1, 1, dt), 'B': _uniform(g, (n, Q, 56), -1, 1, dt),
          'C': _uniform(g, (n, Q, 56), -1, 1, dt)}


def _active(case):
  """Skipped elements: every fourth one (None: all run)."""
  if not case.get('flags'):
    return None
  return (torch.arange(case['n'], device='cuda') % 4 != 3)


def _shift(name, t, case):
  """The operand's buffer: its entries after ``offset`` unused ones when it is per element."""
  off = case.get('offset', 0)
  if off == 0 or not _per_element(name, case):
    return t.reshape(-1)
  buf = torch.zeros(off + t.numel(), device=t.device, dtype=t.dtype)
  buf[off:] = t.reshape(-1)
  return buf


def _per_element(name, case):
  if name.startswith('K') or name in ('r_div_m', 'f_mr_t', 'r_div_mat', 'f_plus', 'r_mat'):
    return False
  return not (case['kind'] == 'gemm' and name == 'A')


def prepare(case, seed):
  arrays = _arrays(case, seed)
  if case['kind'] == 'mixed':
    group, _, _, kernel = _load('mixed')
    bufs = [{k: v.reshape(-1) for k, v in a.items()} for a in arrays]
    return {'case': case, 'group': group, 'kernel': kernel, 'bufs': bufs,
            'counts': W.mixed_counts(case['n'])}
  entry, kernel = _load(_entry_name(case))
  bufs = {k: _shift(k, v, case) for k, v in arrays.items()}
  act = _active(case)
  return {'case': case, 'kernel': kernel, 'bufs': bufs, 'n': case['n'],
          'flags': None if act is None else act.to(torch.int32),
          'offsets': {k: case['offset'] for k in bufs if _per_element(k, case)},
          'dest': _dest(case)}


def _dest(case):
  return {'volume': 'Qp', 'derivative': 'D', 'gemm': 'C',
          'flux': 'i_surf' if case.get('side') == 'local' else 'dofs'}[case['kind']]


def run(state):
  if state['case']['kind'] == 'mixed':
    group = state['group']
    lists = [launch_args(e.generator, b, n)
             for e, b, n in zip(group.members, state['bufs'], state['counts'])]
    state['kernel'](*group.grouped.member_args(lists))
    return [b['Qp'] for b in state['bufs']]
  launch(state['kernel'], state['bufs'], state['n'], state['offsets'], state['flags'])
  return state['bufs'][state['dest']]


# ---------------------------------------------------------------- compulsory work

def work(case):
  size = 4 if case.get('dtype') == 'f32' else 8
  n = case['n']
  if case['kind'] == 'mixed':
    total = {'bytes': 0, 'flops': 0}
    for b, c in zip(W.MIXED_BASES, W.mixed_counts(n)):
      w = _volume_work(b, c, 3 * b * b, 8)
      total = {k: total[k] + w[k] for k in total}
    return total
  act = n if not case['flags'] else n - n // 4
  if case['kind'] == 'volume':
    b = 56 if case['order'] == 6 else 84
    nk = int(sum(m.sum() for m in W.k_patterns(b))) if case['k'] == 'sparse' else 3 * b * b
    return _volume_work(b, act, nk, size)
  if case['kind'] == 'flux':
    shared = 21 * 56 * 2 + (21 * 21 if case['side'] == 'neigh' else 0)
    return {'bytes': act * (3 * 56 * Q + Q * Q) * 8 + shared * 8,
            'flops': 2 * act * (56 * Q * Q + shared * Q)}
  if case['kind'] == 'derivative':
    rows = 48 if case['aligned'] else 35
    reads = 55 * Q if case['aligned'] else (53 + 54 + 55) * Q
    return {'bytes': act * (reads + 3 * Q * Q + 2 * rows * Q) * 8 + rows * 162 * 8,
            'flops': 2 * act * (162 * Q * Q + rows * 162 * Q)}
  return {'bytes': act * 3 * 56 * Q * size + 56 * 56 * size, 'flops': 2 * act * 56 * 56 * Q}


def _volume_work(b, n, nk, size):
  return {'bytes': n * (2 * b * Q + 3 * STAR_NNZ) * size + nk * size,
          'flops': 2 * n * (3 * STAR_NNZ * b + nk * Q)}


# ---------------------------------------------------------------- values in 64 bits

def _volume_exact(a, b, sparse):
  n = a['Q'].shape[0]
  q = a['Q'].double()
  out = torch.zeros(n * Q, b, device='cuda', dtype=torch.float64)
  rc = W.star_entries()
  masks = np.random.default_rng(1).random((3, b, b)) < 0.4 if sparse else [None] * 3
  for d in range(3):
    t = torch.zeros(n, Q, b, device='cuda', dtype=torch.float64)
    for i, (r, c) in enumerate(rc):
      t[:, c] += q[:, r] * a[f'S{d + 1}'][:, i, None].double()
    k = a[f'K{d + 1}'].double()
    if sparse:
      dense = torch.zeros(b, b, device='cuda', dtype=torch.float64)
      rows, cols = np.nonzero(masks[d])
      dense[torch.from_numpy(rows).cuda(), torch.from_numpy(cols).cuda()] = k
      kt = dense.t().contiguous()
    else:
      kt = k.reshape(b, b)               # stored by columns: the reshape is its transpose
    out += t.reshape(n * Q, b) @ kt
  return out.reshape(n, Q, b)


def _times_star(x, star):
  """Rows of ``x`` (elements, column, row) times each element's 9 x 9 matrix."""
  out = torch.zeros(x.shape[0], Q, x.shape[2], device='cuda', dtype=torch.float64)
  for m in range(Q):
    out += star[:, :, m, None] * x[:, m, None, :]
  return out


def exact(case, seed):
  a = _arrays(case, seed)
  if case['kind'] == 'mixed':
    return [_volume_exact(x, b, False).reshape(-1) for x, b in zip(a, W.MIXED_BASES)]
  dest = _dest(case)
  old = a[dest].double()
  n = case['n']
  if case['kind'] == 'volume':
    new = _volume_exact(a, 56 if case['order'] == 6 else 84, case['k'] == 'sparse')
  elif case['kind'] == 'flux':
    if case['side'] == 'local':
      x, mats = a['d_k'], [(a['f_mr_t'], 56, 21), (a['r_div_m'], 21, 56)]
    else:
      x, mats = a['i_dofs'], [(a['r_mat'], 56, 21), (a['f_plus'], 21, 21), (a['r_div_mat'], 21, 56)]
    t = _times_star(x[:, :, :56], a['a_plus']).reshape(n * Q, 56)
    for m, kc, rows in mats:
      t = t @ m[:kc, :rows].contiguous()
    new = old.clone()
    new[:, :, :56] += t.reshape(n, Q, 56)
  elif case['kind'] == 'derivative':
    rows = 48 if case['aligned'] else 35
    new = old.clone()
    for d, kc in enumerate((53, 54, 55)):
      x = a['A' if case['aligned'] else f'A{d + 1}'][:, :, :kc]
      t = _times_star(x, a[f'S{d + 1}']).reshape(n * Q, kc)
      new[:, :, :rows] += (t @ a[f'K{d + 1}'][:, :rows].contiguous()).reshape(n, Q, rows)
  else:
    new = old + (a['B'].double().reshape(n * Q, 56) @ a['A'].double()).reshape(n, Q, 56)
  act = _active(case)
  if act is not None:
    new = torch.where(act[:, None, None], new, old)
  off = case['offset']
  if off:
    flat = torch.zeros(off + new.numel(), device='cuda', dtype=torch.float64)
    flat[off:] = new.reshape(-1)
    return flat
  return new.reshape(-1)
