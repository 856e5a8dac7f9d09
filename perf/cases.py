"""Performance cases of the bond-percolation path, through its public entry points.

A case names its kind and sizes.  The kinds:

* ``pipeline``: a batch of runs of one lattice to the exact microcanonical
  sums (``Pipeline``): permutations (Philox, or numpy's RandomState bit for
  bit), sweep, chunk states, sums;
* ``traces``: the per-run arrays of ``bond_microcanonical_statistics_batch``
  as they are on the device (``BondEngine.sweep`` and ``traces``);
* ``drop_in``: ``hpc.bond_microcanonical_statistics_batch`` on a networkx
  graph, the call a program written for the reference makes;
* ``per_run``: ``hpc.bond_canonical_averages_batch`` and
  ``finalize_canonical_averages``, the canonical statistics of every run;
* ``canonical``: the binomial convolution of microcanonical columns at many
  p (``canonical_fused``, or a kept ``FusedPlan``);
* ``finite_size``: ``FiniteSizeBatch``, many lattice sizes as one HIP graph.
"""
import math

import numpy as np
import torch

from pypercolate_amd import _engine, _graph, hpc, percolate
from pypercolate_amd.batch import FiniteSizeBatch

ALPHA = 0.31731050786291415   # one standard deviation
COLUMN_BYTES = 8


def listed():
    return [
        # a small study's size: 40 bit-exact runs of a small lattice
        {'name': 'pipeline_L16_R40_exact', 'kind': 'pipeline', 'length': 16,
         'runs': 40, 'draw': 'randomstate'},
        # the benchmark's headline batch
        {'name': 'pipeline_L128_R10000', 'kind': 'pipeline', 'length': 128,
         'runs': 10000, 'draw': 'philox'},
        # the same lattice with the reference's own permutations
        {'name': 'pipeline_L128_R4000_exact', 'kind': 'pipeline', 'length': 128,
         'runs': 4000, 'draw': 'randomstate'},
        # an odd lattice whose union-find state no longer fits 16 bits
        {'name': 'pipeline_L181_R600', 'kind': 'pipeline', 'length': 181,
         'runs': 600, 'draw': 'philox'},
        # the reference's permutations on a larger lattice
        {'name': 'pipeline_L256_R200_exact', 'kind': 'pipeline', 'length': 256,
         'runs': 200, 'draw': 'randomstate'},
        # the large-lattice configuration: state in HBM, 64-bit records
        {'name': 'pipeline_L1024_R1000', 'kind': 'pipeline', 'length': 1024,
         'runs': 1000, 'draw': 'philox'},
        # per-run traces of a batch (the per-run arrays a jug task keeps)
        {'name': 'traces_L100_R500', 'kind': 'traces', 'length': 100, 'runs': 500},
        # the unchanged call of a program written for the reference
        {'name': 'drop_in_L32_R40', 'kind': 'drop_in', 'length': 32, 'runs': 40},
        # canonical statistics of every run, mapped and reduced
        {'name': 'per_run_L128_R10000', 'kind': 'per_run', 'length': 128,
         'runs': 10000, 'num_p': 1000, 'p_lo': 0.45, 'p_hi': 0.55},
        # the canonical step of percolate.statistics: all 21 columns
        {'name': 'canonical_L128_21', 'kind': 'canonical', 'length': 128,
         'columns': 21, 'num_p': 201, 'p_lo': 0.4, 'p_hi': 0.6, 'plan': False},
        # the canonical comparison's size: a kept plan on a large lattice
        {'name': 'canonical_L1024_14', 'kind': 'canonical', 'length': 1024,
         'columns': 14, 'num_p': 4096, 'p_lo': 0.3, 'p_hi': 0.7, 'plan': True},
        # the finite-size study: about 2^26 sites' worth of runs per lattice
        {'name': 'finite_size_16_512', 'kind': 'finite_size', 'low': 16, 'count': 6,
         'num_p': 101, 'bonds': 800000000},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _runs(rng, length, lo, hi, cap):
    """Runs so that runs x bonds is spread over lo..hi, at most cap."""
    edges = 2 * length * (length - 1)
    return max(1, min(cap, _log_uniform(rng, lo, hi) // edges))


def draw(rng):
    kind = rng.choice(['pipeline', 'pipeline', 'pipeline', 'exact', 'exact', 'traces',
                       'drop_in', 'per_run', 'canonical', 'canonical', 'finite_size'])
    if kind == 'pipeline':
        length = _log_uniform(rng, 8, 700)
        return {'kind': kind, 'length': length, 'draw': 'philox',
                'runs': _runs(rng, length, 1e5, 4e8, 20000)}
    if kind == 'exact':
        # numpy's draw is a sequential chain of one step per bond and run
        length = _log_uniform(rng, 8, 400)
        return {'kind': 'pipeline', 'length': length, 'draw': 'randomstate',
                'runs': _runs(rng, length, 2e4, 4e7 if length > 128 else 2e8, 10000)}
    if kind == 'traces':
        length = _log_uniform(rng, 8, 500)
        return {'kind': kind, 'length': length,
                'runs': _runs(rng, length, 1e4, 3e7, 10000)}
    if kind == 'drop_in':
        return {'kind': kind, 'length': _log_uniform(rng, 4, 64),
                'runs': _log_uniform(rng, 1, 100)}
    if kind == 'per_run':
        length = _log_uniform(rng, 16, 160)
        centre, half = rng.uniform(0.3, 0.7), rng.uniform(0.01, 0.1)
        return {'kind': kind, 'length': length, 'runs': _runs(rng, length, 2e5, 1e8, 8000),
                'num_p': _log_uniform(rng, 10, 500),
                'p_lo': round(centre - half, 6), 'p_hi': round(centre + half, 6)}
    if kind == 'canonical':
        length = _log_uniform(rng, 16, 1024)
        p_lo = rng.uniform(0.0, 0.45)
        return {'kind': kind, 'length': length, 'columns': rng.choice([7, 14, 18, 21]),
                'num_p': _log_uniform(rng, 1, 2000), 'p_lo': round(p_lo, 6),
                'p_hi': round(rng.uniform(p_lo + 0.02, 1.0), 6),
                'plan': rng.random() < 0.5}
    low, count = rng.choice([8, 12, 16]), rng.choice([2, 3, 4, 5])
    return {'kind': kind, 'low': low, 'count': count, 'num_p': _log_uniform(rng, 11, 200),
            'bonds': _log_uniform(rng, 1e6, 3e8)}


# -- inputs -----------------------------------------------------------------

def _edges(case):
    return 2 * case['length'] * (case['length'] - 1)


def _ps(case, seed):
    """The sorted p grid of the case, moved by a seed-dependent fraction of
    its spacing."""
    lo, hi, n = case['p_lo'], case['p_hi'], case['num_p']
    shift = np.random.RandomState(seed % (1 << 32)).uniform(0.0, 1.0)
    return lo + (hi - lo) * (np.arange(n) + shift) / n


def _columns(case, seed):
    """(S, C) float64 columns like microcanonical averages: largest cluster,
    spanning probability, moments up to the fourth (growing like powers of
    the cluster size below the threshold and falling above), with the
    run-to-run noise of an average, positive, on the GPU."""
    m, c = _edges(case), case['columns']
    g = torch.Generator(device='cuda')
    g.manual_seed(seed)
    s = torch.linspace(0.0, 1.0, m + 1, dtype=torch.float64, device='cuda')
    sites = float(case['length'] ** 2)
    cols = []
    for j in range(c):
        power = j % 7
        if power == 1:            # a probability
            col = torch.sigmoid((s - 0.5) * 60.0)
        elif power == 0:          # the largest cluster
            col = 1.0 + sites * torch.sigmoid((s - 0.5) * 40.0)
        else:                     # a moment of the other clusters
            k = power - 2
            peak = torch.exp(-0.5 * ((s - 0.48) * 12.0) ** 2)
            col = sites * (1.0 - s) + sites ** (1 + 0.45 * k) * peak
        noise = torch.rand(m + 1, generator=g, dtype=torch.float64, device='cuda')
        cols.append(col * (0.95 + 0.1 * noise))
    return torch.stack(cols, dim=1).contiguous()


def _lengths(case):
    return [case['low'] << i for i in range(case['count'])]


def _finite_runs(case):
    lengths = _lengths(case)
    return [max(1, case['bonds'] // (len(lengths) * 2 * v * (v - 1))) for v in lengths]


def _seeds(case, seed):
    return np.random.RandomState(seed % (1 << 32)).randint(
        1 << 32, size=case['runs'], dtype=np.uint64)


def prepare(case, seed):
    kind = case['kind']
    state = {'case': case}
    if kind == 'pipeline':
        engine = _engine.BondEngine(_graph.square_lattice(case['length']))
        seeds = _seeds(case, seed) if case['draw'] == 'randomstate' else None
        state['pipeline'] = _engine.Pipeline(engine, case['runs'], seed=seed, seeds=seeds)
    elif kind == 'traces':
        state['engine'] = _engine.BondEngine(_graph.square_lattice(case['length']))
        state['perm'] = state['engine'].device_permutations(seed, case['runs'])
    elif kind == 'drop_in':
        state['graph'] = percolate.percolation_graph(
            percolate.spanning_2d_grid(case['length']))
        state['seeds'] = [int(s) for s in _seeds(case, seed)]
    elif kind == 'per_run':
        state['graph'] = _graph.square_lattice(case['length'])
        state['ps'] = _ps(case, seed)
        state['seed'] = seed
    elif kind == 'canonical':
        state['x'] = _columns(case, seed)
        state['ps'] = _ps(case, seed)
        if case['plan']:
            state['plan'] = _engine.FusedPlan(state['x'], state['ps'])
    else:
        batch = FiniteSizeBatch(_lengths(case), _finite_runs(case), seed=seed,
                                ps=np.linspace(0.3, 0.7, case['num_p']), tune=False)
        batch.capture()
        state['batch'] = batch
    return state


def run(state):
    case = state['case']
    kind = case['kind']
    if kind == 'pipeline':
        sum1, sum2 = state['pipeline'].run()
        return {'sum1': sum1, 'sum2': sum2}
    if kind == 'traces':
        engine = state['engine']
        largest, spanning, moments = engine.traces(engine.sweep(state['perm']))
        return {'max': largest, 'spanning': spanning, 'moments': moments}
    if kind == 'drop_in':
        rows = hpc.bond_microcanonical_statistics_batch(seeds=state['seeds'],
                                                        **state['graph'])
        return {name: rows[name] for name in rows.dtype.names}
    if kind == 'per_run':
        graph = state['graph']
        averages = hpc.bond_canonical_averages_batch(
            None, graph.num_nodes, graph.num_edges, state['ps'], spanning_sides=[0, 1],
            num_runs=case['runs'], philox_seed=state['seed'], graph_arrays=graph)
        rows = hpc.finalize_canonical_averages(graph.num_nodes, state['ps'], averages,
                                               ALPHA)
        return {name: rows[name] for name in rows.dtype.names}
    if kind == 'canonical':
        if case['plan']:
            return state['plan'].run()
        return _engine.canonical_fused(state['x'], state['ps'])
    state['batch'].run()
    return {str(p.length): {'sum1': p.sum1, 'sum2': p.sum2, 'mean': p.mean,
                            'canonical': p.plan.out} for p in state['batch'].plans}


# -- what a pass cannot do without --------------------------------------------

def _sums_bytes(edges):
    return 7 * (edges + 1) * 5 * 8


def _window(edges, p):
    return min(edges + 1.0, 24.0 * math.sqrt(edges * p * (1.0 - p)) + 97.0)


def work(case):
    """Bytes: inputs read once and outputs written once (permutations, the
    union-find state and merge records need not leave the chip).
    Operations: about ten per bond addition (the draw, two finds, a merge
    and its moments), two per element of a convolution window."""
    kind = case['kind']
    if kind == 'finite_size':
        total = {'bytes': 0.0, 'flops': 0.0}
        for length, runs in zip(_lengths(case), _finite_runs(case)):
            m = 2 * length * (length - 1)
            total['bytes'] += 8.0 * m + _sums_bytes(m) + 7 * 8 * (m + 1 + case['num_p'])
            total['flops'] += 10.0 * runs * m + 14.0 * sum(
                _window(m, p) for p in np.linspace(0.3, 0.7, case['num_p']))
        return total
    m = _edges(case)
    if kind == 'canonical':
        ps = _ps(case, 0)
        return {'bytes': COLUMN_BYTES * case['columns'] * (m + 1.0 + ps.size),
                'flops': 2.0 * case['columns'] * sum(_window(m, p) for p in ps)}
    additions = 10.0 * case['runs'] * m
    if kind == 'pipeline':
        return {'bytes': 8.0 * m + _sums_bytes(m), 'flops': additions}
    if kind == 'traces':
        return {'bytes': 8.0 * m + case['runs'] * (4.0 * m + 45.0 * (m + 1)),
                'flops': additions}
    if kind == 'drop_in':
        return {'bytes': 8.0 * m + case['runs'] * 53.0 * (m + 1), 'flops': additions}
    ps = _ps(case, 0)
    return {'bytes': 8.0 * m + 250.0 * ps.size,
            'flops': additions + 14.0 * case['runs'] * sum(_window(m, p) for p in ps)}


# -- 64-bit values of what is computed in floating point ------------------------

def _weights(n, p, k):
    """Normalised binomial weights over consecutive k, from the exact ratio
    of neighbours in extended precision."""
    if p <= 0.0 or p >= 1.0:
        return (k == (0 if p <= 0.0 else n)).astype(np.float64)
    ld = np.longdouble
    kk = k[1:].astype(ld)
    ratio = (ld(n) - kk + 1) / kk * (ld(p) / (1 - ld(p)))
    # from the largest weight outwards, so that no product overflows
    top = min(max(int(math.floor((n + 1) * p)) - int(k[0]), 0), k.size - 1)
    up = np.cumprod(ratio[top:])
    down = np.cumprod(1 / ratio[:top][::-1])[::-1]
    w = np.concatenate([down, np.ones(1, dtype=ld), up])
    return (w / w.sum()).astype(np.float64)


def exact(case, seed):
    if case['kind'] != 'canonical':
        # whole numbers, or averages over more runs than plain Python sweeps
        return None
    x = _columns(case, seed).cpu().numpy()
    n = x.shape[0] - 1
    ps = _ps(case, seed)
    out = np.empty((ps.size, x.shape[1]))
    for i, p in enumerate(ps):
        half = 13.0 * math.sqrt(n * p * (1.0 - p)) + 64.0
        k = np.arange(max(0, int(n * p - half)), min(n, int(n * p + half) + 1) + 1)
        out[i] = _weights(n, p, k) @ x[k[0]:k[-1] + 1]
    return out
