"""The work this framework is used for, as cases to time.

Four kinds, each through the public entry points:

``search``  ``IndexStaged.search(refine='device')``: host queries in, host
            top-k out, all three stages on the GPU (``traversal`` exact or
            wide), from one query (an online lookup) to a bulk job.
``host``    ``IndexStaged.search`` with its defaults: device candidates,
            refine on the host's cores, chunk by chunk.
``stage``   the GPU search stage alone, as the operator API offers it:
            ``IndexEntry.search`` and ``kernels.traverse_cuda`` on device
            tensors, into the caller's own output buffers.
``build``   ``utils.graph_init``: one proximity graph of an index.

An index is what a serving program keeps for millions of queries: it depends on
the case's sizes only and is kept here between preparations.  The queries (and
the rows of a build) come from the seed.
"""
import contextlib
import io
from collections import OrderedDict

import torch

from pilotann_amd import IndexStaged, kernels, utils

DEVICE = 'cuda:0'


# ---- the cases -------------------------------------------------------------------

def _index(n, d, dp, graph, entry, ratio=0.25, centers=1024, sigma=1.0, unit=True):
    return dict(n=n, d=d, dp=dp, graph=graph, entry=entry, ratio=ratio,
                centers=centers, sigma=sigma, unit=unit)


# The benchmark's index sizes: the plumbing case, the 96-dimensional one, the
# headline (unit-norm 768-dimensional embeddings) and the same with half of the
# nodes sampled.
_SMALL = _index(100_000, 96, 32, 'nsg32', 'random32', centers=64, sigma=0.3, unit=False)
_FLAT = _index(1_000_000, 96, 64, 'nsw32', 'router32x32', centers=256, unit=False)
_HEAD = _index(1_000_000, 768, 128, 'nsw64', 'router64x64')
_HALF = _index(1_000_000, 768, 128, 'nsw64', 'router64x64', ratio=0.5)


def listed():
    def search(name, index, batch, ef, k, traversal='exact'):
        return dict(index, name=name, kind='search', batch=batch, ef=ef, k=k,
                    traversal=traversal)

    def host(name, index, batch, ef, k, chunk):
        return dict(index, name=name, kind='host', batch=batch, ef=ef, k=k, chunk=chunk)

    def stage(name, index, batch, ef):
        return dict(index, name=name, kind='stage', batch=batch, ef=ef)

    def build(name, n, d, graph, sigma, unit):
        return dict(name=name, kind='build', n=n, d=d, graph=graph,
                    centers=max(16, n // 1000), sigma=sigma, unit=unit)

    return [
        # graphs of a small and of a medium set: the offline side, dominated
        # by launches and by the neighbour table respectively
        build('build_20k_d96', 20_011, 96, 'nsw32', 1.0, False),
        build('build_120k_d768', 120_000, 768, 'nsg48', 1.0, True),
        # the plumbing configuration with the index's defaults (host refine,
        # chunks of 128), as a first-time user runs it
        host('host_1k_100k_d96', _SMALL, 1024, 64, 10, 128),
        # the middle configuration at its recall-0.90 point: short rows,
        # few new rows per step; bulk stage, whole search in the wide mode
        stage('stage_10k_1m_d96', _FLAT, 10_000, 64),
        search('wide_3001_1m_d96', _FLAT, 3001, 96, 10, 'wide'),
        # one user's lookup; a small ragged service batch; the batch the
        # reference's own tables are quoted for; the headline bulk batch
        search('search_1_1m_d768', _HEAD, 1, 32, 10),
        search('search_37_1m_d768', _HEAD, 37, 48, 10),
        search('search_1k_1m_d768', _HEAD, 1024, 64, 10),
        search('search_10k_1m_d768', _HEAD, 10_000, 32, 10),
        # the headline metric: router and traversal, inputs resident
        stage('stage_10k_1m_d768', _HEAD, 10_000, 32),
        # the reference's split (refine on the host) at the headline sizes
        host('host_2k_1m_d768', _HEAD, 2000, 32, 10, 500),
        # long candidate lists: top-100 with half of the nodes on the device
        search('top100_10k_1m_d768', _HALF, 10_000, 256, 100),
    ]


def _between(rng, lo, hi):
    """A whole number, its logarithm uniform over [lo, hi]."""
    return min(hi, max(lo, round(lo * (hi / lo) ** rng.random())))


def draw(rng):
    kind = rng.choices(['search', 'stage', 'host', 'build'], [50, 25, 12, 13])[0]
    d = 8 * rng.choice([8, 12, 12, 16, 25, 32, 48, 64, 96, 96])
    unit = d > 128
    if kind == 'build':
        n = _between(rng, 5000, max(20_000, min(250_000, 90_000_000 // d)))
        return dict(kind=kind, n=n, d=d, centers=max(16, n // 1000), sigma=1.0, unit=unit,
                    graph=rng.choice(['nsw32', 'nsw48', 'nsw64', 'nsg32', 'nsg48']))
    n = _between(rng, 20_000, max(100_000, min(1_000_000, 200_000_000 // d)))
    dps = [p for p in (32, 40, 64, 96, 128) if p <= d]
    case = _index(
        n, d, rng.choice(dps), rng.choice(['nsw32', 'nsw48', 'nsw64', 'nsg32', 'nsg48']),
        # a router of R x L entries draws 1024 L different nodes
        rng.choice(['random16', 'random32'] if n < 40_000
                   else ['random32', 'router32x32'] if n < 100_000
                   else ['random32', 'router32x32', 'router64x64', 'router64x64']),
        ratio=round(rng.uniform(0.15, 0.5), 3), centers=max(16, n // 1000), unit=unit)
    ef = _between(rng, 8, 128) if rng.random() < 0.85 else _between(rng, 129, 400)
    case.update(kind=kind, ef=ef)
    if kind == 'stage':
        case.update(batch=_between(rng, 1, 12_000))
        return case
    case.update(k=min(ef, _between(rng, 1, 100)))
    if kind == 'search':
        case.update(batch=_between(rng, 1, 12_000),
                    traversal='wide' if rng.random() < 0.2 else 'exact')
    else:
        chunk = rng.choice([64, 128, 250])
        case.update(ef=min(ef, 128), k=min(case['k'], 128), chunk=chunk,
                    batch=chunk * _between(rng, 1, 2000 // chunk))
    return case


# ---- inputs ----------------------------------------------------------------------

_indexes = OrderedDict()
_INDEX_KEYS = ('n', 'd', 'dp', 'graph', 'entry', 'ratio', 'centers', 'sigma', 'unit')


def _data(case, n, seed, center_seed):
    return utils.gaussian_mixture(
        n, case['d'], case['centers'], case['sigma'], seed=seed, normalize=case['unit'],
        device=DEVICE, center_seed=center_seed, device_rng=True)


def _index_for(case, refine_on_device):
    """The built index of the case's sizes, on the device."""
    key = tuple(case[name] for name in _INDEX_KEYS)
    index = _indexes.get(key)
    if index is None:
        while len(_indexes) > 1:
            _indexes.popitem(last=False)
        index = IndexStaged(
            d_model=case['d'], d_principle=case['dp'], sample_ratio=case['ratio'],
            graph_method=case['graph'], entry_method=case['entry'], seed=11,
            build_device=DEVICE)
        with contextlib.redirect_stdout(io.StringIO()):
            index.train(_data(case, case['n'], 101, 101))
        index.to(DEVICE)
        torch.cuda.empty_cache()
        _indexes[key] = index
    _indexes.move_to_end(key)
    if refine_on_device and index.storage_full_cuda is None:
        index.stage_refine()
    return index


def prepare(case, seed):
    if case['kind'] == 'build':
        return dict(case=case, rows=_data(case, case['n'], seed, seed))
    index = _index_for(case, case['kind'] == 'search')
    query = _data(case, case['batch'], 1_000_003 + seed, 101)
    state = dict(case=case, index=index)
    if case['kind'] == 'stage':
        rotated = kernels.rotate(query, index.VT_cuda)
        state['query'] = rotated[:, :case['dp']].contiguous()
        shape = (case['batch'], 4, case['ef'])
        state['out_I'] = torch.empty(shape, dtype=torch.long, device=DEVICE)
        state['out_D'] = torch.empty(shape, dtype=torch.float, device=DEVICE)
    else:
        state['query'] = query.cpu()
    return state


# ---- one pass --------------------------------------------------------------------

def run(state):
    case = state['case']
    kind = case['kind']
    if kind == 'build':
        graph_type = case['graph'][:3]
        return utils.graph_init(state['rows'], graph_type, int(case['graph'][3:]))
    index = state['index']
    if kind == 'search':
        return index.search(state['query'], k=case['k'], ef_search=case['ef'],
                            refine='device', traversal=case['traversal'])
    if kind == 'host':
        return index.search(state['query'], k=case['k'], ef_search=case['ef'],
                            chunk_size=case['chunk'])
    EP_I, EP_D = index.entry.search(state['query'])
    kernels.traverse_cuda(
        state['out_I'], state['out_D'], index.subgraph_cuda.indptr,
        index.subgraph_cuda.indices, index.mapping_cuda, index.storage_cuda,
        state['query'], EP_I.contiguous(), EP_D.contiguous(), index.n_neighbors)
    return state['out_I'], state['out_D']


# ---- what a pass cannot do without -------------------------------------------------

def work(case):
    n, d, deg = case['n'], case['d'], int(case['graph'][3:])
    if case['kind'] == 'build':
        # the products of the neighbour table (two thirds of all pairs: a node
        # ranks what comes before it) and of the pruning (256 candidates with
        # each other); the rows read, the graph written
        return dict(bytes=4 * n * d + 8 * n * deg,
                    flops=2 * d * (2 / 3 * n * n + 240 * 240 / 2 * n))
    # Per query of the subgraph search, by the search's own counters on the
    # listed indexes: four expansions per unit of ef, at most 1024, and per
    # expansion a share of the degree in rows not seen before (smaller where
    # the rows are short, and as a search gets long).
    dp, ef, batch = case['dp'], case['ef'], case['batch']
    fresh = (0.31 if d > 128 else 0.17) * deg * (0.7 if ef > 160 else 1.0)
    expand = min(1024, 4.0 * ef + 6)
    entries = case['entry'].removeprefix('random').removeprefix('router').split('x')
    n_init = int(entries[-1])
    per_query = (4 * dp + 12 * n_init + expand * 4 * deg
                 + expand * fresh * (4 + 4 * dp) + 4 * ef * 12)
    flops = 3 * dp * (expand * fresh + n_init)
    if case['kind'] != 'stage':
        # the refine: the candidates' remaining coordinates, then a search of
        # the full graph in full dimension, which runs out of new rows at
        # about a thousand of them
        expand = min(1024, 0.95 * ef + 10)
        rows = min(18 * expand, 1000)
        per_query += 4 * d + 4 * ef * 4 * (d - dp) + expand * 4 * deg + rows * (4 + 4 * d) \
            + 12 * case['k']
        flops += 2 * d * d + 3 * (d - dp) * 4 * ef + 3 * d * rows
    return dict(bytes=batch * per_query, flops=batch * flops)


def tolerance(case):
    if case['kind'] == 'build':
        # ids.  Distances are ranked in float32 and compared in the pruning to
        # about 22 bits: a row with a near-tie can come out differently.
        return dict(rel=1e-6, differ=2e-3)
    if case['kind'] == 'stage':
        # a distance is one fixed sum, and the search is the host's step for
        # step: the same numbers, whatever computes them
        return 'exact'
    # The rotation is a float32 product in some order (a host product's sums in
    # place of the device's: distances 9e-8 apart, ids the same on 20 000
    # places).  Where a search turns at a tie within that rounding, a row can
    # end with another id.
    return dict(rel=2e-5, max=1e-2, differ=1e-3)
