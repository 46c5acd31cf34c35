"""The traversal in the form of launches that fill the device (visited bits in the
workspace behind the full-size table in LDS) and in that of smaller ones (visited
bits in LDS), on graphs large enough for both to be chosen: every size of the
lists, every row length with a kernel of its own, against the oracle.  And the
largest graphs whose bits fit LDS, beyond 64 KB of it."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from common import assert_same_search
from pilotann_amd import _lib, kernels

pytestmark = pytest.mark.gpu


def near_bits(n_storage, batch, beside, dp, ef_total):
    form = ctypes.c_int(-1)
    _lib.check(_lib.lib().pa_traverse_form(n_storage, batch, beside, dp, ef_total,
                                           ctypes.byref(form)), 'pa_traverse_form')
    return form.value


class RandomGraph:
    """Sampled nodes with random neighbours, ragged rows; entries of any node."""

    def __init__(self, n_nodes, n_rows, d, deg, n_query, n_init, seed):
        g = torch.Generator().manual_seed(seed)
        self.n_rows, self.deg = n_rows, deg
        self.nodelist = torch.randperm(n_nodes, generator=g)[:n_rows].sort().values
        self.mapping = torch.full((n_nodes,), -1, dtype=torch.long)
        self.mapping[self.nodelist] = torch.arange(n_rows)
        rows = self.nodelist[torch.randint(n_rows, (n_rows, deg), generator=g)]
        length = torch.randint(deg // 2, deg + 1, (n_rows, 1), generator=g)
        rows[torch.arange(deg).unsqueeze(0) >= length] = -1
        self.indices = rows.flatten().contiguous()
        held = torch.zeros(n_nodes, dtype=torch.long)
        held[self.nodelist] = deg
        self.indptr = torch.zeros(n_nodes + 1, dtype=torch.long)
        self.indptr[1:] = torch.cumsum(held, 0)
        self.x = torch.randn(n_nodes, d, generator=g)
        self.query = torch.randn(n_query, d, generator=g)
        self.entries = torch.randint(n_nodes, (n_query, n_init), generator=g)
        self.entries[:, 3] = -1

    def check(self, dp, ef, device, besides):
        """One search for each of ``besides``; returns the counters."""
        B, k = self.query.size(0), 4 * ef
        x = np.ascontiguousarray(self.x[:, :dp].numpy())
        query = np.ascontiguousarray(self.query[:, :dp].numpy())
        dist = np.stack([oracle.square_dist(query[b].copy(), x,
                                            self.entries[b].clamp(min=0).numpy().copy())
                         for b in range(B)])
        ref_I, ref_D = np.empty((B, k), np.int64), np.empty((B, k), np.float32)
        oracle.traverse_cpu(ref_I, ref_D, self.entries.numpy().copy(), dist.copy(),
                            self.indptr.numpy(), self.indices.numpy(), x, query, k)
        graph = kernels.prepare_graph(self.on(device, 'indptr'), self.on(device, 'indices'),
                                      self.on(device, 'mapping'), self.n_rows, self.deg)
        rows = kernels.PreparedRows(self.x[self.nodelist, :dp].contiguous().to(device))

        def at_that_distance(b, ids, dist):
            assert np.array_equal(oracle.square_dist(query[b].copy(), x, ids.copy()),
                                  np.full(len(ids), dist, np.float32))
        tallies = []
        for beside in besides:
            out_I = torch.full((B, 4, ef), -7, dtype=torch.long, device=device)
            out_D = torch.full((B, 4, ef), -7.0, device=device)
            counters = torch.zeros(5, dtype=torch.long, device=device)
            kernels.traverse_prepared(out_I, out_D, graph, rows,
                                      torch.from_numpy(query).to(device),
                                      self.entries.to(device), torch.from_numpy(dist).to(device),
                                      counters, beside=beside)
            assert_same_search(out_I.flatten(1).cpu(), out_D.flatten(1).cpu(), ref_I, ref_D,
                               worst_tie=at_that_distance)
            tallies.append(counters.tolist())
        return tallies

    def on(self, device, name):
        kept = self.__dict__.setdefault('_on', {})
        if name not in kept:
            kept[name] = getattr(self, name).to(device)
        return kept[name]


@pytest.fixture(scope='module')
def graph():
    return RandomGraph(130_000, 100_000, 128, 33, n_query=24, n_init=40, seed=7)


@pytest.mark.parametrize('dp', [32, 40, 64, 72, 128])
@pytest.mark.parametrize('ef', [3, 8, 12, 16, 24, 32, 48, 64, 96, 128, 256, 512])
def test_both_forms(ef, dp, graph, device):
    print('both forms', ef, dp, flush=True)
    B = graph.query.size(0)
    beside = next(b for b in range(0, 8192, 256)
                  if near_bits(graph.n_rows, B, b, dp, 4 * ef) == 0)
    assert near_bits(graph.n_rows, B, 0, dp, 4 * ef) == 1
    near, far = graph.check(dp, ef, device, [0, beside])
    assert near == far


def wavefronts(n_storage, batch, beside, dp, ef_total):
    form = ctypes.c_int(-1)
    _lib.check(_lib.lib().pa_traverse_wavefronts(n_storage, batch, beside, dp, ef_total,
                                                 ctypes.byref(form)), 'pa_traverse_wavefronts')
    return form.value


@pytest.mark.parametrize('dp', [32, 40, 64, 72, 128])
@pytest.mark.parametrize('ef', [3, 8, 12, 16, 24, 32, 48, 64, 96, 128, 256, 512])
def test_bits_in_lds_without_helpers(ef, dp, graph, device):
    """Launches too large for wavefronts that read ahead, whose bits are in LDS still."""
    print('no helpers', ef, dp, flush=True)
    B = graph.query.size(0)
    beside = next(b for b in range(0, 8192, 64)
                  if wavefronts(graph.n_rows, B, b, dp, 4 * ef) == 1)
    assert near_bits(graph.n_rows, B, beside, dp, 4 * ef) == 1
    few, many = graph.check(dp, ef, device, [0, beside])
    assert few == many


def slots(n_storage, batch, dp, ef_total):
    n = ctypes.c_int(-1)
    _lib.check(_lib.lib().pa_traverse_plan(n_storage, batch, dp, ef_total, ctypes.byref(n),
                                           None), 'pa_traverse_plan')
    return n.value


@pytest.fixture(scope='module')
def large_graph():
    """Rows of 128 floats beyond what is read in two passes when the device is full."""
    return RandomGraph(340_000, 330_000, 128, 17, n_query=8, n_init=40, seed=9)


@pytest.mark.parametrize('ef', [3, 8, 12, 16, 24, 32, 48, 64, 96, 128, 256, 512])
def test_rows_one_pass_at_a_time(ef, large_graph, graph, device):
    print('one pass at a time', ef, flush=True)
    many, few = 40_000, large_graph.query.size(0)
    if ef <= 128:       # more wavefronts fit than with two passes
        assert slots(330_000, many, 128, 4 * ef) > slots(100_000, many, 128, 4 * ef)
    assert near_bits(330_000, few, 1 << 40, 128, 4 * ef) == 0
    two, one = large_graph.check(128, ef, device, [0, 1 << 40])
    assert two == one
    # and where a little more than what two passes hold is on the device
    B = graph.query.size(0)
    assert near_bits(graph.n_rows, B, 3500 - B, 128, 4 * ef) == 0
    graph.check(128, ef, device, [3500 - B])


@pytest.mark.parametrize('n', [650_000, 1_140_000])
@pytest.mark.parametrize('ef', [4, 48, 256, 512])
def test_bits_beyond_64_kb(n, ef, device):
    print('bits beyond 64 KB', n, ef, flush=True)
    large = RandomGraph(n, n, 32, 9, n_query=6, n_init=33, seed=n)
    assert near_bits(n, 6, 0, 32, 4 * ef) == 1
    large.check(32, ef, device, [0])


def test_more_queries_than_run_at_once(graph, device):
    """A launch that fills the device several times over, wavefronts taking one
    query after the other: every copy of a query as the oracle has it."""
    print('more queries than run at once', flush=True)
    times, ef, dp = 260, 16, 64
    B = graph.query.size(0) * times
    assert near_bits(graph.n_rows, B, 0, dp, 4 * ef) == 0
    whole = RandomGraph.__new__(RandomGraph)
    whole.__dict__.update({k: v for k, v in graph.__dict__.items() if k != '_on'})
    whole.query = graph.query.repeat(times, 1)
    whole.entries = graph.entries.repeat(times, 1)
    whole.check(dp, ef, device, [0])
