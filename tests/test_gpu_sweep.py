"""GPU parity of the sweep pipeline (permute -> sweep -> chunk_scan ->
microcanonical sums / traces) against the oracle and the golden fixtures.
Integer results must be bit-exact."""
import numpy as np
import pytest

from oracle import oracle
from pypercolate_amd import _graph
from pypercolate_amd._engine import BondEngine, host_sums
from tests.helpers import grid_3x3_graph, spanning_2d_grid

pytestmark = pytest.mark.gpu


def _engine_for(nx_graph, spanning):
    from pypercolate_amd.percolate import percolation_graph
    pg = percolation_graph(nx_graph, spanning_cluster=spanning)
    ga = _graph.from_percolation_graph(**pg)
    return BondEngine(ga), oracle.percolation_graph_arrays(nx_graph, spanning)


def _check_traces(eng, res, expect, runs=None):
    mx, sp, mom = eng.host_traces(res)
    rows = slice(None) if runs is None else runs
    np.testing.assert_array_equal(mx, expect['max_cluster_size'][rows])
    np.testing.assert_array_equal(sp, expect['has_spanning_cluster'][rows])
    np.testing.assert_array_equal(mom, expect['moments'][rows])


def _check_sums(eng, res, expect):
    s1, s2 = host_sums(*eng.microcanonical_sums(res))
    o1, o2 = oracle.microcanonical_sums(expect)
    assert (s1 == o1).all(), 'sum of x differs'
    assert (s2 == o2).all(), 'sum of x**2 differs'


@pytest.mark.parametrize('spanning', [True, False])
def test_kat_3x3(gpu, golden, spanning):
    kat = golden('kat_3x3.json')
    eng, g = _engine_for(grid_3x3_graph(spanning, kat), spanning)
    perm = np.array([kat['permutation']])
    res = eng.sweep(eng.upload_permutations(perm))
    mx, sp, mom = eng.host_traces(res)
    assert mx[0].tolist() == kat['max_cluster_size']
    assert mom[0].tolist() == kat['moments']
    if spanning:
        assert sp[0].tolist() == kat['has_spanning_cluster']


@pytest.mark.parametrize('length', [2, 3, 4, 6])
def test_brute_force_fixtures(gpu, golden, length):
    bf = golden('brute_force.npz')
    eng, g = _engine_for(spanning_2d_grid(length), True)
    res = eng.sweep(eng.upload_permutations(bf['L{}_perm'.format(length)]))
    mx, sp, mom = eng.host_traces(res)
    np.testing.assert_array_equal(mx, bf['L{}_max'.format(length)])
    np.testing.assert_array_equal(mom, bf['L{}_moments'.format(length)])
    np.testing.assert_array_equal(sp, bf['L{}_spanning'.format(length)])


@pytest.mark.parametrize('spanning', [True, False])
def test_config_L16_40_runs(gpu, spanning):
    """spanning_2d_grid(16), 40 runs with RandomState(r) permutations."""
    eng, g = _engine_for(spanning_2d_grid(16), spanning)
    perms = oracle.randomstate_permutations(range(40), g['num_edges'])
    expect = oracle.bond_runs(g, perms)
    res = eng.sweep(eng.upload_permutations(perms))
    _check_traces(eng, res, expect)
    _check_sums(eng, res, expect)


def test_closed_form_lattice_equals_networkx(gpu):
    eng_nx, g = _engine_for(spanning_2d_grid(12), True)
    eng_cf = BondEngine(_graph.square_lattice(12))
    perms = oracle.randomstate_permutations(range(8), g['num_edges'])
    a = eng_nx.host_traces(eng_nx.sweep(eng_nx.upload_permutations(perms)))
    b = eng_cf.host_traces(eng_cf.sweep(eng_cf.upload_permutations(perms)))
    for x, y in zip(a, b):
        np.testing.assert_array_equal(x, y)


def test_random_graph_no_spanning(gpu):
    import networkx as nx
    gnx = nx.gnm_random_graph(300, 900, seed=11)
    eng, g = _engine_for(gnx, False)
    perms = oracle.randomstate_permutations(range(70), g['num_edges'])
    expect = oracle.bond_runs(g, perms)
    res = eng.sweep(eng.upload_permutations(perms))
    _check_traces(eng, res, expect)
    _check_sums(eng, res, expect)


@pytest.mark.parametrize('nodes,edges', [(6000, 18000), (20000, 30000)])
def test_random_graph_two_wavefronts(gpu, nodes, edges):
    """Random graphs past the two-wavefront threshold (4096 nodes), with the
    state in LDS and in HBM: traces and sums equal the oracle's."""
    import networkx as nx
    gnx = nx.gnm_random_graph(nodes, edges, seed=nodes)
    eng, g = _engine_for(gnx, False)
    perms = oracle.randomstate_permutations(range(24), g['num_edges'])
    expect = oracle.bond_runs(g, perms)
    res = eng.sweep(eng.upload_permutations(perms))
    _check_traces(eng, res, expect)
    _check_sums(eng, res, expect)


def test_L128_64_runs(gpu):
    """The L = 128 lattice (N = 16384, M = 32512), LDS state at its limit."""
    eng = BondEngine(_graph.square_lattice(128))
    g = oracle.percolation_graph_arrays(spanning_2d_grid(128), True)
    perms = oracle.randomstate_permutations(range(64), g['num_edges'])
    expect = oracle.bond_runs(g, perms)
    res = eng.sweep(eng.upload_permutations(perms))
    _check_sums(eng, res, expect)
    _check_traces(eng, res, expect)


@pytest.mark.parametrize('length', [130, 257])
def test_global_state(gpu, length):
    """N > 16384 keeps the union-find in HBM; N > 65536 uses 64-bit records."""
    eng = BondEngine(_graph.square_lattice(length))
    g = oracle.percolation_graph_arrays(spanning_2d_grid(length), True)
    perms = oracle.randomstate_permutations(range(6), g['num_edges'])
    expect = oracle.bond_runs(g, perms)
    res = eng.sweep(eng.upload_permutations(perms))
    _check_traces(eng, res, expect)
    _check_sums(eng, res, expect)


@pytest.mark.parametrize('M', [1, 2, 12, 33, 64, 65, 480, 4096, 4097, 32512,
                               32768, 32769, 65536, 65537, 130560, 2095104])
def test_device_permutation_matches_oracle(gpu, M):
    """pc_permute_philox equals the oracle's restatement of the bucket
    shuffle bit for bit: the whole run as one bucket in the 2-wave (M <=
    4096) and the 8-wave group kernel (up to 32768: the L = 128 lattice),
    one sub-bucket or several, then several buckets through count, scan and
    scatter (from 32769 edges; several chunks of those passes at the
    L = 256 and L = 1024 lattices; the count and scatter blocks of 11 runs
    span two groups of eight runs, the second padded)."""
    eng = BondEngine(_graph.GraphArrays(M + 1, np.stack(
        [np.arange(M), np.arange(1, M + 1)], axis=1)))
    runs = 2 if M >= 1000000 else (11 if M > 32768 else 3)
    d = eng.device_permutations(seed=0x1234567890AB, num_runs=runs, first_run=5)
    got = d.cpu().numpy()
    want = oracle.bucket_permutations(0x1234567890AB, 5, runs, M)
    for r in range(runs):
        np.testing.assert_array_equal(got[r], want[r], err_msg='run {}'.format(r))


def test_device_permutation_L128_is_permutation(gpu):
    eng = BondEngine(_graph.square_lattice(128))
    d = eng.device_permutations(seed=1234, num_runs=32)
    srt = d.sort(dim=1).values.cpu().numpy()
    np.testing.assert_array_equal(srt, np.broadcast_to(np.arange(eng.M), srt.shape))


def test_full_size_properties(gpu):
    """L = 128, 10^4 runs from device permutations: size-independent checks
    of the exact sums (end state, identities between columns)."""
    eng = BondEngine(_graph.square_lattice(128))
    R = 10000
    res = eng.sweep(eng.device_permutations(seed=1234, num_runs=R))
    s1, s2 = host_sums(*eng.microcanonical_sums(res))
    N, M = eng.N, eng.M
    # step 0 and step M
    assert s1[0, 0] == R and s1[0, M] == R * N
    assert s1[1, 0] == 0 and s1[1, M] == R
    assert all(s1[2 + k, M] == 0 for k in range(5))
    assert all(s1[2 + k, 0] == R * (N - 1) for k in range(5))
    # moments[1] = N - max for every run and step
    assert (s1[3] == R * N - s1[0]).all()
    # spanning is 0/1: sum of squares equals sum
    assert (s2[1] == s1[1]).all()
    # max cluster size and spanning count never decrease
    assert (np.diff(s1[0].astype(float)) >= 0).all()
    assert (np.diff(s1[1].astype(float)) >= 0).all()
    # Cauchy-Schwarz: R * sum x^2 >= (sum x)^2
    for c in range(7):
        assert (R * s2[c] - s1[c] * s1[c] >= 0).all()


def test_pipeline_matches_single_launch(gpu):
    """Sub-batches on three streams (reduction beside the next sweep) give
    the same exact sums as one launch over all runs."""
    from pypercolate_amd._engine import Pipeline
    eng = BondEngine(_graph.square_lattice(32))
    R = 3000
    res = eng.sweep(eng.device_permutations(9, R))
    ref = [t.cpu().numpy() for t in eng.microcanonical_sums(res)]
    pipe = Pipeline(eng, R, seed=9, sub_batch=700)
    for _ in range(2):  # a second run must restart the accumulation
        s1, s2 = pipe.run()
        gpu.cuda.synchronize()
        assert np.array_equal(s1.cpu().numpy(), ref[0])
        assert np.array_equal(s2.cpu().numpy(), ref[1])


@pytest.mark.parametrize('L,after', [(32, 1), (32, 0), (32, 9), (130, 1)])
def test_pipeline_prefetch_matches_single_launch(gpu, L, after):
    """Permutations of the next run() drawn during this one (prefetch):
    every run() gives the one-launch exact sums, also with other work on
    the caller's stream between runs and for the HBM-state sweep."""
    from pypercolate_amd._engine import Pipeline
    eng = BondEngine(_graph.square_lattice(L))
    R = 3000 if L == 32 else 300
    res = eng.sweep(eng.device_permutations(9, R))
    ref = [t.cpu().numpy() for t in eng.microcanonical_sums(res)]
    pipe = Pipeline(eng, R, seed=9, sub_batch=R // 4 + 1, prefetch=True,
                    prefetch_after=after)
    assert pipe.prefetch
    for k in range(4):
        s1, s2 = pipe.run()
        junk = gpu.ones(1 << 20, device='cuda').sum().item()
        assert junk == float(1 << 20)
        gpu.cuda.synchronize()
        assert np.array_equal(s1.cpu().numpy(), ref[0]), k
        assert np.array_equal(s2.cpu().numpy(), ref[1]), k
        assert np.array_equal(pipe.perm.cpu().numpy(), res.perm.cpu().numpy()), k


@pytest.mark.parametrize('L,relabel', [(1, False), (2, False), (3, False),
                                       (8, False), (16, False), (37, False),
                                       (128, False), (8, True), (136, True),
                                       (264, True), (130, False)])
def test_lattice_edges_equal_edge_list(gpu, L, relabel):
    """pc_sweep_lattice (endpoints computed from the edge index, row-major
    or tiled node order) gives pc_sweep's records, span steps and chunk
    states over the closed-form lattice's edge array, in LDS and HBM state
    (L = 136, 264 tiled; L = 130 row-major in HBM)."""
    ga = _graph.square_lattice(L)
    eng = BondEngine(ga, relabel=relabel)
    assert eng.relabelled == relabel
    assert eng.lattice_length == L and eng.lattice_tiled == relabel
    assert eng.lattice_sweep == (L * L > 16384)
    runs = 6 if L < 200 else 3
    perm = eng.device_permutations(31, runs)
    eng.lattice_sweep = True
    lat = eng.sweep(perm, chunks=True)
    eng.lattice_sweep = False
    ref = eng.sweep(perm, chunks=True)
    M = eng.M   # L = 1 has no edges: nothing is written
    np.testing.assert_array_equal(lat.records.cpu().numpy()[:, :M],
                                  ref.records.cpu().numpy()[:, :M])
    np.testing.assert_array_equal(lat.span_step.cpu().numpy(), ref.span_step.cpu().numpy())
    if M:
        np.testing.assert_array_equal(lat.chunk_state.cpu().numpy(),
                                      ref.chunk_state.cpu().numpy())


def test_lattice_sweep_rejects_bad_sizes(gpu):
    from pypercolate_amd import _native as nat
    lib = nat.load_library()
    one = gpu.zeros(8, dtype=gpu.int32, device='cuda')
    args = (None, 0, nat.ptr(one), 1, 1, nat.ptr(one), 1, nat.ptr(one),
            None, 0, 0, 0, None, None)
    assert lib.pc_sweep_lattice(0, 0, *args) == -1
    assert lib.pc_sweep_lattice(12, 1, *args) == -1       # tiles need L % 8 == 0
    assert lib.pc_sweep_lattice(20000, 0, *args) == -1


@pytest.mark.parametrize('ahead,prefetch', [(True, False), (False, False),
                                            (True, True)])
def test_pipeline_bit_exact_mode_matches_oracle(gpu, ahead, prefetch):
    """The pipeline with device RandomState permutations (seeds = run
    index, the L = 16 configuration) gives the oracle's exact sums over
    numpy's permutations, drawn all before the sweeps, per sub-batch, or
    ahead for the next run() (three run() calls, the later ones on
    prefetched permutations)."""
    from pypercolate_amd._engine import Pipeline
    eng = BondEngine(_graph.square_lattice(16))
    g = oracle.percolation_graph_arrays(spanning_2d_grid(16), True)
    tr = oracle.bond_runs(g, oracle.randomstate_permutations(range(40), g['num_edges']))
    ref1, ref2 = oracle.microcanonical_sums(tr)
    pipe = Pipeline(eng, 40, seeds=np.arange(40), sub_batch=16, permute_ahead=ahead,
                    prefetch=prefetch, prefetch_after=1)
    assert pipe.prefetch == prefetch
    for _ in range(3 if prefetch else 1):
        s1, s2 = host_sums(*pipe.run())
        assert (s1 == ref1).all() and (s2 == ref2).all()


@pytest.mark.parametrize('M', [1, 2, 3, 12, 63, 64, 65, 129, 480, 4097, 32512,
                               32768, 32769, 65536, 70000])
def test_randomstate_permutations_bit_exact(gpu, M):
    """Device MT19937 + legacy shuffle == numpy RandomState(seed).permutation:
    up to 32768 edges the swap targets drawn first (64-word blocks settled
    at once) and the swaps applied all at once (per-position step lists,
    pointer jumping); above, the shuffle walked in sequence (LDS array up
    to 65536 edges, the output row above)."""
    eng = BondEngine(_graph.GraphArrays(M + 1, np.stack(
        [np.arange(M), np.arange(1, M + 1)], axis=1)))
    seeds = [0, 1, 42, 12345, 4294967295, 2 ** 31 + 7]
    got = eng.randomstate_permutations(seeds).cpu().numpy()
    for r, seed in enumerate(seeds):
        np.testing.assert_array_equal(
            got[r], np.random.RandomState(seed).permutation(M), err_msg=str(seed))


def test_randomstate_kat_3x3(gpu, golden):
    """The reference's golden permutation (test_percolate.py:141-142)."""
    kat = golden('kat_3x3.json')
    eng = BondEngine(_graph.square_lattice(3))
    got = eng.randomstate_permutations([kat['seed']]).cpu().numpy()[0]
    assert got.tolist() == kat['permutation']


@pytest.mark.parametrize('length,mode', [(16, 'auto'), (128, 'auto'), (64, 'hbm'),
                                         (130, 'auto'), (257, 'auto')])
def test_sweep_chunk_states_equal_chunk_scan(gpu, length, mode):
    """The chunk states the sweep writes itself are bit-identical to the
    separate pass over the records (pc_chunk_scan): LDS state, HBM state
    with 32-bit records, HBM state with 64-bit records."""
    from pypercolate_amd import _native as nat
    eng = BondEngine(_graph.square_lattice(length))
    if mode == 'hbm':
        eng.state_mode = nat.PC_STATE_HBM
    res = eng.sweep(eng.device_permutations(77, 96), chunks=True)
    fused = res.chunk_state.cpu().numpy()
    scanned = eng.chunk_scan(res).cpu().numpy()
    assert np.array_equal(fused, scanned)


@pytest.mark.parametrize('length', [130, 257])
def test_relabelled_state_gives_same_records(gpu, length):
    """HBM-state graphs store the union-find codes in 4 x 8 tiles of the
    grid (BondEngine relabel): records, span steps and chunk states equal
    those of the graph's own labels."""
    g = _graph.square_lattice(length)
    a, b = BondEngine(g, relabel=True), BondEngine(g, relabel=False)
    assert a.relabelled and not b.relabelled
    perm = a.device_permutations(5, 40)
    ra, rb = a.sweep(perm, chunks=True), b.sweep(perm, chunks=True)
    assert np.array_equal(ra.records.cpu().numpy(), rb.records.cpu().numpy())
    assert np.array_equal(ra.span_step.cpu().numpy(), rb.span_step.cpu().numpy())
    assert np.array_equal(ra.chunk_state.cpu().numpy(), rb.chunk_state.cpu().numpy())


@pytest.mark.parametrize('kind,length', [('grid', 2), ('grid', 5), ('grid', 9),
                                         ('grid', 33), ('chain', 2), ('chain', 3),
                                         ('chain', 200)])
@pytest.mark.parametrize('placement', ['lds', 'hbm'])
def test_two_wavefronts_small_graphs(gpu, kind, length, placement):
    """The two-wavefront sweep forced onto small graphs, whose only batch
    or last batch is partial: traces and sums equal the oracle's, and the
    chunk states it writes equal the separate pass."""
    from pypercolate_amd import _native as nat
    from tests.helpers import spanning_1d_chain
    if kind == 'grid':
        ga, nxg = _graph.square_lattice(length), spanning_2d_grid(length)
    else:
        ga, nxg = _graph.linear_chain(length), spanning_1d_chain(length)
    g = oracle.percolation_graph_arrays(nxg, True)
    eng = BondEngine(ga)
    eng.state_mode = nat.PC_SWEEP_TWO_WAVES | (
        nat.PC_STATE_LDS if placement == 'lds' else nat.PC_STATE_HBM)
    perms = oracle.randomstate_permutations(range(12), g['num_edges'])
    expect = oracle.bond_runs(g, perms)
    res = eng.sweep(eng.upload_permutations(perms), chunks=True)
    _check_traces(eng, res, expect)
    _check_sums(eng, res, expect)
    assert np.array_equal(res.chunk_state.cpu().numpy(),
                          eng.chunk_scan(res).cpu().numpy())


@pytest.mark.parametrize('kind', ['star', 'complete', 'wheel'])
def test_hbm_state_hub_graphs(gpu, kind):
    """HBM state forced onto graphs whose merges keep hitting one root (a
    star with extra rim edges, a complete graph, a wheel): the root the
    finder hands over is changed by the resolver in nearly every batch, so
    the resolver's stamp test and re-reads, the star merges and the folder
    wave are all exercised.  Traces and sums equal the oracle's, and the
    chunk states equal the separate pass."""
    import networkx as nx
    from pypercolate_amd import _native as nat
    if kind == 'star':
        gnx = nx.star_graph(3000)
        gnx.add_edges_from((i, i + 1) for i in range(1, 3000, 7))
    elif kind == 'complete':
        gnx = nx.complete_graph(90)
    else:
        gnx = nx.wheel_graph(2500)
    eng, g = _engine_for(gnx, False)
    eng.state_mode = nat.PC_STATE_HBM
    perms = oracle.randomstate_permutations(range(10), g['num_edges'])
    expect = oracle.bond_runs(g, perms)
    res = eng.sweep(eng.upload_permutations(perms), chunks=True)
    _check_traces(eng, res, expect)
    _check_sums(eng, res, expect)
    assert np.array_equal(res.chunk_state.cpu().numpy(),
                          eng.chunk_scan(res).cpu().numpy())


@pytest.mark.parametrize('chunks', [True, False])
def test_hbm_sweep_with_fewer_slots_than_runs(gpu, chunks):
    """A union-find workspace of 7 run slots for 40 runs: each workgroup
    sweeps several runs in turn, clearing its slot, claim and stamp tables
    between them.  Records, span steps and chunk states equal those of a
    workspace with a slot per run."""
    eng = BondEngine(_graph.square_lattice(130))
    assert eng.N > 16384
    perm = eng.device_permutations(11, 40)
    full = eng.sweep(perm, chunks=chunks)
    ws = gpu.empty((7 * eng.N * 4,), dtype=gpu.uint8, device='cuda')
    part = eng.sweep(perm, workspace=ws, chunks=chunks)
    assert np.array_equal(part.records.cpu().numpy(), full.records.cpu().numpy())
    assert np.array_equal(part.span_step.cpu().numpy(), full.span_step.cpu().numpy())
    if chunks:
        assert np.array_equal(part.chunk_state.cpu().numpy(),
                              full.chunk_state.cpu().numpy())


def _tiled_and_untiled(eng, perm, chunks=True):
    """The sweep as the library picks it and with every node's code in HBM."""
    from pypercolate_amd import _native as nat
    assert eng.state_mode == nat.PC_STATE_AUTO
    assert eng.workspace_bytes(perm.shape[0]) > 0
    auto = eng.sweep(perm, chunks=chunks)
    eng.state_mode = nat.PC_STATE_HBM | nat.PC_SWEEP_TWO_WAVES
    hbm = eng.sweep(perm, chunks=chunks)
    eng.state_mode = nat.PC_STATE_AUTO
    return auto, hbm


def _same_sweep(a, b, chunks=True):
    assert np.array_equal(a.records.cpu().numpy(), b.records.cpu().numpy())
    assert np.array_equal(a.span_step.cpu().numpy(), b.span_step.cpu().numpy())
    if chunks:
        assert np.array_equal(a.chunk_state.cpu().numpy(), b.chunk_state.cpu().numpy())


@pytest.mark.parametrize('length,runs', [(65, 2), (65, 600), (80, 40), (95, 1024), (96, 1500),
                                         (100, 3), (127, 700), (128, 200), (128, 1025),
                                         (129, 5), (129, 300), (136, 9), (181, 40), (192, 3),
                                         (255, 2), (256, 200), (257, 8), (512, 2), (513, 2), (700, 1),
                                         (1000, 1), (400, 300)])
def test_tiled_lattice_sweep_equals_untiled(gpu, length, runs):
    """The tiled sweep's records, span steps and chunk states equal those of
    the sweep with every node's code in HBM: tiles of up to 32 x 32 nodes (few
    runs) and 64 x 64, whole and ragged, state within the LDS limit, 32- and
    64-bit records (from 257), open nodes in LDS (a run or several per CU)
    and in HBM (1000; 400 for more than 256 runs), one workgroup per run or
    several."""
    eng = BondEngine(_graph.square_lattice(length))
    perm = eng.device_permutations(17, runs)
    _same_sweep(*_tiled_and_untiled(eng, perm))


@pytest.mark.parametrize('length', [128, 130, 264])
def test_tiled_lattice_sweep_orders(gpu, length):
    """Orders that are far from random: the bonds in their own order and
    reversed, all bonds down before those to the right, a far corner first;
    and rows that are not permutations (one bond twice in another's place,
    one bond throughout), which go through the untiled sweep, beside one
    that is."""
    eng = BondEngine(_graph.square_lattice(length))
    M = eng.M
    one = np.arange(M)
    edges = eng.graph.edges
    down = edges[:, 1] - edges[:, 0] == length
    twice = np.random.RandomState(3).permutation(M)
    twice[5] = twice[M // 2]
    perm = eng.upload_permutations(np.stack(
        [one, one[::-1], np.argsort(~down, kind='stable'), np.argsort(-edges[:, 1], kind='stable'),
         twice, np.full(M, 7), np.random.RandomState(4).permutation(M)]))
    _same_sweep(*_tiled_and_untiled(eng, perm))


@pytest.mark.parametrize('sides', ['none', 'scattered'])
def test_tiled_lattice_sweep_sides(gpu, sides):
    """No spanning sides; and sides on nodes anywhere, so that clusters
    inside a tile touch one side, or both."""
    ga = _graph.square_lattice(200, spanning_cluster=False)
    if sides == 'scattered':
        rng = np.random.RandomState(8)
        ga.node_sides = (rng.randint(0, 400, ga.num_nodes) % 3 *
                         (rng.randint(0, 500, ga.num_nodes) == 0)).astype(np.uint8)
        assert set(np.unique(ga.node_sides)) == {0, 1, 2}
    eng = BondEngine(ga)
    _same_sweep(*_tiled_and_untiled(eng, eng.device_permutations(23, 12)))


def test_tiled_lattice_sweep_small_workspaces(gpu):
    """Workspaces for the lists of some of the runs (slabs), and of too few
    (the untiled sweep): the same records."""
    eng = BondEngine(_graph.square_lattice(264))
    perm = eng.device_permutations(29, 30)
    full = eng.sweep(perm)
    for nbytes in (eng.workspace_bytes(30) // 2, eng.workspace_bytes(10),
                   2 * eng.N * 4, eng.N * 4):
        ws = gpu.empty((nbytes,), dtype=gpu.uint8, device='cuda')
        _same_sweep(eng.sweep(perm, workspace=ws), full)


def test_tiled_lattice_sweep_matches_oracle(gpu):
    """L = 300 (64-bit records): traces and exact sums over two numpy
    permutations equal the oracle's."""
    eng = BondEngine(_graph.square_lattice(300))
    g = oracle.square_lattice_graph(300)
    perms = oracle.randomstate_permutations(range(2), eng.M)
    expect = oracle.bond_runs(g, perms)
    res = eng.sweep(eng.upload_permutations(perms))
    _check_traces(eng, res, expect)
    _check_sums(eng, res, expect)


@pytest.mark.parametrize('M,runs', [(32769, 3), (40000, 1), (65537, 2), (130560, 5),
                                    (524288, 2), (524289, 2), (2095104, 1)])
def test_randomstate_permutations_in_buckets(gpu, M, runs):
    """Runs above 32768 edges in position buckets (32-bit entries up to 2^19
    edges, 64-bit above) equal numpy's, with a workspace for every run, for
    one run, and for none (the swaps in sequence, for the smaller sizes)."""
    import ctypes
    from pypercolate_amd import _native as nat
    eng = BondEngine(_graph.GraphArrays(M + 1, np.stack(
        [np.arange(M), np.arange(1, M + 1)], axis=1)))
    seeds = [3, 4294967295, 77, 0, 123456][:runs]
    want = np.stack([np.random.RandomState(s).permutation(M) for s in seeds])
    np.testing.assert_array_equal(eng.randomstate_permutations(seeds).cpu().numpy(), want)
    b = ctypes.c_uint64(0)
    nat.check(eng.lib.pc_permute_randomstate_workspace_size(M, 1, ctypes.byref(b)), 'size')
    d_seeds = eng.upload_seeds(seeds)
    for nbytes in [b.value] + ([0] if M <= 65537 else []):
        ws = gpu.empty((nbytes,), dtype=gpu.uint8, device='cuda')
        out = gpu.empty((runs, M), dtype=gpu.int32, device='cuda')
        nat.check(eng.lib.pc_permute_randomstate_ws(
            nat.ptr(d_seeds), runs, M, nat.ptr(out), M, nat.ptr(ws), nbytes,
            nat.stream_handle(gpu)), 'pc_permute_randomstate_ws')
        np.testing.assert_array_equal(out.cpu().numpy(), want)


@pytest.mark.parametrize('length,runs,sub', [(20, 3, None), (20, 64, None), (20, 65, None),
                                             (20, 700, 300), (131, 5, 3), (300, 70, None)])
def test_sums_groups(gpu, length, runs, sub):
    """Exact sums with fewer runs than a workgroup's waves, one group of runs
    (stored, into buffers that hold something else) or several (added),
    batches added to one another, for narrow, wide and 64-bit records: equal
    to the sums of the per-run traces."""
    from pypercolate_amd._engine import limbs_to_int
    eng = BondEngine(_graph.square_lattice(length))
    perm = eng.device_permutations(41, runs)
    s1 = gpu.full((7, eng.S, 2), -3, dtype=gpu.int64, device='cuda')
    s2 = gpu.full((7, eng.S, 3), -3, dtype=gpu.int64, device='cuda')
    for i, r0 in enumerate(range(0, runs, sub or runs)):
        res = eng.sweep(perm[r0:r0 + (sub or runs)])
        eng.microcanonical_sums(res, sum1=s1, sum2=s2, accumulate=i > 0)
    mx, sp, mom = eng.host_traces(eng.sweep(perm))
    cols = [mx, sp] + [mom[:, :, k] for k in range(5)]
    got1, got2 = limbs_to_int(s1.cpu().numpy()), limbs_to_int(s2.cpu().numpy())
    steps = np.unique(np.concatenate([np.arange(0, eng.S, max(1, eng.S // 500)),
                                      [1, 63, 64, 65, eng.S - 2, eng.S - 1]]))
    for k in range(7 if length <= 128 else 5):   # moments 3, 4 may pass 2**64
        x = cols[k][:, steps].astype(object)
        assert (got1[k][steps] == x.sum(axis=0)).all(), k
        assert (got2[k][steps] == (x * x).sum(axis=0)).all(), k


@pytest.mark.parametrize('M', [63, 4095, 8191, 8192, 8193, 16385, 32767, 131073, 1048577])
def test_device_permutation_label_bits(gpu, M):
    """Around the edge counts at which the labels gain a bit (0 to 9 bits: 7
    are matched through LDS, the rest by ballots) and the chunks and groups
    end: the oracle's permutations."""
    eng = BondEngine(_graph.GraphArrays(M + 1, np.stack(
        [np.arange(M), np.arange(1, M + 1)], axis=1)))
    got = eng.device_permutations(seed=77, num_runs=3, first_run=9).cpu().numpy()
    want = oracle.bucket_permutations(77, 9, 3, M)
    for r in range(3):
        np.testing.assert_array_equal(got[r], want[r], err_msg='run {}'.format(r))


@pytest.mark.parametrize('N,runs', [(16384, 2500), (16385, 1100), (65536, 1100), (65537, 3),
                                    (1 << 21, 2)])
def test_sums_at_their_bounds(gpu, N, runs):
    """Two clusters of half the nodes each, the largest moments there are,
    at the node counts where the sums' arithmetic changes or ends and with
    more runs than one group holds: sums and sums of squares in closed
    form."""
    h = N // 2
    eng = BondEngine(_graph.GraphArrays(N, np.stack([np.arange(N - 1), np.arange(1, N)], axis=1)))
    order = np.concatenate([np.arange(h - 1), np.arange(h, N - 1), [h - 1]])
    perm = gpu.from_numpy(order.astype(np.int32)).cuda().repeat(runs, 1)
    res = eng.sweep(perm)
    s1, s2 = eng.microcanonical_sums(res)
    steps = np.unique(np.concatenate([np.arange(40), np.arange(h - 70, h + 70),
                                      np.linspace(0, N - 1, 300).astype(int),
                                      np.arange(N - 70, N)]))
    at = gpu.from_numpy(steps).cuda()
    s1 = s1[:, at].cpu().numpy().view(np.uint64)
    s2 = s2[:, at].cpu().numpy().view(np.uint64)
    for j, s in enumerate(int(v) for v in steps):
        sizes = [s + 1] if s < h else [h, s - h + 2] if s < N - 1 else [N]
        singles = N - sum(sizes)
        big = max(sizes)
        x = [big, 0] + [singles + sum(c ** k for c in sizes) - big ** k for k in range(5)]
        for k in range(7):
            assert sum(int(w) << (64 * i) for i, w in enumerate(s1[k, j])) == runs * x[k], (s, k)
            assert sum(int(w) << (64 * i) for i, w in enumerate(s2[k, j])) == runs * x[k] ** 2, (s, k)


@pytest.mark.parametrize('length,runs,orders', [(725, 2, 'own'), (1100, 1, 'own'), (700, 80, 'random'),
                                                (2048, 1, 'random')])
def test_tiled_lattice_sweep_windows(gpu, length, runs, orders):
    """More steps than a list entry tells apart (2^19): the bonds in their
    own order and reversed, so that a tile's list lies in few windows and
    others are empty for it, and random ones, in short segments of the steps
    and in long ones."""
    eng = BondEngine(_graph.square_lattice(length))
    if orders == 'own':
        one = np.arange(eng.M)
        perm = eng.upload_permutations(np.stack([one, one[::-1]][:runs]))
    else:
        perm = eng.device_permutations(31, runs)
    _same_sweep(*_tiled_and_untiled(eng, perm))


@pytest.mark.parametrize('runs', [300, 600])
@pytest.mark.parametrize('M', [2, 3, 64, 65, 127, 128, 480, 1025])
def test_randomstate_permutations_near_masks(gpu, M, runs):
    """Many seeds at the sizes where every accepted word shifts the steps
    that the others in its block may serve, a workgroup a run and a
    wavefront: numpy's permutations."""
    eng = BondEngine(_graph.GraphArrays(M + 1, np.stack(
        [np.arange(M), np.arange(1, M + 1)], axis=1)))
    seeds = [7 * r + M for r in range(runs)]
    got = eng.randomstate_permutations(seeds).cpu().numpy()
    want = np.stack([np.random.RandomState(s).permutation(M) for s in seeds])
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize('spanning', [True, False])
@pytest.mark.parametrize('length', [2, 6, 9, 33, 130, 257])
def test_structured_rows_equal_traces(gpu, length, spanning):
    """The packed rows (53 or 52 bytes, so at every offset from a word) hold
    the traces, the permutation and the row of step 0: narrow and wide
    moments, 32- and 64-bit records, whole and ragged chunks, permutations
    in a wider buffer."""
    from pypercolate_amd import hpc
    eng = BondEngine(_graph.square_lattice(length, spanning_cluster=spanning))
    wide = gpu.full((5, eng.M + 3), -1, dtype=gpu.int32, device='cuda')
    perm = eng.device_permutations(41, 5)
    wide[:, :eng.M] = perm
    res = eng.sweep(perm)
    res.perm = wide[:, :eng.M]
    rows = eng.host_rows(res, hpc.microcanonical_statistics_dtype(spanning))
    mx, sp, mom = eng.host_traces(res)
    assert rows.shape == mx.shape and rows.flags.writeable
    np.testing.assert_array_equal(rows['n'], np.broadcast_to(np.arange(eng.S), mx.shape))
    np.testing.assert_array_equal(rows['edge'][:, 1:], perm.cpu().numpy())
    assert (rows['edge'][:, 0] == 0).all()
    np.testing.assert_array_equal(rows['max_cluster_size'], mx)
    np.testing.assert_array_equal(rows['moments'], mom)
    if spanning:
        np.testing.assert_array_equal(rows['has_spanning_cluster'], sp)


@pytest.mark.parametrize('M,runs,room', [(600000, 16, 40 << 20), (40000, 300, 0)])
def test_randomstate_permutations_without_room(gpu, M, runs, room):
    """With room on the GPU for the workspace of some of the runs, or of
    none, the permutations are still drawn."""
    eng = BondEngine(_graph.GraphArrays(M + 1, np.stack(
        [np.arange(M), np.arange(1, M + 1)], axis=1)))
    seeds = eng.upload_seeds(range(runs))
    out = gpu.empty((runs, M), dtype=gpu.int32, device='cuda')
    gpu.cuda.empty_cache()
    total = gpu.cuda.get_device_properties(0).total_memory
    gpu.cuda.set_per_process_memory_fraction((gpu.cuda.memory_reserved() + room) / total)
    try:
        eng.randomstate_permutations(seeds, out=out)
    finally:
        gpu.cuda.set_per_process_memory_fraction(1.0)
    for r in (0, 1, runs // 2, runs - 1):
        np.testing.assert_array_equal(out[r].cpu().numpy(),
                                      np.random.RandomState(r).permutation(M))


def _allocations(gpu, call):
    before = gpu.cuda.memory_stats()['allocation.all.allocated']
    call()
    gpu.cuda.synchronize()
    return gpu.cuda.memory_stats()['allocation.all.allocated'] - before


@pytest.mark.parametrize('ahead', [True, False])
def test_pipeline_keeps_the_randomstate_workspace(gpu, ahead):
    """A pipeline of numpy's permutations above 32768 edges draws them in a
    workspace of its own: run() allocates nothing."""
    from pypercolate_amd._engine import Pipeline
    pipe = Pipeline(BondEngine(_graph.square_lattice(150)), 7, seeds=range(7), sub_batch=3,
                    permute_ahead=ahead)
    pipe.run()
    assert _allocations(gpu, pipe.run) == 0
    np.testing.assert_array_equal(pipe.perm[5].cpu().numpy(),
                                  np.random.RandomState(5).permutation(pipe.engine.M))


@pytest.mark.parametrize('length,runs,sub', [(70, 1600, 1100), (70, 2700, 1100), (130, 7, 3)])
def test_pipeline_allocates_nothing_in_run(gpu, length, runs, sub):
    """run() finds a workspace for each of its sub-batches, also for a last
    one of fewer runs that is swept in tiles where the others are not (L =
    70, 1024 runs)."""
    from pypercolate_amd._engine import Pipeline
    pipe = Pipeline(BondEngine(_graph.square_lattice(length)), runs, seed=3, sub_batch=sub)
    pipe.run()
    assert _allocations(gpu, pipe.run) == 0


@pytest.mark.parametrize('length,runs,part', [(64, 9, 1), (65, 5, 1), (95, 1024, 1), (95, 1025, 1),
                                              (128, 200, 1), (128, 200, 2), (128, 200, 400)])
def test_lattice_sweep_way_taken(gpu, length, runs, part):
    """A lattice whose codes fit LDS uses its workspace, or a part of it, if
    and only if tiled_runs says that it is swept in tiles; the records are
    the same."""
    eng = BondEngine(_graph.square_lattice(length))
    nbytes = (eng.workspace_bytes(runs) or 1 << 20) // part
    ws = gpu.full((nbytes,), 0xA5, dtype=gpu.uint8, device='cuda')
    perm = eng.device_permutations(11, runs)
    res = eng.sweep(perm, workspace=ws, chunks=False)
    assert bool((ws != 0xA5).any()) == (eng.tiled_runs(runs, nbytes) > 0)
    assert (eng.tiled_runs(runs, nbytes) > 0) == (length > 64 and runs != 1025 and part < 400)
    _same_sweep(res, eng.sweep(perm, chunks=False), chunks=False)


@pytest.mark.parametrize('room', [120 << 20, 0])
def test_tiled_sweep_without_room(gpu, room):
    """L = 128, whose codes fit LDS: with room for the lists of some of the
    runs, or of none, the same records."""
    eng = BondEngine(_graph.square_lattice(128))
    perm = eng.device_permutations(13, 3000)
    want = eng.sweep(perm, chunks=False)
    records, span = gpu.empty_like(want.records), gpu.empty_like(want.span_step)
    assert eng.workspace_bytes(3000) > room + (128 << 20)
    gpu.cuda.empty_cache()
    total = gpu.cuda.get_device_properties(0).total_memory
    gpu.cuda.set_per_process_memory_fraction((gpu.cuda.memory_reserved() + room) / total)
    try:
        eng.sweep(perm, records=records, span_step=span, chunks=False)
    finally:
        gpu.cuda.set_per_process_memory_fraction(1.0)
    assert gpu.equal(records, want.records) and gpu.equal(span, want.span_step)


@pytest.mark.parametrize('M,resident', [(8192, 4), (14620, 4), (16380, 4), (19404, 3), (21424, 3),
                                        (23113, 2), (32736, 2), (32768, 2)])
def test_shuffle_of_whole_runs_fills_the_gpu(gpu, M, resident):
    """The masks that labels are matched in through LDS leave as many
    workgroups on a CU as there are without them where that pays, the largest
    runs among them, and the permutations are the oracle's with any number of
    bits matched so (7, and in many runs of 14620 edges or more 6 or 5)."""
    import ctypes
    from pypercolate_amd import _native as nat
    blocks = ctypes.c_int32(0)
    nat.check(nat.load_library().pc_permute_philox_occupancy(M, ctypes.byref(blocks)), 'occupancy')
    eng = BondEngine(_graph.GraphArrays(M + 1, np.stack(
        [np.arange(M), np.arange(1, M + 1)], axis=1)))
    want = oracle.bucket_permutations(78, 5, 3, M)
    for runs in (3, 1100):
        got = eng.device_permutations(seed=78, num_runs=runs, first_run=5)[:3].cpu().numpy()
        np.testing.assert_array_equal(got, want)
    assert blocks.value == resident


@pytest.mark.parametrize('length,sub', [(2, 1), (2, 150), (16, 24), (16, 25), (20, 1), (130, 1),
                                        (130, 2), (300, 1), (514, 1)])
def test_sums_of_few_runs_added(gpu, length, sub):
    """Batches of few runs, a wavefront each, and of the next more, added one
    after another: the sums of all runs at once."""
    eng = BondEngine(_graph.square_lattice(length))
    perm = eng.device_permutations(43, 3 * sub)
    want = eng.microcanonical_sums(eng.sweep(perm))
    sums = gpu.zeros_like(want[0]), gpu.zeros_like(want[1])
    for r0 in range(0, 3 * sub, sub):
        eng.microcanonical_sums(eng.sweep(perm[r0:r0 + sub]), *sums, accumulate=True)
    assert gpu.equal(sums[0], want[0]) and gpu.equal(sums[1], want[1])


def test_structured_rows_without_room(gpu):
    """Rows of more bytes than there is room for on the GPU, in pieces."""
    from pypercolate_amd import hpc
    eng = BondEngine(_graph.square_lattice(60))
    res = eng.sweep(eng.device_permutations(47, 600))
    dtype = hpc.microcanonical_statistics_dtype(True)
    want = eng.host_rows(res, dtype)
    assert want.nbytes > 200 << 20
    gpu.cuda.empty_cache()
    total = gpu.cuda.get_device_properties(0).total_memory
    gpu.cuda.set_per_process_memory_fraction((gpu.cuda.memory_reserved() + (40 << 20)) / total)
    try:
        got = eng.host_rows(res, dtype)
    finally:
        gpu.cuda.set_per_process_memory_fraction(1.0)
    assert got.tobytes() == want.tobytes()
