"""GPU contraction at every precision against numpy FP64 (and so against
each other): Q[p][c] = sum_k w[p][k] X[start_p + k][c].  Tolerances:
FP64 forms 1e-13 relative; the FP32-input forms 2e-6 relative to the sum of
|w X| (FP32 inputs round at 2^-24)."""
import numpy as np
import pytest

from pypercolate_amd import _engine as E
from pypercolate_amd import _native as nat

pytestmark = pytest.mark.gpu

TOL = {'fp64': 1e-13, 'fp64_mfma': 1e-13, 'fp32_mfma': 2e-6, 'bf16x3_mfma': 2e-6}


def _numpy_contract(x, wt):
    w = wt.w.cpu().numpy()
    out = np.zeros((w.shape[0], x.shape[1]))
    mag = np.zeros_like(out)
    for i in range(w.shape[0]):
        s, L = int(wt.host_start[i]), int(wt.host_length[i])
        out[i] = w[i, :L] @ x[s:s + L]
        mag[i] = w[i, :L] @ np.abs(x[s:s + L])
    return out, mag


@pytest.mark.parametrize('precision', sorted(TOL))
@pytest.mark.parametrize('S,P,C', [(481, 101, 7), (4001, 37, 14), (32513, 40, 21),
                                   (2000, 16, 1)])
def test_contract_precisions(gpu, precision, S, P, C):
    rng = np.random.RandomState(S + P + C)
    # column c scaled by 10^(c mod 5): asymmetric in p and c, wide range
    x = rng.rand(S, C) * (10.0 ** (np.arange(C) % 5))[None, :]
    x[:, 0] -= 0.3  # one column with mixed signs
    ps = np.sort(rng.uniform(0.05, 0.95, size=P))
    wt = E.binomial_weights(S - 1, ps)
    dx = gpu.from_numpy(x).cuda()
    got = E.contract(dx, wt, nat.PRECISIONS[precision]).cpu().numpy()
    ref, mag = _numpy_contract(x, wt)
    err = np.abs(got - ref) / mag
    assert err.max() < TOL[precision], (precision, err.max())


def test_contract_deterministic(gpu):
    rng = np.random.RandomState(0)
    x = rng.rand(8001, 14)
    wt = E.binomial_weights(8000, np.linspace(0.3, 0.7, 64))
    dx = gpu.from_numpy(x).cuda()
    for prec in ('fp64_mfma', 'fp32_mfma', 'bf16x3_mfma'):
        plan = E.ContractPlan(dx, wt, nat.PRECISIONS[prec])
        a = plan.run().cpu().numpy().copy()
        b = plan.run().cpu().numpy()
        assert np.array_equal(a, b)


@pytest.mark.parametrize('S,P,C,lo,hi', [(481, 101, 70, 0.05, 0.95),
                                         (8001, 130, 1100, 0.2, 0.8),
                                         (4001, 1000, 4160, 0.45, 0.55)])
def test_contract_wide_fp64_mfma(gpu, S, P, C, lo, hi):
    """The wide FP64 matrix-core kernel (64 x 64 tiles through LDS, from 64
    columns on): with K-slices (few tiles) and without (>= 1024 tiles),
    partial tiles in p and in columns."""
    rng = np.random.RandomState(S + P)
    x = rng.rand(S, C) * (10.0 ** (np.arange(C) % 5))[None, :]
    x[:, 1] -= 0.5
    ps = np.sort(rng.uniform(lo, hi, size=P))
    wt = E.binomial_weights(S - 1, ps)
    dx = gpu.from_numpy(x).cuda()
    plan = E.ContractPlan(dx, wt, 'fp64_mfma')
    got = plan.run().cpu().numpy().copy()
    ref, mag = _numpy_contract(x, wt)
    err = np.abs(got - ref) / mag
    assert err.max() < 1e-13, err.max()
    assert np.array_equal(got, plan.run().cpu().numpy())


@pytest.mark.parametrize('R,cols', [(1, 7), (255, 6), (1000, 7), (4099, 8)])
def test_run_moments(gpu, R, cols):
    """pc_run_moments: mean and sum of squared deviations over runs of
    q[p][r * cols + c], against numpy (one workgroup per p, runs strided
    over 256 threads)."""
    rng = np.random.RandomState(R)
    P = 9
    q = rng.rand(P, R, cols) * 100.0 + rng.rand(P, 1, cols) * 1e4
    dq = gpu.from_numpy(q.reshape(P, R * cols)).cuda()
    mean = gpu.empty((P, cols), dtype=gpu.float64, device='cuda')
    m2 = gpu.empty_like(mean)
    lib = nat.load_library()
    nat.check(lib.pc_run_moments(nat.ptr(dq), P, R, cols, nat.ptr(mean),
                                 nat.ptr(m2), nat.stream_handle(gpu)),
              'pc_run_moments')
    mu = q.mean(axis=1)
    np.testing.assert_allclose(mean.cpu().numpy(), mu, rtol=1e-13)
    d2 = ((q - mu[:, None, :]) ** 2).sum(axis=1)
    np.testing.assert_allclose(m2.cpu().numpy(), d2, rtol=1e-10, atol=1e-12)


@pytest.mark.parametrize('S,lens,C', [
    (1, [1], 64), (2, [2], 65), (3, [1, 2, 3, 0, 3], 64), (4, [4, 0, 1, 3, 2], 66),
    (15, list(range(16)) * 5, 127), (16, [16] * 64, 128), (17, [17, 3, 16, 1] * 17, 129),
    (31, [5, 0, 31] * 43, 70), (33, [33, 1, 2, 15, 16, 17] * 11, 191),
    (700, [3, 700, 64, 1, 350] * 26, 65), (2500, [1200] * 200, 4096)])
def test_contract_wide_windows(gpu, S, lens, C):
    """The wide kernel's blocks of 16 steps against windows of every length
    and phase (shorter than the four weights a lane reads, empty, starting
    and ending inside a block, the last ending at the last step), p and
    column counts around its tiles, with and without K-slices, and the
    columns of a wider X."""
    rng = np.random.RandomState(S + C)
    lens = np.minimum(np.array(lens, dtype=np.int64), S)
    start = np.array([rng.randint(0, S - n + 1) for n in lens], dtype=np.int64)
    start[-1] = S - lens[-1]
    if S == 2500:       # neighbouring p share most of their steps
        start = np.sort(start)
    kmax = max(int(lens.max()), 1)
    w = rng.rand(len(lens), kmax) - 0.3
    x = np.ascontiguousarray(rng.rand(S, C) * 10.0 ** (np.arange(C) % 5))
    wt = E.Weights(S - 1, np.zeros(len(lens)), gpu.from_numpy(start).cuda(),
                   gpu.from_numpy(lens).cuda(), kmax, gpu.from_numpy(w).cuda())
    wt.host_start, wt.host_length = start, lens
    ref = _numpy_contract(x, wt)[0]
    mag = np.array([np.abs(w[i, :n]) @ x[a:a + n]        # sum of |w X|
                    for i, (a, n) in enumerate(zip(start, lens))])
    q = E.contract(gpu.from_numpy(x).cuda(), wt, 'fp64_mfma').cpu().numpy()
    assert (np.abs(q - ref) <= 1e-13 * mag).all()
    # an infinite step outside every window changes nothing
    used = np.zeros(S, dtype=bool)
    for a, n in zip(start, lens):
        used[a:a + n] = True
    lo, hi = (np.nonzero(used)[0][[0, -1]] if used.any() else (0, S - 1))
    y = x.copy()
    y[:lo] = np.inf
    y[hi + 1:] = np.nan
    z = E.contract(gpu.from_numpy(y).cuda(), wt, 'fp64_mfma').cpu().numpy()
    np.testing.assert_array_equal(z, q)


@pytest.mark.parametrize('precision', sorted(TOL))
@pytest.mark.parametrize('C', [7, 14, 30, 70])
def test_contract_windows_past_the_last_step(gpu, precision, C):
    """The C entry leaves out weights of steps past the last one, which meet no
    row of X, in every form (the rows behind X hold NaN here)."""
    if precision == 'fp64' and C > 32:
        return
    rng = np.random.RandomState(C)
    S, lens, start = 300, np.array([40, 300, 290, 7]), np.array([270, 0, 20, 299])
    kmax = 330
    w = rng.rand(4, kmax)
    buf = np.full((S + 40, C), np.nan)
    buf[:S] = rng.rand(S, C)
    wt = E.Weights(S - 1, np.zeros(4), gpu.from_numpy(start).cuda(),
                   gpu.from_numpy(lens).cuda(), kmax, gpu.from_numpy(w).cuda())
    wt.host_start, wt.host_length = start, np.minimum(lens, S - start)
    got = E.contract(gpu.from_numpy(buf).cuda()[:S], wt, precision).cpu().numpy()
    for i, (a, n) in enumerate(zip(start, np.minimum(lens, S - start))):
        ref = w[i, :n] @ buf[a:a + n]
        assert (np.abs(got[i] - ref) <= TOL[precision] * ref).all(), i
