"""SIP on the GPU is bit-exact with the oracle (csrc/sip.cu:33-167) given the
same scores and offsets: ids and weights compared as raw bits."""
import numpy as np
import pytest
import torch

from ab_attention import _C

pytestmark = pytest.mark.gpu


def _run_gpu(scores: np.ndarray, offsets: np.ndarray, samples: int):
    s = torch.from_numpy(scores).cuda()
    o = torch.from_numpy(offsets).cuda()
    ids = torch.empty((scores.shape[0], samples), dtype=torch.int32, device="cuda")
    logw = torch.empty((scores.shape[0], samples), dtype=torch.float32, device="cuda")
    _C.sip(s, o, ids, logw)
    torch.cuda.synchronize()
    return ids.cpu().numpy(), logw.cpu().numpy()


def _assert_bit_exact(scores, offsets, samples, oracle_mod):
    print(f"sip case rows={scores.shape[0]} pop={scores.shape[1]} samples={samples}", flush=True)
    ids_g, w_g = _run_gpu(scores, offsets, samples)
    ids_o, w_o = oracle_mod.sip(scores, offsets, samples)
    bad_ids = np.argwhere(ids_g != ids_o)
    assert bad_ids.size == 0, f"ids differ at {bad_ids[:5].tolist()}"
    bad_w = np.argwhere(w_g.view(np.uint32) != w_o.view(np.uint32))
    assert bad_w.size == 0, f"weights differ at {bad_w[:5].tolist()}"
    return ids_g, w_g


def _local_masses(rng, rows, pop, peak=0.0):
    """Smooth positive masses with optional spikes (to force certainty)."""
    x = rng.gamma(0.3, size=(rows, pop)).astype(np.float64)
    if peak > 0:
        hot = rng.integers(0, pop, size=(rows, max(1, pop // 64)))
        np.put_along_axis(x, hot, x.max(axis=1, keepdims=True) * peak, axis=1)
    x /= x.sum(axis=1, keepdims=True)
    return x.astype(np.float32)


def test_known_answers(oracle_mod):
    ids, w = _assert_bit_exact(np.ones((1, 8), np.float32), np.array([0.25], np.float32), 2, oracle_mod)
    assert ids.tolist() == [[1, 5]] and w.tolist() == [[2.0, 2.0]]
    ids, w = _assert_bit_exact(np.array([[10, 1, 1, 1, 1, 1, 1, 1]], np.float32),
                               np.array([0.5], np.float32), 2, oracle_mod)
    assert ids.tolist() == [[0, 4]]
    assert w[0, 0] == 0.0 and w[0, 1] == np.float32(np.log2(7.0))


@pytest.mark.parametrize("pop,samples,peak", [
    (512, 64, 0.0), (512, 64, 50.0), (513, 100, 0.0), (1001, 999, 0.0), (8190, 2048, 0.0),
    (8190, 2048, 20.0), (18900, 2048, 0.0), (18900, 2048, 200.0),
])
def test_random_rows(pop, samples, peak, oracle_mod):
    rng = np.random.default_rng(pop * 7 + samples)
    rows = 48
    scores = _local_masses(rng, rows, pop, peak)
    offsets = rng.random(rows, dtype=np.float32)
    _assert_bit_exact(scores, offsets, samples, oracle_mod)


def test_global_row_path(oracle_mod):
    """Hunyuan-size population (29,700 KV4 blocks) exceeds LDS for the
    in-LDS row copy and runs the global-memory row path."""
    rng = np.random.default_rng(3)
    scores = _local_masses(rng, 16, 29700, 30.0)
    offsets = rng.random(16, dtype=np.float32)
    _assert_bit_exact(scores, offsets, 2272, oracle_mod)


def test_degenerate_rows(oracle_mod):
    """Zeros (clamped to 1e-30), tiny and huge masses, one dominant block."""
    rng = np.random.default_rng(11)
    pop = 600
    rows = [np.zeros(pop), np.full(pop, 1e-38), rng.random(pop) * 1e-35,
            np.r_[1e6, np.ones(pop - 1)], np.r_[np.zeros(pop - 5), np.ones(5)]]
    scores = np.stack(rows).astype(np.float32)
    offsets = np.array([0.0, 0.999999, 0.5, 0.25, 0.75], np.float32)
    _assert_bit_exact(scores, offsets, 7, oracle_mod)
    _assert_bit_exact(scores, offsets, 599, oracle_mod)


@pytest.mark.parametrize("pop,rows,peak", [(24577, 8, 0.0), (26001, 8, 40.0), (29700, 600, 30.0), (32768, 8, 0.0),
                                           (39001, 8, 30.0), (41000, 8, 30.0)])
def test_kept_prefix_rows(pop, rows, peak, oracle_mod):
    """Rows whose masses fit in LDS without all prefixes, from the smallest to
    the largest, several per workgroup (600 rows), and one past them; 39,001 and
    41,000 blocks take this many samples from global memory."""
    rng = np.random.default_rng(pop)
    scores = _local_masses(rng, rows, pop, peak)
    scores[1, pop // 2:] = 0.0  # draws fall in the first half, the last residuals at the floor
    offsets = rng.random(rows, dtype=np.float32)
    _assert_bit_exact(scores, offsets, 2272, oracle_mod)


@pytest.mark.parametrize("pop", [8190, 24577, 29700, 41000])
@pytest.mark.parametrize("case", ["infinite masses", "offsets outside [0, 1)"])
def test_irregular_rows(pop, case, oracle_mod):
    """Rows whose prefixes are not finite or whose thresholds do not start in
    [0, 1) are answered as the reference's probes answer them in every storage
    scheme: LDS, kept prefixes (24,577 and 29,700 blocks) and global memory.
    Weights of infinite masses are NaN, of either sign."""
    rng = np.random.default_rng(pop)
    if case == "infinite masses":
        scores, offsets = _local_masses(rng, 5, pop, 30.0), rng.random(5, dtype=np.float32)
        for row, at in ((0, [0]), (1, [pop // 2]), (2, [pop - 1]), (3, [100, 101, pop // 3])):
            scores[row, at] = np.inf
    else:
        offsets = np.array([1.0, 1.75, 600.0, -0.5, -3.25, 1e17, -1e17, np.inf, -np.inf, np.nan], np.float32)
        scores = _local_masses(rng, len(offsets), pop, 30.0)
    print(f"sip irregular rows pop={pop} {case}", flush=True)
    ids_g, w_g = _run_gpu(scores, offsets, 500)
    ids_o, w_o = oracle_mod.sip(scores, offsets, 500)
    assert np.array_equal(ids_g, ids_o)
    assert np.array_equal(w_g, w_o, equal_nan=True)


@pytest.mark.parametrize("pop,rows,samples", [(37001, 8, 1000), (39001, 8, 1024), (39001, 8, 1025), (24577, 8, 6000),
                                              (24577, 300, 6000), (32768, 300, 6553), (32768, 300, 6554)])
def test_kept_prefix_rule(pop, rows, samples, oracle_mod):
    """Both sides of the rule that gives long rows to kept prefixes or to global
    memory: few kept prefixes per chunk, and many samples with more rows than
    CUs."""
    rng = np.random.default_rng(pop + samples)
    scores = _local_masses(rng, 16, pop, 3.0)[np.arange(rows) % 16]
    _assert_bit_exact(scores, rng.random(rows, dtype=np.float32), samples, oracle_mod)
