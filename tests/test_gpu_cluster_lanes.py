"""The clustering runs with two lanes per query on calls of few query blocks
and one on others: a head's centroids, populations and pooled keys are the
same bits in every call it is part of (the small calls are checked against the
oracle in test_gpu_ibcs.py)."""
import pytest
import torch

from ab_attention import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ordered", [(4, False), (36, False), (68, True), (124, False), (128, False), (260, True),
                                       (1000, False)])
def test_lanes_agree(n, ordered):
    """Last blocks that fill part of the first 32 queries, of the first half, of
    the second, or all; equal rows (ties) and a token order among the cases.
    700 heads or more take one lane per query, 5 take two."""
    lib = _lib.load()
    heads, qb, fb = 700, -(-n // 128), n // 4
    g = torch.Generator(device="cuda").manual_seed(n)
    q, k = (torch.randn(1, heads, n, 128, device="cuda", generator=g).to(torch.bfloat16) for _ in range(2))
    q[:, 1, ::2] = q[:, 1, :1]  # half of a head's queries are equal
    q[:, 2] = 0.0
    order = torch.randperm(n, device="cuda", generator=g).to(torch.int32) if ordered else None
    print(f"cluster lanes n={n} ordered={ordered}", flush=True)

    def run(count):
        rows = count * qb
        cent = torch.full((rows, 8, 128), float("nan"), dtype=torch.bfloat16, device="cuda")
        pops = torch.full((rows, 8), float("nan"), device="cuda")
        pooled = torch.full((count, fb, 2, 128), float("nan"), dtype=torch.bfloat16, device="cuda")
        stream = _lib.stream(q.device)
        if order is None:
            _lib.check(lib.ab_ibcs_cluster_pool(_lib.ptr(q), _lib.ptr(k), count, n, _lib.ptr(cent), _lib.ptr(pops),
                                                _lib.ptr(pooled), stream))
            return cent.view(torch.int16), pops, pooled.view(torch.int16)
        size = lib.ab_ibcs_workspace_bytes(count, n)  # centroids lie first in it
        ws = torch.zeros(size, dtype=torch.uint8, device="cuda")
        scores = torch.empty(rows, fb, device="cuda")
        _lib.check(lib.ab_ibcs_ordered(_lib.ptr(q), _lib.ptr(k), _lib.ptr(order), count, n, _lib.ptr(ws), size,
                                       _lib.ptr(scores), stream))
        return ws[:rows * 8 * 128 * 2].view(torch.int16).view(rows, 8, 128), scores

    whole, few = run(heads), run(5)
    torch.cuda.synchronize()
    for a, b in zip(few, whole):
        assert torch.equal(a, b[:len(a)])


@pytest.mark.parametrize("valid", [4, 28, 36, 60])
@pytest.mark.parametrize("heads", [5, 700])
def test_nan_in_a_short_last_block(heads, valid):
    """A NaN among fewer than 64 queries leaves no distance to the mean that is
    a number: the farthest query is then a padding one, a zero row, and every
    query falls to it (two lanes per query for 5 heads, one for 700)."""
    n, lib = 128 + valid, _lib.load()
    g = torch.Generator(device="cuda").manual_seed(valid)
    q, k = (torch.randn(1, heads, n, 128, device="cuda", generator=g).to(torch.bfloat16) for _ in range(2))
    q[0, 1, n - 1, 5] = float("nan")  # the last query
    q[0, 2, n - 1] = float("nan")
    q[0, 3, 128, 7] = float("nan")  # the block's first
    cent = torch.empty(2 * heads, 8, 128, dtype=torch.bfloat16, device="cuda")
    pops = torch.empty(2 * heads, 8, device="cuda")
    pooled = torch.empty(heads, n // 4, 2, 128, dtype=torch.bfloat16, device="cuda")
    print(f"cluster NaN heads={heads} valid={valid}", flush=True)
    _lib.check(lib.ab_ibcs_cluster_pool(_lib.ptr(q), _lib.ptr(k), heads, n, _lib.ptr(cent), _lib.ptr(pops),
                                        _lib.ptr(pooled), _lib.stream(q.device)))
    torch.cuda.synchronize()
    for head in (1, 2, 3):
        row = 2 * head + 1
        assert pops[row].tolist() == [valid] + 7 * [0]
        assert bool((torch.isnan(cent[row, 0]) == torch.isnan(q[0, head, 128:]).any(0)).all())
        assert not bool(cent[row, 1:].any())
    assert bool((pops.sum(1) == torch.tensor([128, valid], device="cuda").repeat(heads)).all())
