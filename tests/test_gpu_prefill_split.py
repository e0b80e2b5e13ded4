"""The prefill with each row's keys split over several workgroups (ab_prefill
with a workspace) and without (workspace NULL), both against the exact oracle
within the bf16 bars of the unsplit tests: splitting only reorders float32
sums."""
import numpy as np
import pytest
import torch

from ab_attention import _lib

MAX_ABS, REL_L2, LSE_ABS = 2e-2, 1e-2, 1e-3
UNIT_BYTES = 16 * 256 * 16 + 128 * 8


def _run(q, k, v, ids, w, order, split):
    bh, nq, nk = q.shape[1], q.shape[2], k.shape[2]
    samples = _lib.PREFILL_DENSE if ids is None else ids.shape[1]
    lib = _lib.load()
    size = lib.ab_prefill_workspace_bytes(bh, nq, nk, samples)
    assert size > 0 and size % UNIT_BYTES == 0
    ws = torch.empty(size, dtype=torch.uint8, device="cuda") if split else None
    out = torch.full_like(q, float("nan"))
    lse = torch.full(q.shape[:3], float("nan"), device="cuda")
    args = _lib.PrefillArgs(*(_lib.ptr(t) for t in (q, k, v, order, ids, w, out, lse)), 1, bh, nq, nk, samples,
                            *(_lib.in_place(t)[1] for t in (q, k, v, out)), None, None, 0,
                            _lib.ptr(ws), size if split else 0)
    _lib.check(lib.ab_prefill(args, _lib.stream(q.device)))
    torch.cuda.synchronize()
    return out.float().cpu().numpy()[0], lse.cpu().numpy()[0]


# (heads, queries, keys, listed blocks or None, logit scale, order): one query
# block and several, ragged queries and keys, part counts that do and do not
# divide the tiles, a first tile whose maximum later parts exceed by far
# (their safe pass), and a token order.
@pytest.mark.gpu
@pytest.mark.parametrize("heads,nq,nk,samples,scale,ordered", [
    (1, 4, 1024, None, 1, False), (2, 200, 4100, None, 1, False), (3, 130, 9000, None, 1, False),
    (1, 128, 8192, None, 40, False), (1, 1000, 4096, 520, 1, False), (2, 2048, 2048, 264, 1, True),
    (2, 2048, 2048, 256, 40, False),
])
def test_split_rows(oracle_mod, heads, nq, nk, samples, scale, ordered):
    torch.manual_seed(nq + nk)
    print(f"split prefill heads={heads} nq={nq} nk={nk} samples={samples} scale={scale}", flush=True)
    q = (torch.randn(1, heads, nq, 128) * scale).to(torch.bfloat16)
    k, v = (torch.randn(1, heads, nk, 128).to(torch.bfloat16) for _ in range(2))
    rows, fb = heads * -(-nq // 128), nk // 4
    ids = w = order = None
    listed = np.tile(np.arange(fb, dtype=np.int32), (rows, 1)), np.zeros((rows, fb), np.float32)
    if samples is not None:
        rng = np.random.default_rng(nq)
        listed = (np.stack([np.sort(rng.choice(fb, samples, replace=False)) for _ in range(rows)]).astype(np.int32),
                  rng.random((rows, samples)).astype(np.float32) * 3)
        # Row 0: its first 96 blocks removed (every block of its first part);
        # row 1: all of them (no output).
        listed[1][0, :96] = -np.inf
        listed[1][1] = -np.inf
        ids, w = (torch.from_numpy(t).cuda() for t in listed)
    if ordered:
        order = torch.randperm(nq, generator=torch.Generator().manual_seed(1))
    f32 = lambda t: t.float().numpy()[0]
    q_seen = q if order is None else q[:, :, order]
    ref_o, ref_l = oracle_mod.prefill(f32(q_seen), f32(k), f32(v), *listed)
    order_d = None if order is None else order.to(torch.int32).cuda()
    for split in (False, True):
        got, lse = _run(q.cuda(), k.cuda(), v.cuda(), ids, w, order_d, split)
        if order is not None:
            got, lse = got[:, order], lse[:, order]
        assert np.abs(got - ref_o).max() <= MAX_ABS, split
        assert np.linalg.norm(got - ref_o) / np.linalg.norm(ref_o) <= REL_L2, split
        finite = np.isfinite(ref_l)
        assert np.array_equal(finite, np.isfinite(lse)), split
        # float32 logits of magnitude L carry about 2^-22 L.
        assert np.abs(lse[finite] - ref_l[finite]).max() <= LSE_ABS * max(1, scale / 4), split


def test_split_rule():
    """Calls with a row per CU or more are not split; the units of a split
    call stay within two per CU and within a row's tiles."""
    size = _lib.load().ab_prefill_workspace_bytes
    dense = _lib.PREFILL_DENSE
    assert size(12, 32760, 32760, dense) == size(80, 75600, 75600, 2048) == size(1, 257 * 128, 8192, dense) == 0
    assert size(0, 128, 128, dense) == size(1, 128, 128, 0) == 0
    assert size(1, 128, 32, dense) == 0  # a single tile
    for bh, nq, nk, samples in [(24, 256, 119056, dense), (1, 4, 119056, dense), (2, 2048, 2048, 256), (2, 16384, 16384, dense)]:
        rows, tiles = bh * -(-nq // 128), -(-(nk // 4 if samples == dense else samples) // 8)
        units, rest = divmod(size(bh, nq, nk, samples), UNIT_BYTES)
        assert rest == 0 and units % rows == 0 and rows < units <= 512 and units // rows * 8 <= tiles


def test_split_rejects_a_bad_workspace():
    lib, a, rows = _lib.load(), 4096, 4 * [(1 << 20, 1 << 14, 128)]  # a stand-in address: rejected before any launch
    for ws, size, message in ((a, 64, b"smaller than"), (a + 8, 1 << 30, b"16-byte aligned")):
        args = _lib.PrefillArgs(a, a, a, None, None, None, a, None, 1, 24, 256, 119056, _lib.PREFILL_DENSE, *rows,
                                None, None, 0, ws, size)
        assert lib.ab_prefill(args, None) == 1 and message in lib.ab_last_error()
    args = _lib.PrefillArgs(a, a, a, None, None, None, a, None, 1, 1, 128, 128, 0, *rows, None, None, 0,
                            None, 0)
    assert lib.ab_prefill(args, None) == 1 and b"multiple of 8" in lib.ab_last_error()
    for bad in ((1 << 20, 1 << 14, 132), (-8, 1 << 14, 128), (1 << 20, 1 << 14, 1 << 21)):
        args = _lib.PrefillArgs(a, a, a, None, None, None, a, None, 1, 1, 128, 128, _lib.PREFILL_DENSE, rows[0], bad,
                                *rows[:2], None, None, 0, None, 0)
        assert lib.ab_prefill(args, None) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("heads,samples,tail", [(2, 8, 8), (2, 504, 24), (2, 512, 8), (3, 1016, 520), (40, 128, 16)])
def test_shared_list(heads, samples, tail):
    """Blocks listed once for all rows equal the same blocks appended to every
    row's list, bit for bit: lists that end inside, at and beyond a batch of 512
    listed blocks, on split calls and (40 heads) an unsplit one."""
    from ab_attention.paged import _prefill_kv

    print(f"shared list heads={heads} samples={samples} tail={tail}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(samples + tail)
    n, fb = 1000, 4096
    q = torch.randn(1, heads, n, 128, device="cuda", generator=g).to(torch.bfloat16)
    k, v = (torch.randn(1, heads, 4 * fb, 128, device="cuda", generator=g).to(torch.bfloat16) for _ in range(2))
    rows = heads * -(-n // 128)
    ids = torch.randint(fb, (rows, samples), device="cuda", generator=g, dtype=torch.int32)
    w = torch.rand(rows, samples, device="cuda", generator=g) * 3
    tail_ids = torch.randint(fb, (1, tail), device="cuda", generator=g, dtype=torch.int32)
    tail_w = torch.zeros(1, tail, device="cuda")
    tail_w[:, -3:] = float("-inf")
    got = _prefill_kv(q, k, v, ids, w, return_lse=True, tail=(tail_ids, tail_w, tail))
    want = _prefill_kv(q, k, v, torch.cat([ids, tail_ids.expand(rows, tail)], 1),
                       torch.cat([w, tail_w.expand(rows, tail)], 1), return_lse=True)
    torch.cuda.synchronize()
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.gpu
@pytest.mark.parametrize("heads,nq,nk,samples", [
    (1, 4, 1024, None), (3, 130, 9000, None), (24, 256, 20000, None), (1, 128, 4100, 520), (2, 2048, 8192, 1024),
    (2, 1000, 16384, 256),
])
def test_split_rounds_as_unsplit(heads, nq, nk, samples):
    """Every part exponentiates against the reference of the whole row, so P has
    the unsplit pass's bf16 bits and only float32 sums are reordered: they
    differ by a few 2^-24 * sqrt(keys) of their size (1e-5 here), which turns
    the bf16 rounding of about 1e-5 / 2^-8 = 0.3 % of the outputs by one step
    (2^-8): 2e-4 of their norm. P rounded against another reference gives 3e-3."""
    print(f"split against unsplit heads={heads} nq={nq} nk={nk} samples={samples}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(nq + nk)
    q = torch.randn(1, heads, nq, 128, device="cuda", generator=g).to(torch.bfloat16)
    k, v = (torch.randn(1, heads, nk, 128, device="cuda", generator=g).to(torch.bfloat16) for _ in range(2))
    ids = w = None
    if samples is not None:
        rows = heads * -(-nq // 128)
        ids = torch.randint(nk // 4, (rows, samples), device="cuda", generator=g, dtype=torch.int32)
        w = torch.rand(rows, samples, device="cuda", generator=g) * 3
    (o, lse), (ref, ref_lse) = (_run(q, k, v, ids, w, None, split) for split in (True, False))
    assert np.linalg.norm(o - ref) / np.linalg.norm(ref) <= 4e-4
    assert np.abs(lse - ref_lse).max() <= 2e-5


def test_longest_lists():
    """Rows of up to 2^30 - 8 listed blocks are taken (these calls stop at the
    misaligned output behind the check of the list), longer ones refused."""
    lib, a, stride = _lib.load(), 4096, (1 << 20, 1 << 14, 128)
    for samples, tail, message in ((1 << 29, 0, b"aligned"), ((1 << 30) - 8, 0, b"aligned"),
                                   ((1 << 30) - 16, 8, b"aligned"), (1 << 30, 0, b"2^30"), ((1 << 30) - 8, 8, b"2^30"),
                                   (8, (1 << 62), b"2^30")):
        args = _lib.PrefillArgs(a, a, a, None, a, a, a + 1, None, 1, 1, 128, 128, samples, *4 * [stride], a, a, tail,
                                None, 0)
        assert lib.ab_prefill(args, None) == 1 and message in lib.ab_last_error(), (samples, tail)
