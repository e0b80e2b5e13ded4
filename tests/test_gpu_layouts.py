"""Q, K and V that are not contiguous are read where they lie (or copied where
their rows cannot be): every public call equals the same call on contiguous
tensors bit for bit, for each form of strides the dispatch distinguishes."""
import contextlib

import pytest
import torch

from ab_attention import _C, _lib, apply_plan, attention, build_plan, paged, video
from ab_attention.video import apply_cube_plan, cube_plan, exact_attention

B, H, N, GRID = 2, 3, 1920, (6, 16, 20)


def _forms(x):
    """Views equal to x [B, H, N, 128] in every layout; True: read in place."""
    b, h, n, d = x.shape
    wide = torch.zeros(b, h, n + 20, d, dtype=x.dtype, device=x.device)
    wide[:, :, 12:12 + n] = x
    odd = torch.zeros(b * h * n * d + 4, dtype=x.dtype, device=x.device)
    odd[4:] = x.transpose(1, 2).reshape(-1)
    packed = torch.zeros(b, n, h, 3, d, dtype=x.dtype, device=x.device)  # one projection of Q, K and V
    packed[:, :, :, 1] = x.transpose(1, 2)
    return {
        "token major": (x.transpose(1, 2).contiguous().transpose(1, 2), True),
        "token slice": (wide[:, :, 12:12 + n], True),
        "batch inside": (x.permute(2, 0, 1, 3).contiguous().permute(1, 2, 0, 3), True),
        "packed": (packed[:, :, :, 1].transpose(1, 2), True),
        "misaligned rows": (odd[4:].view(b, n, h, d).transpose(1, 2), False),
        "dims outside": (x.transpose(2, 3).contiguous().transpose(2, 3), False),
    }


def test_forms_read_in_place():
    x = torch.randn(B, H, 64, 128).to(torch.bfloat16)
    for name, (view, in_place) in _forms(x).items():
        got, strides = _lib.in_place(view)
        assert torch.equal(got, x), name
        assert (got.data_ptr() == view.data_ptr()) == in_place, name
        assert strides == got.stride()[:3], name
    one = torch.zeros(1, 1, 64, 128).as_strided((1, 1, 64, 128), (5, 3, 128, 1))
    assert _lib.in_place(one)[0] is one and _lib.in_place(one)[1] == (64 * 128, 64 * 128, 128)
    still = torch.zeros(1, 1, 1, 128).expand(2, 2, 64, 128)
    assert _lib.in_place(still)[0].is_contiguous()  # a token stride of 0 is copied


@pytest.mark.parametrize("batch,heads,tokens,q_tokens", [(1, 1024, 131072, 131072), (2, 1024, 131072, 131072),
                                                         (2, 2048, 65536, 64), (1, 2048, 131072, 128)])
def test_long_batch_strides(batch, heads, tokens, q_tokens, monkeypatch):
    """Tensors of 2^27 tokens and more per batch item (their batch stride does
    not fit 32 bits) pass the library's checks of strides: it stops at the
    stand-in addresses put in here. A token-major q is copied beside them."""
    lib, seen = _lib.load(), []

    class Library:
        ab_ibcs_sip_workspace_bytes = lib.ab_ibcs_sip_workspace_bytes
        ab_prefill_workspace_bytes = lib.ab_prefill_workspace_bytes

        @staticmethod
        def ab_prefill(args, stream):
            args.q = args.k = args.v = args.out = 4097
            return seen.append((lib.ab_prefill(args, None), lib.ab_last_error())) or 0

        @staticmethod
        def ab_plan(args, stream):
            args.q = args.k = args.offsets = args.ids = args.log_weights = 4097
            return seen.append((lib.ab_plan(args, None), lib.ab_last_error())) or 0

    monkeypatch.setattr(_lib, "load", lambda: Library)
    monkeypatch.setattr(_lib, "on", lambda device: contextlib.nullcontext())
    monkeypatch.setattr(_lib, "stream", lambda device: None)
    like = dict(dtype=torch.bfloat16, device="meta")
    k = torch.empty(batch, heads, tokens, 128, **like)
    for q in (torch.empty(batch, heads, q_tokens, 128, **like),
              torch.empty(batch, q_tokens, heads, 128, **like).transpose(1, 2)):
        paged._run(q, k, k, None, None, _lib.PREFILL_DENSE, None, False)
    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    rows = tokens // 128
    _C.plan_heads(k, k, 0, 1, torch.empty(rows, device="meta"), torch.empty(rows, 32, device="meta", dtype=torch.int32),
                  torch.empty(rows, 32, device="meta"), 32)
    assert [rc for rc, _ in seen] == [1, 1, 1] and all(b"aligned" in message for _, message in seen), seen


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["token major", "token slice", "batch inside", "packed", "misaligned rows",
                                  "dims outside", "shared heads"])
def test_layouts_equal_contiguous(form, monkeypatch):
    print(f"layout {form}", flush=True)
    torch.manual_seed(4)
    q, k, v = (torch.randn(B, H, N, 128, device="cuda").to(torch.bfloat16) for _ in range(3))
    if form == "shared heads":  # K/V of one head for all of them: a head stride of 0
        ks, vs = k[:, :1].expand(B, H, N, 128), v[:, :1].expand(B, H, N, 128)
        qs, k, v = q, ks.contiguous(), vs.contiguous()
    else:
        qs, ks, vs = (_forms(t)[form][0] for t in (q, k, v))
    want = build_plan(q, k, sample_pages=4)
    for heads in (B * H, 1, 4):  # heads per chunk; a chunk of 4 crosses the batch items
        monkeypatch.setattr(attention, "_heads_per_chunk", lambda *_: heads)
        plan = build_plan(qs, ks, sample_pages=4)
        assert torch.equal(plan.descriptor, want.descriptor)
        assert torch.equal(plan.log_weights.view(torch.int32), want.log_weights.view(torch.int32))
    cube = cube_plan(qs, ks, GRID, sample_pages=4)
    assert torch.equal(cube.descriptor, cube_plan(q, k, GRID, sample_pages=4).descriptor)
    for call in (lambda *t: apply_plan(*t, want, return_lse=True), lambda *t: exact_attention(*t, return_lse=True),
                 lambda *t: apply_cube_plan(*t, cube, GRID, return_lse=True)):
        for got, ref in zip(call(qs, ks, vs), call(q, k, v)):
            assert got.is_contiguous() and torch.equal(got, ref)
    torch.cuda.synchronize()


@pytest.mark.gpu
def test_folded_batch():
    """K and V whose batch stride does not fit 32 bits, read where they lie as
    heads of one batch item (51.5 GB of untouched memory around them)."""
    print("folded batch", flush=True)
    b, h, n, far = 2, 2, 256, 1 << 34
    g = torch.Generator(device="cuda").manual_seed(5)
    q, k, v = (torch.randn(b, h, n, 128, device="cuda", generator=g).to(torch.bfloat16) for _ in range(3))
    memory = torch.empty(far + far // 2 + 2 * n * 128, dtype=torch.bfloat16, device="cuda")
    views = [memory[i * n * 128:].as_strided((b, h, n, 128), (far, far // 2, 128, 1)) for i in range(2)]
    for view, t in zip(views, (k, v)):
        view.copy_(t)
    want, out = exact_attention(q, k, v), torch.empty_like(q)
    ws = torch.empty(_lib.load().ab_prefill_workspace_bytes(b * h, n, n, _lib.PREFILL_DENSE) + 16, dtype=torch.uint8,
                     device="cuda")
    near, wide = (h * n * 128, n * 128, 128), (far, far // 2, 128)
    args = _lib.PrefillArgs(*(_lib.address(t) for t in (q, *views, None, None, None, out, None)), b, h, n, n,
                            _lib.PREFILL_DENSE, near, wide, wide, near, None, None, 0, _lib.address(ws), ws.numel())
    _lib.check(_lib.load().ab_prefill(args, _lib.stream(q.device)))
    torch.cuda.synchronize()
    assert torch.equal(out, want)


def test_plan_heads_checks(monkeypatch):
    """Tensors that do not match each other never reach the library, which reads
    and writes them by their strides and row counts."""
    class Library:
        ab_ibcs_sip_workspace_bytes = staticmethod(lambda *_: 16)
        ab_plan = staticmethod(lambda *_: pytest.fail("reached the library"))

    monkeypatch.setattr(_lib, "load", lambda: Library)
    monkeypatch.setattr(_lib, "on", lambda device: contextlib.nullcontext())
    monkeypatch.setattr(_lib, "stream", lambda device: None)
    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    q = torch.empty(2, 3, 1000, 128, dtype=torch.bfloat16)
    rows = 4 * 8  # heads 1 .. 4
    good = dict(q=q, k=q, offsets=torch.empty(rows), ids=torch.empty(rows, 32, dtype=torch.int32),
                logs=torch.empty(rows, 32))
    for name, bad in (("k", q[:, :, :996]), ("k", q[:, :2]), ("k", q[0]), ("offsets", torch.empty(rows - 1)),
                      ("offsets", torch.empty(2 * rows)[::2]), ("ids", torch.empty(rows - 1, 32, dtype=torch.int32)),
                      ("ids", torch.empty(rows, 32)), ("logs", torch.empty(rows, 31)),
                      ("logs", torch.empty(rows, 32, dtype=torch.float64)),
                      ("logs", torch.empty(rows, 64)[:, ::2]), ("ids", torch.empty(rows, 32, device="meta"))):
        a = dict(good, **{name: bad})
        with pytest.raises(RuntimeError):
            _C.plan_heads(a["q"], a["k"], 1, 5, a["offsets"], a["ids"], a["logs"], 32)


def test_plans_are_checked(monkeypatch):
    """A plan on another device, or with other rows than the queries', never
    reaches the library (a kept plan can be another video's)."""
    class Library:
        ab_prefill_workspace_bytes = staticmethod(lambda *_: 0)
        ab_prefill = ab_remap_ids = staticmethod(lambda *_: pytest.fail("reached the library"))

    monkeypatch.setattr(_lib, "load", lambda: Library)
    monkeypatch.setattr(_lib, "on", lambda device: contextlib.nullcontext())
    monkeypatch.setattr(_lib, "stream", lambda device: None)
    monkeypatch.setattr(video, "_check_qkv", lambda *_: None)
    monkeypatch.setattr(paged, "check_prefill_inputs", lambda *_: None)
    q = torch.empty(2, 3, 4 * 16 * 16 + 32, 128, dtype=torch.bfloat16)
    cube = q[:, :, :1024]
    for device, rows, weight_rows in (("meta", 48, 48), ("cpu", 40, 40), ("cpu", 48, 40), ("cpu", 96, 96)):
        plan = attention.SamplePlan(torch.zeros(rows, 2, 32, dtype=torch.int32, device=device),
                                    torch.zeros(weight_rows, 2, 32))
        schedule = video.VideoAttention(2)
        schedule.step, schedule.plan = 12, lambda *_: plan
        with pytest.raises(ValueError):
            video.hunyuan_attention(schedule, 1, q, q, q, 1024, 32)
        with pytest.raises(ValueError):
            apply_cube_plan(cube, cube, cube, plan, (4, 16, 16))


def _token_major(*tensors):
    return tuple(t.transpose(1, 2).contiguous().transpose(1, 2) for t in tensors)


def _split_parts(heads, nq, nk, samples):
    return _lib.load().ab_prefill_workspace_bytes(heads, nq, nk, samples) > 0


@pytest.mark.gpu
@pytest.mark.parametrize("heads,n,samples,tail,split", [
    (2, 2048, 512, 0, True), (1, 1000, 520, 24, True), (2, 1000, 504, 520, True),
    (40, 1000, 128, 0, False), (40, 1000, 64, 16, False), (3, 12000, 2000, 8, False),
])
def test_strided_lists(heads, n, samples, tail, split):
    """The sparse kernels on token-major K/V, with and without shared blocks, in
    split calls (lists that end inside and beyond a batch of 512 blocks) and
    unsplit ones."""
    print(f"strided lists heads={heads} n={n} samples={samples} tail={tail}", flush=True)
    assert _split_parts(heads, n, n, samples + tail) == split
    g = torch.Generator(device="cuda").manual_seed(samples)
    q, k, v = (torch.randn(1, heads, n, 128, device="cuda", generator=g).to(torch.bfloat16) for _ in range(3))
    rows = heads * -(-n // 128)
    ids = torch.randint(n // 4, (rows, samples), device="cuda", generator=g, dtype=torch.int32)
    w = torch.rand(rows, samples, device="cuda", generator=g) * 3
    shared = (None, None, 0)
    if tail:
        shared = (torch.randint(n // 4, (1, tail), device="cuda", generator=g, dtype=torch.int32),
                  torch.zeros(1, tail, device="cuda"), tail)
    want = paged._prefill_kv(q, k, v, ids, w, return_lse=True, tail=shared)
    for form in (_token_major(q, k, v), (q, *_token_major(k), v)):
        got = paged._prefill_kv(*form, ids, w, return_lse=True, tail=shared)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.gpu
@pytest.mark.parametrize("heads,nq,nk,split", [(40, 1000, 2000, False), (3, 12000, 1000, False), (2, 200, 4100, True)])
def test_strided_dense(heads, nq, nk, split):
    """The dense kernels on token-major tensors, split and not."""
    print(f"strided dense heads={heads} nq={nq} nk={nk}", flush=True)
    assert _split_parts(heads, nq, nk, _lib.PREFILL_DENSE) == split
    g = torch.Generator(device="cuda").manual_seed(nk)
    q = torch.randn(1, heads, nq, 128, device="cuda", generator=g).to(torch.bfloat16)
    k, v = (torch.randn(1, heads, nk, 128, device="cuda", generator=g).to(torch.bfloat16) for _ in range(2))
    want = exact_attention(q, k, v, return_lse=True)
    for form in (_token_major(q, k, v), (q, k, *_token_major(v))):
        for got, ref in zip(exact_attention(*form, return_lse=True), want):
            assert torch.equal(got, ref)


@pytest.mark.gpu
@pytest.mark.parametrize("heads", [2, 24])
@pytest.mark.parametrize("layout", ["contiguous", "token major"])
def test_hunyuan_batches(heads, layout):
    """Every part of the partition at two batch items, written into its slice of
    the output, against the same parts computed from contiguous copies and
    concatenated (2 heads split the video's rows, 24 do not)."""
    n_video, prompt, padding, pages = 2560, 40, 24, 16
    n, end = n_video + prompt + padding, n_video + prompt
    print(f"hunyuan batches heads={heads} {layout}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(heads)
    q, k, v = (torch.randn(2, heads, n, 128, device="cuda", generator=g).to(torch.bfloat16) for _ in range(3))
    part = lambda t, *s: t[:, :, slice(*s)].contiguous()
    plan = build_plan(part(q, n_video), part(k, n_video), sample_pages=pages)
    rows = plan.descriptor.shape[0]
    assert _split_parts(2 * heads, n_video, end, 32 * pages + 16) == (heads == 2)
    text = [t.expand(rows, -1) for t in video._dense_pages(1, prompt // 4, "cuda", offset=n_video // 4)]
    ids, w = (torch.cat([p.reshape(rows, -1), t], 1) for p, t in zip(plan, text))
    seen = part(k, end), part(v, end)
    rest = exact_attention(part(q, end, n), part(k, end, n), part(v, end, n))
    sparse = torch.cat([paged._prefill_kv(part(q, n_video), *seen, ids, w),
                        exact_attention(part(q, n_video, end), *seen), rest], 2)
    dense = torch.cat([exact_attention(part(q, end), *seen), rest], 2)
    given = (q, k, v) if layout == "contiguous" else _token_major(q, k, v)
    schedule = video.VideoAttention(pages)
    assert torch.equal(video.hunyuan_attention(schedule, 1, *given, n_video, prompt), dense)
    schedule.step, schedule.plan = 12, lambda *_: plan
    assert torch.equal(video.hunyuan_attention(schedule, 1, *given, n_video, prompt), sparse)
    torch.cuda.synchronize()
