"""The pair-LSE runs with 8, 4 or 2 query blocks per workgroup, by the number
of them in the call: a head's results are the same bits in every call it is
part of."""
import pytest
import torch

from ab_attention import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [4, 252, 260, 1300, 2048])
def test_workgroup_sizes_agree(n):
    """Ragged last groups, chunks and rounds (a round is 256 tokens); 450 heads
    take workgroups of 8 query blocks, 100 of 4 and 3 of 2."""
    lib = _lib.load()
    qb, fb, ld = -(-n // 128), n // 4, lib.ab_ibcs_lse_stride(n)
    per_head = -(-qb // 8)
    g = torch.Generator(device="cuda").manual_seed(n)
    heads = 450
    cent = (torch.randn(heads * qb, 8, 128, device="cuda", generator=g) * 0.2).to(torch.bfloat16)
    pooled = torch.randn(heads, fb, 2, 128, device="cuda", generator=g).to(torch.bfloat16)

    def run(count):
        lse = torch.full((count * qb, 8, ld), float("nan"), dtype=torch.float16, device="cuda")
        mx, den = (torch.full((count * qb, 8), float("nan"), device="cuda") for _ in range(2))
        _lib.check(lib.ab_ibcs_lse(_lib.ptr(cent), _lib.ptr(pooled), count, n, _lib.ptr(lse), _lib.ptr(mx),
                                   _lib.ptr(den), _lib.stream(cent.device)))
        torch.cuda.synchronize()
        return lse[:, :, :fb].contiguous().view(torch.int16), mx, den

    print(f"pair-LSE workgroups n={n} groups per head {per_head}", flush=True)
    whole = run(heads)
    assert torch.isfinite(whole[1]).all() and torch.isfinite(whole[2]).all()
    for count in (100 if per_head < 4 else 40, 3):
        for part, all_heads in zip(run(count), whole):
            assert torch.equal(part, all_heads[:count * qb])
