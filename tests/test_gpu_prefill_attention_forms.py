"""GPU parity of the prefill attention forms (nanovllm/layers/attention.py:64-70)
where the launch rule changes: single prompts past 1024 tokens, ragged batches
whose short members end inside a first block, and larger grids of short prompts
on four waves.

Reference: float64 on the CPU.  Tolerance: P rounds to bf16 (2^-8 of each
weight, hence of the largest |v| of the head) and the result once more (2^-8 of
it); an output is a convex combination of v, so 2^-7 of the head's largest |v|.
Over many keys of independent v both roundings and the result are random sums of
the same weights, so by the 2-norm over a head's rows the error stays below 2^-7
of the result, in the first 512 rows and in the later ones, whose outputs are the smallest."""
import pytest
import torch

from nv4.attention import prefill_attention

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("hq,hkv,lens", [(32, 8, [1025]), (32, 8, [1499]), (16, 8, [1100, 3, 65]), (8, 8, [1300]),
                                         (4, 1, [1200, 1, 31, 129]), (8, 2, [300] * 60), (32, 8, [130] * 16),
                                         (32, 8, [200] * 8)])
def test_against_64_bits(hq, hkv, lens):
    print(f"[prefill_forms] hq={hq} hkv={hkv} lens={lens[:4]} x{len(lens)}", flush=True)
    g = torch.Generator("cpu").manual_seed(len(lens) + lens[0])
    n = sum(lens)
    q, k, v = (torch.randn(n, h, 128, generator=g).to(torch.bfloat16) for h in (hq, hkv, hkv))
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32)
    out = prefill_attention(q.to(DEV), k.to(DEV), v.to(DEV), lens, 128**-0.5).cpu()
    assert out.isfinite().all()
    heads = sorted({0, hq - 1, hq // 2})
    for s in sorted({0, len(lens) // 2, len(lens) - 1}):
        a, b = int(cu[s]), int(cu[s + 1])
        for h in heads:
            kh, vh = (t[a:b, h // (hq // hkv)].double() for t in (k, v))
            scores = q[a:b, h].double() @ kh.T * 128**-0.5
            scores.masked_fill_(torch.ones(b - a, b - a, dtype=torch.bool).triu(1), float("-inf"))
            ref = scores.softmax(-1) @ vh
            error = out[a:b, h].double() - ref
            assert error.abs().max() <= 2.0**-7 * vh.abs().max()
            for rows in (slice(0, 512), slice(512, None)):
                assert error[rows].norm() <= 2.0**-7 * ref[rows].norm()
