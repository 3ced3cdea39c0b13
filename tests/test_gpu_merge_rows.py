"""The selective merge where its workgroups walk their rows: fewer rows than workgroups, one and a
few each, more than the 64 whose counts one load brings; requests of 0, 1, 2, 16, 17 and 20 splits in
an order that deals every kind to every wave.  The merged rows are bitwise what the every-row
merge writes, the others untouched."""
import pytest
import torch

from sglang_decode import _lib
from sglang_decode._lib import ptr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bcap,hq,d,smax", [(3, 5, 128, 20), (130, 16, 256, 20), (700, 20, 128, 17),
                                            (4096, 48, 64, 2)])
@pytest.mark.parametrize("min_splits", [2, 17])
def test_rows_walked(bcap, hq, d, smax, min_splits):
    g = torch.Generator(device="cuda").manual_seed(bcap)
    kinds = torch.tensor([n for n in (0, 1, 2, 16, 17, 20) if n <= smax], device="cuda", dtype=torch.int32)
    counts = kinds[torch.randint(len(kinds), (bcap,), generator=g, device="cuda")].contiguous()
    partial = torch.randn((bcap, hq, smax, d), generator=g, device="cuda")
    lse = torch.randn((bcap, hq, smax), generator=g, device="cuda") * 3
    active = torch.tensor([bcap], dtype=torch.int32, device="cuda")
    error = torch.zeros(1, dtype=torch.int32, device="cuda")
    lib, outs = _lib.lib(), []
    for least in (1, min_splits):
        out = torch.full((bcap, hq, d), 7.0, dtype=torch.bfloat16, device="cuda")
        assert lib.sgd_merge_splits_min(ptr(partial), ptr(lse), ptr(counts), ptr(active), ptr(error), ptr(out), bcap, hq,
                                        d, smax, least, _lib.SGD_BF16, _lib.stream_handle(out.device)) == 0
        outs.append(out)
    torch.cuda.synchronize()
    merged = (counts == 0) | (counts >= min_splits)
    assert torch.equal(outs[1][merged].view(torch.int16), outs[0][merged].view(torch.int16))
    assert (outs[1][~merged].float() == 7.0).all()
