"""The KV write and q staging where a token's 16-byte pieces do not fill its last workgroup
(256 pieces each): one piece short, exact, one over, several with a remainder; KV and q together
and alone; batches around the limit of workgroups past which a token's workgroups loop over its
pieces (1536 over the batch).  Bit-exact against torch's scatter and copy, a slot outside the pool skipped."""
import pytest
import torch

from sglang_decode.kernels.kv_store import store_kv_and_stage_q

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv,d", [(3, 2, 8), (16, 8, 64), (255, 1, 8), (256, 1, 8), (10, 5, 128), (5, 1, 1000)])
@pytest.mark.parametrize("kv,staged", [(True, True), (True, False), (False, True)])
def test_pieces_remainders(hq, hkv, d, kv, staged):
    batch, tokens = 5, 11
    g = torch.Generator(device="cuda").manual_seed(hq + d)
    new = lambda *s: torch.randn(s, generator=g, device="cuda").to(torch.bfloat16)
    k, v, q = new(batch, hkv, d), new(batch, hkv, d), new(batch, hq, d)
    kc, vc, qo = new(tokens, hkv, d), new(tokens, hkv, d), new(batch + 1, hq, d)
    loc = torch.tensor([10, 0, tokens, 3, 7], dtype=torch.int32, device="cuda")
    ek, ev, eq = kc.clone(), vc.clone(), qo.clone()
    if kv:
        keep = torch.tensor([0, 1, 3, 4], device="cuda")
        ek[loc[keep].long()] = k[keep]
        ev[loc[keep].long()] = v[keep]
    if staged:
        eq[:batch] = q
    store_kv_and_stage_q(*((k, v, loc, kc, vc) if kv else ()), **(dict(q_in=q, q_out=qo) if staged else {}))
    torch.cuda.synchronize()
    assert torch.equal(kc, ek) and torch.equal(vc, ev) and torch.equal(qo, eq)


@pytest.mark.parametrize("batch", [306, 308, 511, 513, 767, 769, 1536, 1537, 4096])
@pytest.mark.parametrize("hq,hkv,d", [(64, 8, 128), (9, 1, 64), (40, 5, 40)])
@pytest.mark.parametrize("loc64", [False, True])
def test_looping_workgroups(batch, hq, hkv, d, loc64):
    g = torch.Generator(device="cuda").manual_seed(batch)
    new = lambda *s: torch.randn(s, generator=g, device="cuda").to(torch.float16)
    k, v, q = new(batch, hkv, d), new(batch, hkv, d), new(batch, hq, d)
    kc, vc, qo = new(5000, hkv, d), new(5000, hkv, d), new(batch, hq, d)
    loc = torch.randperm(5000, generator=g, device="cuda")[:batch].to(torch.int64 if loc64 else torch.int32)
    ek, ev = kc.clone(), vc.clone()
    ek[loc[3:].long()], ev[loc[3:].long()] = k[3:], v[3:]
    loc[:3] = torch.tensor([-1, 5000, -(1 << 31)], dtype=loc.dtype, device="cuda")
    store_kv_and_stage_q(k, v, loc, kc, vc, q_in=q, q_out=qo)
    torch.cuda.synchronize()
    assert torch.equal(kc, ek) and torch.equal(vc, ev) and torch.equal(qo, q)
