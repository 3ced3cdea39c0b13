"""The pipelined attention kernel at the edges of its tiles: contexts around one tile of one
wave (16 or 32 tokens) and of all waves (64 to 256), empty and one-token rows, split and
unsplit, every head_dim, groups 1 to 16 (up to 4, 8 and 16 heads merge differently), CSR and
pages of 16 and 12 tokens; two workers walk long task chains, 512 leave most without a
task.  Against the FP32 oracle at the path's tolerance, and bitwise equal on a second launch
(the merge order is fixed, and no value of an earlier launch's LDS is read)."""
import pytest
import torch

from oracle import attention as OA
from sglang_decode import workloads as W
from sglang_decode.config import DecodeConfig
from sglang_decode.runtime.engine import DecodeEngine

from gpu_util import close

pytestmark = pytest.mark.gpu

LENGTHS = [0, 1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 255, 256, 257, 1000]


@pytest.mark.parametrize("group,dtype", [(1, torch.float16), (4, torch.bfloat16), (8, torch.bfloat16),
                                         (16, torch.float16)])
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("page,workers,mode", [(1, 2, 3), (1, 512, 1), (16, 7, 4), (12, 2, 0)])
def test_tile_edges(group, dtype, d, page, workers, mode):
    c = DecodeConfig(batch_capacity=len(LENGTHS), max_splits=4, max_context=1024, query_heads=2 * group, kv_heads=2,
                     head_dim=d, page_size=page, workers=workers)
    print(f"group {group} d {d} page {page} workers {workers} mode {mode} {dtype}", flush=True)
    splits = [1 + r % 4 for r in range(len(LENGTHS))]
    if page == 1:
        q, k, v, indptr, pages = W.make_csr_inputs(c, LENGTHS, seed=group + d, dtype=dtype)
        expected = OA.csr_attention(q, k, v, indptr, pages, LENGTHS)
    else:
        (q, k, v, pages), indptr = W.make_inputs(c, LENGTHS, seed=group + d, dtype=dtype), None
        expected = OA.paged_attention(q, k, v, pages, LENGTHS, page)
    engine = DecodeEngine(c, dtype=dtype, force_mode=mode)
    W.update_plan(engine, LENGTHS, splits)
    layer = engine.layers[0]
    outs = []
    for _ in range(2):
        layer.partial.fill_(float("nan"))
        layer.lse.fill_(float("nan"))
        engine.prepare()
        outs.append(engine.execute(q, k, v, pages, indptr=indptr).clone())
        assert layer.counter.item() == 0
    assert engine.attention_kernel_name() == ("valu" if group <= 4 else "mfma")
    close(outs[0], expected)
    assert torch.equal(outs[0], outs[1])
