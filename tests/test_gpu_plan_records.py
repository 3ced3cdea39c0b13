"""The plan's units on both sides of the record count up to which the records are kept in LDS
(2048; beyond it each unit finds its record by a search), for every mode that writes units:
plan tables and dispatch table bit-exact against the oracle.  Rows of one to four records,
weights over eight buckets, KV groups that are and are not a power of two."""
import pytest

from oracle import plan as OP
from sglang_decode.config import DecodeConfig
from sglang_decode.planning.builder import build_plan
from sglang_decode.runtime.workspace import PlanBuffers

from gpu_util import assert_plan_equal, cfg_ns, read_plan
from test_gpu_plan import expected_table, load, poison

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("force", [1, 2, 3, 4])
@pytest.mark.parametrize("records,kv_heads", [(2047, 4), (2048, 3), (2049, 3), (4100, 4)])
def test_units_around_the_lds_records(records, kv_heads, force):
    c = DecodeConfig(batch_capacity=4000, max_splits=4, max_context=16384, query_heads=4 * kv_heads,
                     kv_heads=kv_heads, workers=96)
    rows = records - 300  # 100 rows of four records among rows of one
    splits = [4 if r % 17 == 0 and r < 1700 else 1 for r in range(rows)]
    lengths = [4096 + 97 * r % 12288 if s == 4 else 1 + (r * 7919) % (128 << r % 8) for r, s in enumerate(splits)]
    plan = PlanBuffers(c, "cuda")
    load(plan, lengths, splits)
    poison(plan)
    plan.dispatch.fill_(-9)
    build_plan(plan, force)
    pad = c.batch_capacity - rows
    ref = OP.full_plan(lengths + [0] * pad, splits + [1] * pad, rows, cfg_ns(c), [], force)
    assert ref["record_count"] == records
    assert_plan_equal(read_plan(plan), ref, c, rows, f"records={records} force={force}")
    expected = expected_table(ref, c, force)
    got = plan.dispatch.cpu()
    assert got[:len(expected)].tolist() == expected
    assert (got[len(expected):] == -9).all()
