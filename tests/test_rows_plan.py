"""Which tile and how many K slices a batched linear gets (host code, no GPU)."""
import numpy as np
import pytest

import three_llm_amd.tlm as tlm
import three_llm_amd.weights as W
from test_gpu_op_rows import CASES

CUS = 256


def partial_gemms(name):
    """(N, K) of the QKV, O and down GEMMs of a workload's prefill."""
    c = W.WORKLOADS[name].config
    h, inner, hq, hkv = (c[k] for k in ("hidden_size", "intermediate_size", "num_attention_heads",
                                        "num_key_value_heads"))
    d = c.get("head_dim") or h // hq
    return [((hq + 2 * hkv) * d, h), (h, hq * d), (h, inner)]


@pytest.mark.parametrize("name", ["qwen2.5-0.5b", "llama-3.2-1b", "llama-3.2-3b"])
def test_partial_sums_take_the_cheaper_tile(name):
    """Each tile is weighed with the slices that it would run in."""
    for n, k in partial_gemms(name):
        for rows in range(65, 2049):
            plan, us, rejected = tlm.rows_plan(tlm.FMT_Q4, rows, n, k, CUS, partial=True)
            assert us <= rejected, f"{rows} x {n} x {k}: {plan} {us} against {rejected}"


@pytest.mark.parametrize("rows,n,k", [(65, 2048, 8192), (71, 2048, 8192), (128, 1024, 8192), (128, 512, 8192),
                                      (148, 432, 7104), (70, 256, 7584)])
def test_short_prompts_keep_the_small_tile_in_slices(rows, n, k):
    (tile_rows, _, slices), us, rejected = tlm.rows_plan(tlm.FMT_Q4, rows, n, k, CUS, partial=True)
    assert tile_rows == 32 and slices > 1
    assert us < 0.75 * rejected


@pytest.mark.parametrize("fmt,rows,n,k,tile,sliced", [(c[0], *c[1:4], c[5], c[6]) for c in CASES])
def test_cases_of_the_op_reach_the_tiles_that_they_are_for(fmt, rows, n, k, tile, sliced):
    plan, _, _ = tlm.rows_plan(fmt, rows, n, k, CUS)
    assert plan[:2] == tile and (plan[2] > 1) == sliced


@pytest.mark.parametrize("fmt,rows,n,k,tile", [
    # the edges of the tiles for few rows over many columns
    (tlm.FMT_Q4, 33, 49153, 896, (64, 256)), (tlm.FMT_Q4, 33, 49152, 896, (32, 64)),
    (tlm.FMT_Q4, 64, 98304, 512, (32, 256)), (tlm.FMT_Q4, 64, 98305, 512, (64, 256)),
    (tlm.FMT_Q4, 32, 130817, 1024, (32, 256)), (tlm.FMT_Q4, 32, 130816, 1024, (32, 64)),
    (tlm.FMT_Q4, 16, 131072, 1056, (32, 64)), (tlm.FMT_Q4, 17, 131072, 1056, (32, 256)),
    (tlm.FMT_F16, 33, 16385, 896, (64, 128)), (tlm.FMT_F16, 33, 16384, 896, (32, 64)),
    (tlm.FMT_F16, 33, 16384, 4096, (64, 128)), (tlm.FMT_F16, 32, 49152, 1024, (64, 128)),
    (tlm.FMT_F16, 32, 49024, 1024, (32, 64)), (tlm.FMT_F16, 8, 98304, 4096, (64, 128)),
    (tlm.FMT_F16, 8, 98305, 4096, (32, 64)), (tlm.FMT_F16, 1, 151936, 8192, (32, 64)),
])
def test_few_rows_over_many_columns(fmt, rows, n, k, tile):
    plan, _, _ = tlm.rows_plan(fmt, rows, n, k, CUS)
    assert plan == (*tile, 1)


def test_plan_refuses_what_the_op_refuses():
    with pytest.raises(tlm.TlmError):
        tlm.rows_plan(tlm.FMT_Q4, 64, 64, 33, CUS)
    with pytest.raises(tlm.TlmError):
        tlm.rows_plan(tlm.FMT_F32, 64, 64, 64, CUS)
