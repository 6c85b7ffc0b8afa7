"""Which calls take several whole rows to a workgroup, and which stay where they were (planner only)."""
import pytest
import torch

from linrec_amd import _native as nat


def _kernel(shape, dtype=torch.float32, is_bwd=False, **kw):
    t = torch.empty_strided(shape, kw["strides"], dtype=dtype) if "strides" in kw else torch.empty(shape, dtype=dtype)
    plan = nat.plan(t, False, is_bwd)
    return nat.kernel_table()[plan["kernel_id"]], plan


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rows_of_a_workgroup_fit_its_lanes(dtype):
    ve = 4 if dtype == torch.float32 else 8
    for elements in (1 << 22, 1 << 23, 1 << 25):
        for L in list(range(ve, 70)) + [99, 127, 255, 333, 400, 500, 1000, 1001, 1401, 2041, 2047, 2730, 4001, 4093]:
            for is_bwd in (False, True):
                name, p = _kernel((elements // L + 1, L), dtype, is_bwd)
                if "packed" not in name:
                    continue
                slack = ve - 1 if L % ve else 0
                assert 2 <= p["tasks"] and p["tasks"] * L + slack <= p["waves"] * 128 * ve, (L, p)
                assert (p["grid"] - 1) * p["tasks"] < elements // L + 1 <= p["grid"] * p["tasks"], (L, p)
                assert (p["family"], p["workspace_bytes"], p["tail_rows"]) == (nat.FAMILY_TILE, 0, 0)


def test_calls_that_stay_where_they_were():
    big = 1 << 23
    for L in (150, 333, 700):
        assert "packed" in _kernel((big // L, L))[0]
        assert "packed" not in _kernel(((1 << 21) // L, L))[0]                 # little work
        assert "packed" not in _kernel((big // L, L), strides=(L + 1, 1))[0]                         # gaps between the rows
        assert "packed" not in _kernel((big // L, L), strides=(1, big // L))[0]                      # strided scan axis
    for L in (64, 100, 121, 256, 512, 2048):  # lanes that share a row; rows that fill their own workgroup
        assert "packed" not in _kernel((big // L, L))[0], L
    for L in (3, 8191, 8193):
        assert "packed" not in _kernel((big // L, L))[0], L
    t = torch.empty(big + 8)[1:1 + big // 333 * 333].view(-1, 333)  # a base inside a slot
    assert "packed" in nat.kernel_table()[nat.plan(t)["kernel_id"]]
    for family in (nat.FAMILY_TILE, nat.FAMILY_FLAT):  # a caller who names the family gets what it always meant
        p = nat.plan(torch.empty(big // 150, 150), False, False, nat.Tuning(family))
        assert "packed" not in nat.kernel_table()[p["kernel_id"]]
