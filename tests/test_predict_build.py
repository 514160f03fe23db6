"""Batch prediction is built in two MFMA forms: accumulators in ordinary registers (few rows) and in the accumulator
file (many). A flag meant for the training kernel alone once left only the first, and 500 000 rows took 6 % longer."""
from test_spill_masks import LIB, code_objects, functions


def test_prediction_has_both_forms(mm, tmp_path):
    mm.lib()
    found = []
    for co in code_objects(LIB, str(tmp_path)):
        for name, body in functions(co):
            if "predict_kernel" in name:
                found.append(sum(ins.startswith("v_accvgpr_read") for _, ins, _ in body))
    assert len(found) == 2 and min(found) == 0 and max(found) > 0, found
