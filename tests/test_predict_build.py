"""Batch prediction is built with the compiler's own MFMA form: its accumulators live in the accumulator file, which
leaves the ordinary registers to five waves per SIMD with their activations. The form the training kernel asks for
(ordinary registers) made 500 000 rows 6 % slower."""
from test_spill_masks import LIB, code_objects, functions


def test_prediction_keeps_its_accumulators_in_the_accumulator_file(mm, tmp_path):
    mm.lib()
    found = []
    for co in code_objects(LIB, str(tmp_path)):
        for name, body in functions(co):
            if "predict_kernel" in name:
                found.append(sum(ins.startswith("v_accvgpr_read") for _, ins, _ in body))
    assert len(found) == 1 and found[0] > 0, found
