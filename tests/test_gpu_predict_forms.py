"""The two forms of batch prediction (up to 348 000 rows, and beyond) give the same outputs."""
import pytest

pytestmark = pytest.mark.gpu


def test_forms_agree(mm, gpu):
    import torch

    model = mm.Surrogate(seed=7)
    few = 348_000
    g = torch.Generator(device="cuda").manual_seed(3)
    rows = torch.randn((few + 65, 17), generator=g, device="cuda")
    out = [torch.full((n, 2), -9.0, device="cuda") for n in (few, few + 1, few + 65)]
    for o in out:
        model.predict(rows[:len(o)].contiguous(), o)
    torch.cuda.synchronize()
    for o in out[1:]:
        assert torch.equal(o[:few].view(torch.int32), out[0].view(torch.int32))
    tail = torch.full((65, 2), -9.0, device="cuda")
    model.predict(rows[few:].contiguous(), tail)
    torch.cuda.synchronize()
    assert torch.equal(tail.view(torch.int32), out[2][few:].view(torch.int32))
