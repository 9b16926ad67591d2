"""Device memory of an open model.  Prompt batches of the Q4_K model convert
their activations into memory the model has anyway (the attention's score
rows), so that opening it takes the weights, their tiled copy and the state of
its context and nothing more: 31446 MiB at 512 positions.  A buffer of its own
for the longest batch would be 136 MiB more."""
import pytest

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(300)]


def test_open_model_memory(device):
    import torch
    from conftest import synthetic_model
    from q38hip.model import Model
    path = synthetic_model("q4km")
    torch.zeros(1, device=device)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    with Model.open(path, 512):
        used = (before - torch.cuda.mem_get_info()[0]) / 2**20
    print("open model: %.1f MiB" % used, flush=True)
    assert 31000 < used < 31500
