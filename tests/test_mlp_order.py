"""A prediction queued on a caller's stream uses the weights and biases of the time of the call: new
parameters, set while it has not started, wait for it."""
import os

import numpy as np
import pytest
import torch  # before the ddx library: one HIP runtime for both
from conftest import ROOT

pytestmark = pytest.mark.gpu
MODEL = os.path.join(ROOT, "dds_gpu_amd", "models", "tricknet.bin")


@pytest.mark.parametrize("n", [40, 700])
def test_parameters_wait_for_queued_predictions(ddx, n):
    hands = ddx.random_deals(77, n, 13)
    d_hands = torch.from_numpy(hands.view(np.int64)).cuda()
    d_seeds = torch.zeros((n, 20), dtype=torch.uint8, device="cuda")
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with_old, other = ddx.TrickNet(path=MODEL), ddx.TrickNet(seed=5)
    want, new = with_old.predict(hands), other.predict(hands)
    p = other.params()
    assert (want != new).mean() > 0.1
    print("delay, prediction, new parameters:", n, flush=True)
    with torch.cuda.stream(side):
        torch.cuda._sleep(20_000_000)
    with_old.predict_device(d_hands.data_ptr(), n, d_seeds.data_ptr(), stream=side.cuda_stream)
    assert not side.query()  # it has not started
    with_old.set_params(p)
    side.synchronize()
    assert np.array_equal(d_seeds.cpu().numpy(), want)
    assert np.array_equal(with_old.params(), p) and np.array_equal(with_old.predict(hands), new)
    with_old.close()
    other.close()
