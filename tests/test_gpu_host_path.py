"""The Python layer around the entry points: workspaces and stream capture."""
import numpy as np
import pytest

from .test_gpu_parity import _say

pytestmark = pytest.mark.gpu


def test_workspace_of_a_device_without_index(gpu):
    """torch.device("cuda") names the current device, as in torch's own calls."""
    import torch
    import llima_amd
    _say("workspace of a device without index")
    dev = torch.device("cuda")
    buf = llima_amd.Workspace.get(dev, "host path test", 1000)
    assert buf.numel() >= 1000 and buf.device.index == torch.cuda.current_device()
    assert llima_amd.Workspace.get(dev, "host path test", 500).data_ptr() == buf.data_ptr()


def test_scoring_under_capture_raises_and_leaves_scoring_usable(gpu):
    """Scoring checks device-resident targets on the host, so it cannot be
    captured: it raises before it records anything, and neither the capture's
    other work nor later scoring calls are spoiled."""
    import torch
    import llima_amd
    _say("scoring under capture")
    g = torch.Generator(device=gpu).manual_seed(3)
    x = torch.randn(4, 9000, device=gpu, generator=g)
    hid = torch.randn(4, 256, device=gpu, generator=g).to(torch.bfloat16)
    w = torch.randn(512, 256, device=gpu, generator=g).to(torch.bfloat16)
    tg = torch.randint(0, 512, (4,), device=gpu, generator=g).to(torch.int32)
    calls = [lambda: llima_amd.score_logits(x, tg), lambda: llima_amd.lm_head_score(hid, w, tg)]
    y = torch.zeros(4, device=gpu)
    cap = torch.cuda.Stream(gpu)
    for call in calls:
        ref = [t.cpu().numpy() for t in call()]
        cap.wait_stream(torch.cuda.current_stream(gpu))
        with torch.cuda.stream(cap):
            call()
        torch.cuda.synchronize(gpu)
        y.zero_()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=cap):
            with pytest.raises(RuntimeError):
                call()
            y.add_(1.0)
        for _ in range(3):
            graph.replay()
        torch.cuda.synchronize(gpu)
        assert (y.cpu().numpy() == 3.0).all()
        for _ in range(3):
            assert all(np.array_equal(a, t.cpu().numpy()) for a, t in zip(ref, call()))
