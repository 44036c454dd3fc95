"""The Python layer around the entry points: workspaces and stream capture."""
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
