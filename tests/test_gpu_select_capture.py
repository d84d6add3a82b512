"""The selector entry points on a stream that is being captured: refused with
GG_ERR_HIP before anything is recorded, the caller's capture and the stream
stay usable."""
import ctypes

import pytest
import torch

from gemma_amd import capi

from gpu_util import say

pytestmark = pytest.mark.gpu
GG_ERR_HIP = -3
THREAD_LOCAL, RELAXED = 1, 2


def _hip():
    """The HIP runtime that this process already runs on."""
    with open("/proc/self/maps") as f:
        return ctypes.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))


@pytest.mark.parametrize("entry", ["workspace", "noalloc"])
@pytest.mark.parametrize("mode", [THREAD_LOCAL, RELAXED])
def test_select_refuses_a_capturing_stream(gpu, entry, mode):
    hip, n = _hip(), 4096
    logits = torch.randn(n, device=gpu)
    best = int(logits.argmax())
    ws = torch.zeros(capi.select_workspace_size(n), dtype=torch.uint8, device=gpu)
    torch.cuda.synchronize()
    opt, out = capi.sample(0.0, 0.9, 1.0), ctypes.c_int32(-1)
    stream, graph, nodes = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_size_t()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(stream), 1) == 0

    def select():
        head = (logits.data_ptr(), n, None, ctypes.byref(opt), 0.0)
        if entry == "workspace":
            return capi.lib().gg_select_logits(*head, ws.data_ptr(), None, ctypes.byref(out), stream)
        return capi.lib().gg_select_logits_noalloc(*head, None, ctypes.byref(out), stream)

    say("select under capture", entry, mode)
    assert hip.hipStreamBeginCapture(stream, mode) == 0
    rc = select()
    assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
    assert rc == GG_ERR_HIP and out.value == -1
    assert hip.hipGraphGetNodes(graph, None, ctypes.byref(nodes)) == 0 and nodes.value == 0
    assert hip.hipGraphDestroy(graph) == 0
    assert select() == 0 and out.value == best
    assert hip.hipStreamDestroy(stream) == 0
