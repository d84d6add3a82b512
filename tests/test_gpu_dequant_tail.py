"""Q8_0 dequantisation around the 128-block groups of the 16-byte path, and
off 16-byte alignment (the byte path), bit for bit; and at the sizes where the
two paths change over."""
import numpy as np
import pytest
import torch

from gemma_amd import capi, gguf
from oracle import oracle as orc

from gpu_util import dev, say, stream

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [1, 2, 7, 8, 127, 128, 129, 255, 1000])
@pytest.mark.parametrize("src_off,out_off", [(0, 0), (1, 0), (2, 0), (8, 0), (0, 4), (0, 8)])
def test_dequant_groups_and_alignment(gpu, nb, src_off, out_off):
    rng = np.random.default_rng(nb)
    q = rng.integers(-128, 128, size=(nb, 32)).astype(np.int8)
    codes = rng.integers(0, 0x7C00, size=nb).astype(np.uint16) | (rng.integers(0, 2, nb).astype(np.uint16) << 15)
    blocks = gguf.q8_0_blocks(codes.view(np.float16), q)
    say("dequant", nb, src_off, out_off)
    raw = np.zeros(src_off + nb * 34, np.uint8)
    raw[src_off:] = np.frombuffer(np.ascontiguousarray(blocks).tobytes(), np.uint8)
    src = dev(raw)
    n = nb * 32
    out = torch.full((n + 2 + 64,), -7.0, dtype=torch.float32, device="cuda:0")
    capi.q8_0_dequant(src.data_ptr() + src_off, out.data_ptr() + out_off, n, stream())
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    first = out_off // 4
    ref = orc.q8_0_dequant(blocks, n)
    assert np.array_equal(got[first:first + n].view(np.uint32), ref.view(np.uint32))
    assert np.all(got[:first] == -7.0) and np.all(got[first + n:] == -7.0)


# the 16-byte path takes 16 to 384 blocks and 24576 on, the byte path the rest
@pytest.mark.parametrize("nb", [15, 16, 17, 383, 384, 385, 513, 24575, 24576, 24577, 24576 + 127, 24576 + 129])
@pytest.mark.parametrize("out_off", [0, 4])
def test_dequant_where_the_paths_change(gpu, nb, out_off):
    rng = np.random.default_rng(nb)
    q = rng.integers(-128, 128, size=(nb, 32)).astype(np.int8)
    codes = rng.integers(0, 0x7C00, size=nb).astype(np.uint16) | (rng.integers(0, 2, nb).astype(np.uint16) << 15)
    blocks = gguf.q8_0_blocks(codes.view(np.float16), q)
    say("dequant", nb, out_off)
    n, first = nb * 32, out_off // 4
    out = torch.full((n + 66,), -7.0, dtype=torch.float32, device="cuda:0")
    src = dev(np.frombuffer(np.ascontiguousarray(blocks).tobytes(), np.uint8))
    capi.q8_0_dequant(src.data_ptr(), out.data_ptr() + out_off, n, stream())
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    ref = orc.q8_0_dequant(blocks, n)
    assert np.array_equal(got[first:first + n].view(np.uint32), ref.view(np.uint32))
    assert np.all(got[:first] == -7.0) and np.all(got[first + n:] == -7.0)
