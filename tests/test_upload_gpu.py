"""skv_upload_i32: small host arrays on the device, in stream order, the host
array free to change once the call has returned."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 255, 256, 257, 4096, 4097])
def test_upload_i32(n):
    from simple_llm_amd import _lib
    host = np.arange(n, dtype=np.int32) * 7919 - 2 ** 30
    want = host.copy()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        got = _lib.upload_i32(host, torch.device("cuda", 0), stream.cuda_stream)
        host[:] = -1
        got = got.cpu().numpy()
    assert got.dtype == np.int32 and (got == want).all()
