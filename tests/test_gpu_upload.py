"""Host arrays on their way to the device."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_uploads_keep_what_the_array_held_at_the_call():
    """Uploads behind work that keeps the stream busy, from arrays that are changed and given back at once, one after the other and
    on a second stream: each tensor holds what its array held."""
    from inferx_amd import ops
    from inferx_amd.engine.runtime import Runtime
    rt = Runtime("bfloat16")
    busy = torch.randn(2048, 2048, device="cuda:0")
    side = torch.cuda.Stream()
    got, want = [], []
    for i in range(60):
        busy = busy @ busy * 1e-3
        a = np.arange(i, i + 5 + 300 * (i % 7), dtype=np.int32 if i % 2 else np.int64)
        want.append(a.copy())
        if i % 3 == 2:
            with torch.cuda.stream(side):
                got.append(ops.upload(a, rt.device))
        else:
            got.append(ops.upload(a[::1], rt.device))
        a[:] = -1
    strided = np.arange(40, dtype=np.int32).reshape(4, 10)[:, ::2]
    got.append(ops.upload(strided, rt.device))
    want.append(strided)
    got.append(ops.upload(np.empty(0, np.int32), rt.device))
    want.append(np.empty(0, np.int32))
    torch.cuda.synchronize()
    for g, w in zip(got, want):
        assert g.device == rt.device and np.array_equal(g.cpu().numpy(), w)
