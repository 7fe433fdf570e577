"""A batch whose launch would hold exactly 2^32 work-items, HIP's limit (65536 hafnians
of side 28, 1024 workgroups each), runs in two launches and returns the values of
its matrices alone."""
import numpy as np
import pytest

from conftest import rng_symmetric

pytestmark = pytest.mark.gpu


def test_hafnians_at_the_launch_limit():
    import torch
    from gbskernels_amd import _lib
    L = _lib.lib()
    N, B, base = 28, 65537, 61
    print(f"haf N={N} B={B}", flush=True)
    A = torch.from_numpy(rng_symmetric(base, N, 2828, 0.2)).cuda()
    stack = A.repeat((B + base - 1) // base, 1, 1)[:B].contiguous()
    st = torch.cuda.current_stream().cuda_stream

    def run(x):
        n = x.shape[0]
        out = torch.full((n,), float("nan"), dtype=torch.complex128, device="cuda")
        ws = torch.empty(int(L.gbs_workspace_bytes(1, 0, N, n)), dtype=torch.uint8, device="cuda")
        _lib.check(L.gbs_eval_device(1, 0, x.data_ptr(), N, n, out.data_ptr(), None, ws.data_ptr(), ws.numel(), st),
                   "gbs_eval_device")
        torch.cuda.synchronize()
        return out.cpu().numpy()

    few, many = run(A), run(stack)
    assert np.all(np.isfinite(few))
    assert np.array_equal(many, np.tile(few, (B + base - 1) // base)[:B])
