"""The shared-expert FFN of several tokens (the MFMA kernels of xl_shared.hip):
every token's output bit-identical to its own single-token call (the row
kernels of xl_per32.hip, themselves bit-exact against the oracle's rows), over
the four dense formats, K of one block up to one that needs several links per
chain, and token counts around the 16- and 32-token tiles."""
from __future__ import annotations

import numpy as np
import pytest

import crosslane_amd as xl
from tests.dense import dense_matrix

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


@pytest.mark.parametrize("types,dim,ff,T,lim", [
    ((13, 13, 14), 4096, 3072, 16, 0.0), ((13, 13, 14), 4096, 256, 33, 7.0), ((14, 14, 13), 256, 2304, 17, 0.0),
    ((12, 12, 8), 768, 512, 3, 10.0), ((8, 8, 12), 5120, 1280, 47, 7.0), ((14, 14, 12), 4096, 3072, 96, 0.0), ((13, 8, 14), 1024, 768, 32, 0.0),
    ((12, 14, 8), 2304, 256, 65, 0.0)])
def test_tokens_equal_single_calls(types, dim, ff, T, lim):
    print(f"[gpu-step] shared FFN types={types} dim={dim} ff={ff} T={T}", flush=True)
    rng = np.random.default_rng(dim + ff + T)
    mats = [dev(dense_matrix(t, *((ff, dim) if r < 2 else (dim, ff)), seed=r + T)) for r, t in enumerate(types)]
    x = rng.standard_normal((T, dim)).astype(np.float32)
    x[0, :32] = 0.0                      # an all-zero sub-block
    x[T - 1] *= 1e3
    with xl.Lane(dim, 256, 1, 1, np.full((1, 1, 3), 29, np.int32), swiglu_limit=lim) as lane:
        big = torch.zeros(T * dim + 1, dtype=torch.float32, device="cuda")
        dx = dev(x)
        work = torch.empty(xl.shared_work_bytes(dim, ff, T), dtype=torch.uint8, device="cuda")
        outs = []
        for off in (0, 1):               # 16-byte aligned rows, and rows that are only 4-byte aligned
            xv = torch.zeros(T * dim + 1, dtype=torch.float32, device="cuda")
            xv[off:off + T * dim] = dx.reshape(-1)
            torch.cuda.synchronize()
            lane.shared_forward_async(types, *mats, ff, xv[off:off + T * dim], big[off:off + T * dim], work)
            lane.sync()
            outs.append(big[off:off + T * dim].cpu().numpy().reshape(T, dim).copy())
        one = torch.zeros(dim, dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        for t in range(T):
            lane.shared_forward_async(types, *mats, ff, dx[t], one, work)
            lane.sync()
            want = one.cpu().numpy().view(np.uint32)
            assert np.array_equal(outs[0][t].view(np.uint32), want), t
            assert np.array_equal(outs[1][t].view(np.uint32), want), t
