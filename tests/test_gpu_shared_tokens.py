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
    ((12, 14, 8), 2304, 256, 65, 0.0),
    # three to eight tokens on both sides of the line to the row kernels
    ((12, 12, 8), 768, 2048, 3, 10.0), ((13, 13, 14), 5120, 256, 3, 0.0), ((13, 13, 14), 4096, 512, 3, 0.0),
    ((8, 8, 8), 1024, 512, 3, 0.0), ((14, 14, 14), 512, 512, 4, 7.0), ((14, 14, 14), 768, 512, 4, 0.0),
    ((12, 12, 12), 256, 256, 8, 0.0), ((12, 12, 12), 256, 256, 9, 0.0)])
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


@pytest.mark.parametrize("T", [3, 16, 33, 512])
def test_a_sub_block_of_nans_stays_nan(T):
    """32 gate rows whose scales are NaN make one per-32 block of h NaN in all its
    values, and with it the block's scale and every output, as in a single call; NaNs
    beside finite values of h take no part in the block's maximum."""
    print(f"[gpu-step] shared FFN, NaN rows, T={T}", flush=True)
    dim, ff = 256, 2048
    for rows in (32, 31):                # the whole block; one finite value in it
        mats = [dense_matrix(8, *((ff, dim) if r < 2 else (dim, ff)), seed=r).copy() for r in range(3)]
        mats[0].reshape(ff, dim // 32, 34)[64:64 + rows, :, :2] = np.frombuffer(np.float16("nan").tobytes(), np.uint8)
        mats = [dev(m) for m in mats]
        dx = dev(np.random.default_rng(T).standard_normal((T, dim)).astype(np.float32))
        work = torch.empty(xl.shared_work_bytes(dim, ff, T), dtype=torch.uint8, device="cuda")
        out, one = torch.zeros((T, dim), device="cuda"), torch.zeros(dim, device="cuda")
        torch.cuda.synchronize()
        with xl.Lane(dim, 256, 1, 1, np.full((1, 1, 3), 29, np.int32)) as lane:
            lane.shared_forward_async((8, 8, 8), *mats, ff, dx, out, work)
            for t in (0, T - 1):
                lane.shared_forward_async((8, 8, 8), *mats, ff, dx[t], one, work)
                lane.sync()
                assert bool(torch.isnan(one).all()) == (rows == 32)
                assert int((torch.isnan(out[t]) != torch.isnan(one)).sum()) == 0, (rows, t)
                assert rows == 32 or int((out[t].view(torch.int32) != one.view(torch.int32)).sum()) == 0, (rows, t)
