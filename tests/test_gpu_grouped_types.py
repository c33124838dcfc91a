"""Grouped calls over layers of any block types (the MFMA kernels' IQ1_M and
mixed-type instances): against the oracle chain and the per-token layer calls
within 1e-3, bit-identical reruns. Types mixed per expert and between gate/up
and down, tasks of one, two and more tiles, shapes with 1 to 20 blocks per row."""
from __future__ import annotations

import numpy as np
import pytest

import crosslane_amd as xl
from perf import cases
from tests.conftest import max_rel

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
TOL = 1e-3


def type_map(kind, E, rng):
    t = np.zeros((1, E, 3), np.int32)
    if kind == "iq1":
        t[:] = 29
    elif kind == "swapped":                # IQ2_XS gate/up, IQ2_XXS down
        t[..., :2], t[..., 2] = 17, 16
    elif kind == "split":                  # gate/up and down typed apart, every pair of types
        gu, dn = np.meshgrid([16, 17, 29], [16, 17, 29])
        for e in range(E):
            t[0, e] = (gu.flat[e % 9], gu.flat[e % 9], dn.flat[e % 9])
    else:                                  # whole experts, mostly IQ1_M
        t[:] = rng.choice([16, 17, 29], size=(1, E), p=[0.19, 0.17, 0.64])[..., None]
    return t


@pytest.mark.parametrize("kind,dim,ff,E,T,k,skew,lim", [
    ("iq1", 1024, 512, 16, 20, 4, False, 0.0), ("iq1", 4096, 3072, 24, 33, 6, False, 0.0),
    ("iq1", 256, 256, 4, 40, 2, True, 7.0), ("mixed", 4096, 3072, 32, 24, 6, False, 7.0),
    ("mixed", 5120, 2304, 20, 17, 8, False, 10.0), ("mixed", 1024, 512, 64, 13, 6, False, 0.0),
    ("mixed", 1024, 512, 64, 200, 6, True, 0.0),
    ("swapped", 1024, 768, 8, 16, 3, True, 0.0), ("split", 2048, 1024, 18, 64, 6, False, 0.0),
    ("split", 768, 4096, 9, 13, 5, False, 0.0)])
def test_grouped_types(orc, kind, dim, ff, E, T, k, skew, lim):
    print(f"[gpu-step] grouped {kind} {dim}x{ff} E={E} T={T} k={k}", flush=True)
    rng = np.random.default_rng(dim + ff + T)
    types = type_map(kind, E, rng)
    logits = rng.standard_normal((T, E)) + (np.where(np.arange(E) < 3, 4.0, 0.0) if skew else 0.0)
    ids = np.argsort(-logits, axis=1, kind="stable")[:, :k].astype(np.int32)
    w = rng.random((T, k)).astype(np.float32)
    x = rng.standard_normal((T, dim)).astype(np.float32)
    shared = rng.standard_normal((T, dim)).astype(np.float32)
    with xl.Lane(dim, ff, 1, E, types, max_picks=8, max_tokens=T, swiglu_limit=lim) as lane:
        lane.generate(seed=21)
        counts = lane.launch_counts()
        got = lane.grouped_forward(0, ids, w, x, shared)
        assert lane.launch_counts() == counts          # no per-token layer call served it
        assert np.array_equal(got.view(np.uint32), lane.grouped_forward(0, ids, w, x, shared).view(np.uint32))
        per = np.stack([lane.layer_forward(0, ids[t], w[t], x[t], shared[t]) for t in range(T)])
    assert max(max_rel(got[t], per[t]) for t in range(T)) < TOL
    for t in sorted({0, T // 2, T - 1}):
        rows = []
        for e in ids[t]:
            tt = tuple(int(v) for v in types[0, e])
            rows.append(orc.expert(tt, *orc.gen_expert(tt, 21, 0, int(e), dim, ff), dim, ff, x[t], limit=lim))
        want = orc.combine(ids[t], w[t], np.stack(rows), shared[t])
        assert max_rel(got[t], want) < TOL, (t, max_rel(got[t], want))


@pytest.mark.parametrize("dim,ff", [(1024, 512), (768, 256), (2304, 1024)])
def test_tasks_of_several_tiles(dim, ff):
    """Many pairs per expert: tasks of up to 64 pairs (1 to 4 tiles and their
    remainders) give the bits of 16-pair tasks, which the traced call keeps."""
    counts = [16, 17, 32, 33, 48, 49, 64, 65, 1, 129, 15]
    print(f"[gpu-step] tasks of several tiles {dim}x{ff}", flush=True)
    E, T = len(counts), sum(counts)
    rng = np.random.default_rng(dim)
    ids = rng.permutation(np.repeat(np.arange(E), counts)).astype(np.int32).reshape(T, 1)
    types = np.zeros((1, E, 3), np.int32)
    types[..., :2], types[..., 2] = 16, 17
    d_ids = torch.from_numpy(ids).cuda()
    d_w = torch.from_numpy(rng.random((T, 1)).astype(np.float32)).cuda()
    d_x = torch.from_numpy(rng.standard_normal((T, dim)).astype(np.float32)).cuda()
    out, traced = (torch.zeros((T, dim), dtype=torch.float32, device="cuda") for _ in range(2))
    y = torch.zeros((T, dim), dtype=torch.float32, device="cuda")
    q8x = torch.zeros(T * (dim // 256) * 292, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    with xl.Lane(dim, ff, 1, E, types, max_picks=1, max_tokens=T) as lane:
        lane.generate(seed=4)
        lane.grouped_forward_async(0, d_ids, d_w, d_x, out)
        lane.grouped_trace_async(0, d_ids, d_w, d_x, traced, q8x=q8x, y=y)
        lane.sync()
    assert float(out.abs().max()) > 0
    assert torch.equal(out.view(torch.int32), traced.view(torch.int32))


@pytest.mark.parametrize("dim,ff", [(768, 1024), (2304, 1024), (1024, 3072), (4096, 2304)])
@pytest.mark.parametrize("kind", ["iq1", "mixed", "swapped", "split"])
def test_tasks_of_several_tiles_of_any_types(kind, dim, ff):
    """The same pairs in one call, about 43 per expert (tasks of 1 to 4 tiles and their
    remainders), and in calls of 512 pairs or fewer, 8 per expert (16-pair tasks,
    other kernels): the same bits. Rows of an odd number of blocks, and of more than
    eight (whose float sums are chains of eight)."""
    counts = [16, 17, 32, 33, 48, 49, 64, 65, 1, 129, 15, 50, 63]
    print(f"[gpu-step] tasks of several tiles {kind} {dim}x{ff}", flush=True)
    E = 64
    per = np.resize(counts, E)
    T = int(per.sum())
    rng = np.random.default_rng(dim + ff)
    ids = rng.permutation(np.repeat(np.arange(E), per)).astype(np.int32).reshape(T, 1)
    types = type_map(kind, E, rng)
    d_ids, d_w, d_x = (torch.from_numpy(a).cuda() for a in (ids, rng.random((T, 1)).astype(np.float32),
                                                            rng.standard_normal((T, dim)).astype(np.float32)))
    out, parts = torch.zeros((T, dim), device="cuda"), torch.zeros((T, dim), device="cuda")
    torch.cuda.synchronize()
    with xl.Lane(dim, ff, 1, E, types, max_picks=1, max_tokens=T) as lane:
        lane.generate(seed=4)
        lane.grouped_forward_async(0, d_ids, d_w, d_x, out)
        for t in range(0, T, 512):
            n = min(512, T - t) if T - t >= 600 else T - t   # no call below the 13 tokens of the grouped kernels
            lane.grouped_forward_async(0, d_ids[t:t + n], d_w[t:t + n], d_x[t:t + n], parts[t:t + n])
            if t + n == T:
                break
        lane.sync()
    assert float(out.abs().max()) > 0
    assert int((out.view(torch.int32) != parts.view(torch.int32)).sum()) == 0


@pytest.mark.parametrize("dim,ff", [(4096, 3072), (5120, 2304), (1024, 512)])
@pytest.mark.parametrize("kind", ["iq1", "mixed"])
@pytest.mark.parametrize("T", [64, 160])     # tasks of up to 16 pairs, and of up to 64
def test_no_further_from_64_bits_than_layer_calls(monkeypatch, kind, dim, ff, T):
    """A grouped call over IQ1_M or mixed layers replaces the layer calls of its
    tokens: its tokens' errors against the same arithmetic in 64 bits (the median, which
    no moved quant of h reaches) are no larger than theirs."""
    print(f"[gpu-step] error against 64 bits {kind} {dim}x{ff} T={T}", flush=True)
    case = {"job": "grouped", "dim": dim, "ff": ff, "experts": 48, "kind": kind, "tokens": T, "picks": 6, "limit": 0.0,
            "routed": False}
    want = cases.exact(case, 1)["out"].cuda()
    err = {}
    for path in ("0", "1"):                  # layer calls, grouped kernels
        monkeypatch.setenv("XL_GROUPED_PATH", path)
        s = cases.prepare(case, 1)
        with s["lane"]:
            out = cases.run(s)["out"]
            torch.cuda.synchronize()
            err[path] = float(((out.double() - want).norm(dim=1) / want.norm(dim=1)).median())
    print(f"layer calls {err['0']:.3e}, grouped {err['1']:.3e}", flush=True)
    assert err["1"] <= err["0"]


@pytest.mark.parametrize("dim,ff,E,T,k", [
    (1024, 512, 8, 64, 8), (2048, 1024, 64, 4, 6), (2048, 1024, 64, 64, 6), (1024, 512, 64, 64, 7), (1024, 512, 224, 64, 7),
    (4096, 3072, 8, 20, 6), (256, 256, 8, 256, 8), (768, 4096, 6, 50, 4), (2304, 2048, 40, 1, 8), (1024, 512, 8, 512, 8)])
def test_plans_keep_the_bits(dim, ff, E, T, k):
    """However a call's tiles are cut (waves per workgroup, down rows per tile, pairs
    per task: by the work that the host expects), an IQ2 call has the bits of the
    traced one, which is always cut the same way."""
    print(f"[gpu-step] plans {dim}x{ff} E={E} T={T} k={k}", flush=True)
    rng = np.random.default_rng(dim + E + T)
    types = np.zeros((1, E, 3), np.int32)
    types[..., :2], types[..., 2] = 16, 17
    ids = np.stack([rng.permutation(E)[:k] for _ in range(T)]).astype(np.int32)
    if T > 1:
        ids[T // 2] = -1                        # a token without a valid pick: the shared row alone
    args = [torch.from_numpy(a).cuda() for a in (ids, rng.random((T, k)).astype(np.float32),
                                                 rng.standard_normal((T, dim)).astype(np.float32))]
    out, traced = torch.zeros((T, dim), device="cuda"), torch.zeros((T, dim), device="cuda")
    q8x = torch.zeros(T * (dim // 256) * 292, dtype=torch.uint8, device="cuda")
    shared = torch.from_numpy(rng.standard_normal((T, dim)).astype(np.float32)).cuda()
    torch.cuda.synchronize()
    with xl.Lane(dim, ff, 1, E, types, max_picks=8, max_tokens=T) as lane:
        lane.generate(seed=9)
        lane.grouped_forward_async(0, *args, out, shared=shared)
        lane.grouped_trace_async(0, *args, traced, q8x=q8x, shared=shared)
        if T > 1:
            with pytest.raises(xl.XLError, match="expert id"):
                lane.sync()
        else:
            lane.sync()
    assert int((out.view(torch.int32) != traced.view(torch.int32)).sum()) == 0
    assert T == 1 or int((out[T // 2] != shared[T // 2]).sum()) == 0
    assert float(out.abs().max()) > 0


@pytest.mark.parametrize("gu,dn", [(16, 17), (29, 17), (16, 29), (29, 29)])
def test_only_iq1_banks_have_its_workspace(gu, dn):
    """The sums that IQ1_M's MFMAs take are allocated with a bank that has IQ1_M
    matrices of that role, and with no other."""
    dim, ff, E, T, k = 1024, 512, 8, 64, 4
    types = np.zeros((1, E, 3), np.int32)
    types[..., :2], types[..., 2] = gu, dn
    tiles = T * k // 16 + E + 1
    with xl.Lane(dim, ff, 1, E, np.full((1, E, 3), 16, np.int32), max_picks=k, max_tokens=T) as lane:
        least = lane.info()["workspace_bytes"]
    with xl.Lane(dim, ff, 1, E, types, max_picks=k, max_tokens=T) as lane:
        assert lane.info()["workspace_bytes"] - least == 4 * tiles * (dim * (gu == 29) + ff * (dn == 29))
