"""
The batch decision of more tokens than one workgroup levels by itself (their levels are made over
the whole chip, the decision's launch tallies them a pair per thread): the sizes around that line
and around the pairs held in LDS (4096), against moehip_batch_levels + moehip_dispatch +
moehip_batch_vote, every output bit-exact.
"""

import ctypes

import numpy as np
import pytest
import torch

from moelab_hip import _lib
from moelab_hip.policy import PrecisionPolicy

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,shared,T", [(64, False, 64), (64, False, 65), (128, True, 65), (64, False, 512),
                                        (512, True, 455), (512, True, 456), (1023, True, 700)])
@pytest.mark.parametrize("mode", ["hobbit", "weight"])
def test_batch_decide_many_tokens_matches_steps(dev, E, shared, T, mode):
    k, P = 8, 2
    ks, EA = (k + 1, E + 1) if shared else (k, E)
    g = np.random.default_rng(E + T)
    idx = np.argsort(g.random((T, E)), axis=1)[:, :k].astype(np.int64)
    w = (g.random((T, k)) ** 2 + 0.01).astype(np.float32)
    if shared:
        idx = np.concatenate([idx, np.full((T, 1), E, np.int64)], 1)
        w = np.concatenate([w, g.random((T, 1)).astype(np.float32)], 1)
    pol = PrecisionPolicy("hobbit", t1=0.5, t2=0.85) if mode == "hobbit" else PrecisionPolicy("weight", t1=0.3)
    cpol = pol.device_policy(0)
    rtab = torch.from_numpy(np.where(g.random((P, E)) < 0.8, (np.arange(P * E).reshape(P, E) + 1) * 4096, 0)).to(dev)
    srec = (ctypes.c_int64 * P)(*[(1 << 40) + 4096 * p for p in range(P)])
    offs = torch.tensor([[0, 8, 16, 24], [0, 64, 128, 192]], dtype=torch.int64, device=dev)
    planned = torch.ones(P, dtype=torch.int32, device=dev)
    lv2p = (ctypes.c_int * 3)(0, 1, 1)
    idx_d, w_d = torch.from_numpy(np.ascontiguousarray(idx)).to(dev), torch.from_numpy(np.ascontiguousarray(w)).to(dev)
    st, hv = _lib.stream_of(dev), float(pol.hi_vote)

    def bufs():
        i32 = lambda *n: torch.full(n, -7, dtype=torch.int32, device=dev)  # noqa: E731
        return dict(levels=i32(T * ks), skip=torch.full((T * ks,), 9, dtype=torch.uint8, device=dev), counts=i32(EA),
                    offsets=i32(EA + 1), sorted_pos=i32(T * ks), rank=i32(T * ks),
                    tabs=torch.full((P, EA, 4), -7, dtype=torch.int64, device=dev),
                    info=torch.full((EA,), -7.0, device=dev), miss=torch.zeros(1, device=dev))

    a, b = bufs(), bufs()
    p = {n: t.data_ptr() for n, t in a.items()}
    _lib.call("moehip_batch_decide", w_d.data_ptr(), idx_d.data_ptr(), T, k, ks, ctypes.byref(cpol), p["levels"],
              p["skip"], E, 1 if shared else 0, p["counts"], p["offsets"], p["sorted_pos"], p["rank"], hv, lv2p,
              rtab.data_ptr(), srec, P, offs.data_ptr(), planned.data_ptr(), p["tabs"], p["info"], p["miss"], None, st)
    p = {n: t.data_ptr() for n, t in b.items()}
    _lib.call("moehip_batch_levels", w_d.data_ptr(), T, k, ks, ctypes.byref(cpol), p["levels"], p["skip"], st)
    _lib.call("moehip_dispatch", idx_d.data_ptr(), p["skip"], T, ks, EA, p["counts"], p["offsets"], p["sorted_pos"],
              p["rank"], st)
    _lib.call("moehip_batch_vote", p["levels"], E, 1 if shared else 0, p["offsets"], p["sorted_pos"], hv,
              ctypes.byref(cpol), lv2p, rtab.data_ptr(), srec, P, offs.data_ptr(), planned.data_ptr(), p["tabs"],
              p["rank"], p["info"], p["miss"], st)
    torch.cuda.synchronize()
    for name in a:
        assert torch.equal(a[name], b[name]), name
    # the dispatch both share: stable by expert in pair order
    keep = np.nonzero(a["skip"].cpu().numpy() == 0)[0]
    order = keep[np.argsort(idx.reshape(-1)[keep], kind="stable")]
    assert np.array_equal(a["sorted_pos"].cpu().numpy()[:order.size], order)
