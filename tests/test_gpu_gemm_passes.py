"""
The MFMA launches' work units and K loops at their edges: experts with 1 to 257 tokens (whole and
partial 32-token tiles, one to three passes) at 64- and at 128-token passes, d_ff of one chunk, an
odd number of chunks, an even one, and more than one factor segment, for every record precision
and both activation dtypes, against the oracle's layer.
"""

import numpy as np
import pytest
import torch

import oracle as O
from moelab_hip.policy import PrecisionPolicy
from moelab_hip.prefill import GroupedLayer
from test_gpu_batch import _mats, _store
from test_gpu_parity import assert_layer_close

pytestmark = pytest.mark.gpu

# tokens of each expert; the mean (>= 48 or not) decides the tokens per pass
COUNTS = {"64": [1, 0, 31, 33, 64, 65, 129] + [0] * 9, "128": [128, 129, 31, 257, 96]}


@pytest.mark.parametrize("I", [128, 384, 512, 1280])
@pytest.mark.parametrize("tok", list(COUNTS))
@pytest.mark.parametrize("prec,dtype", [("int4", torch.float16), ("int4", torch.bfloat16), ("int8", torch.float16),
                                        ("fp8", torch.bfloat16), ("fp16", torch.float16), ("bf16", torch.bfloat16)])
def test_passes_and_chunks(dev, prec, dtype, tok, I):
    H, counts = 512, COUNTS[tok]
    E, T = len(counts), sum(counts)
    st = _store(dev, [prec], H, I, E, 31)
    g = torch.Generator().manual_seed(I + len(counts))
    idx = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(T, generator=g)].view(T, 1)
    w = torch.rand(T, 1, generator=g).float() + 0.05
    x = torch.randn(T, H, generator=g).to(dtype)
    gl = GroupedLayer(st, 1, T, PrecisionPolicy("lo"), dtype, gemv_tokens=0)
    out = torch.zeros(T, H, dtype=dtype, device=dev)
    gl.layer(0, x.to(dev), out, idx.to(dev), w.to(dev))
    torch.cuda.synchronize()
    assert gl.miss.item() == 0
    mats = {e: _mats(st, prec, 0, e) for e in range(E) if counts[e]}
    ref = O.moe_layer_grouped(x.float().numpy(), idx.numpy(), w.numpy().astype(np.float64), lambda e: mats[e])
    assert_layer_close(out.float().cpu().numpy(), ref, dtype)


@pytest.mark.parametrize("I", [384, 512])
@pytest.mark.parametrize("tok", list(COUNTS))
@pytest.mark.parametrize("hi", ["fp16", "bf16", "int8"])
def test_two_precisions(dev, hi, tok, I):
    """Experts of both precisions in one batch: 16-bit + int4 in one launch, the odd number of int4
    chunks (I = 384) and int8 + int4 in a launch each."""
    H, counts = 512, COUNTS[tok]
    E, T = len(counts), sum(counts)
    st = _store(dev, [hi, "int4"], H, I, E, 37)
    g = torch.Generator().manual_seed(I + len(counts))
    idx = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(T, generator=g)].view(T, 1)
    w = torch.where(idx % 3 == 0, 0.8, 0.2).float()  # every third expert's tokens vote for the first precision
    x = torch.randn(T, H, generator=g).half()
    gl = GroupedLayer(st, 1, T, PrecisionPolicy("weight", t1=0.5, upgrade=False), x.dtype, gemv_tokens=0)
    out = torch.zeros(T, H, dtype=x.dtype, device=dev)
    gl.layer(0, x.to(dev), out, idx.to(dev), w.to(dev))
    torch.cuda.synchronize()
    info = gl.info[0].cpu().tolist()
    assert [info[e] for e in range(E) if counts[e]] == [0 if e % 3 == 0 else 1 for e in range(E) if counts[e]]
    mats = {e: _mats(st, hi if e % 3 == 0 else "int4", 0, e) for e in range(E) if counts[e]}
    ref = O.moe_layer_grouped(x.float().numpy(), idx.numpy(), w.numpy().astype(np.float64), lambda e: mats[e])
    assert_layer_close(out.float().cpu().numpy(), ref, x.dtype)
