"""
The mse scale search at the quotients where a reciprocal product and the rounded division may round
to different integers: weights at half-integer multiples of a candidate scale and one float to
either side, for int4 and int8, bit-exact against the oracle.
"""

import numpy as np
import pytest
import torch

import oracle as O
from moelab_hip.quant import quantize

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,gs", [(4, 64), (4, 34), (8, 64), (8, 6)])
def test_mse_at_half_integers(dev, bits, gs):
    rng = np.random.default_rng(bits * 100 + gs)
    qmax = 7 if bits == 4 else 127
    rows, ng = 96, 8
    w = np.zeros((rows, ng * gs), np.float32)
    for r in range(rows):
        for g in range(ng):
            # a scale of the search's grid (absmax / qmax * (1 - 0.02 i), rounded to fp16) and ties of it
            amax = np.float32(np.exp2(rng.integers(-8, 3)) * rng.uniform(1, 2))
            s = np.float32(np.float16(np.float32(amax / np.float32(qmax)) * np.float32(1.0 - 0.02 * rng.integers(0, 16))))
            k = rng.integers(-qmax, qmax, gs).astype(np.float32) + np.float32(0.5)
            v = (k * s).astype(np.float32)
            side = rng.integers(0, 3, gs)
            v = np.where(side == 1, np.nextafter(v, np.float32(np.inf)), np.where(side == 2, np.nextafter(v, np.float32(-np.inf)), v))
            v = np.clip(v, -amax, amax).astype(np.float32)
            v[rng.integers(0, gs)] = amax
            w[r, g * gs:(g + 1) * gs] = v
    q, s = quantize(torch.from_numpy(w).to(dev), bits, gs, "mse")
    q_ref, s_ref = O.quantize(w, bits, gs, "mse")
    assert np.array_equal(s.cpu().numpy().view(np.uint16), np.asarray(s_ref).view(np.uint16))
    assert np.array_equal(q.cpu().numpy().view(np.uint8), np.asarray(q_ref).view(np.uint8))


@pytest.mark.parametrize("prec,scale", [("int4", "mse"), ("int4", "absmax"), ("int8", "mse"), ("int8", "absmax"),
                                        ("fp8", None), ("fp16", None)])
@pytest.mark.parametrize("H,I", [(256, 128), (192, 100), (130, 66)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_encode_record_from_16_bit_weights(dev, prec, scale, H, I, dtype):
    """A record encoded from 16-bit weights (widened in the quantiser) into a used buffer: the bytes of
    the same record encoded from their float32 copies into a fresh one, its padding zero."""
    from moelab_hip.store import encode_record_, record_layout

    lay = record_layout(prec, H, I, 64, scale=scale)
    g = torch.Generator().manual_seed(H + I)
    gu = (torch.randn(2 * I, H, generator=g) * 0.02).to(dtype).to(dev)
    dn = (torch.randn(H, I, generator=g) * 0.02).to(dtype).to(dev)
    ref = encode_record_(lay, torch.zeros(lay["record_bytes"], dtype=torch.uint8, device=dev), gu.float(), dn.float())
    got = encode_record_(lay, torch.full((lay["record_bytes"],), 0xA5, dtype=torch.uint8, device=dev), gu, dn)
    # a view with other strides: made contiguous first
    got2 = encode_record_(lay, torch.full_like(got, 0x5A), gu.t().contiguous().t(), dn)
    assert torch.equal(ref, got) and torch.equal(ref, got2)
