"""CPU: the line between the batched GEMVs and the MFMA tiles, at the measured sizes on either side."""

import pytest

from moelab_hip.prefill import gemv_pays
from moelab_hip.store import record_layout


@pytest.mark.parametrize("kind,H,I,E,k,shared,gemv,tiles", [
    ("int4", 2048, 1024, 64, 8, False, 8, 24), ("int4", 2048, 768, 128, 8, False, 24, 40),
    ("int4", 2048, 512, 512, 10, True, 64, 96), ("int8", 2048, 1024, 64, 8, False, 12, 24),
    ("fp8", 2048, 512, 512, 10, True, 48, 64), ("fp8", 2048, 1024, 64, 8, False, 8, 16),
    ("fp16", 2048, 1024, 64, 8, False, 16, 24), ("bf16", 2048, 1024, 16, 4, False, 16, 32),
    ("int4", 512, 256, 16, 4, False, 64, 1024),
])
def test_the_line(kind, H, I, E, k, shared, gemv, tiles):
    rb = record_layout(kind, H, I, 64)["record_bytes"]
    assert gemv_pays(1, k, E, shared, kind, rb) and gemv_pays(gemv, k, E, shared, kind, rb)
    assert not gemv_pays(tiles, k, E, shared, kind, rb)
    side = [gemv_pays(T, k, E, shared, kind, rb) for T in range(1, 1100)]
    assert side == sorted(side, reverse=True)  # one line: never back to the GEMVs with more tokens
