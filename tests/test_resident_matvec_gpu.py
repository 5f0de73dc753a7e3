"""Many-token products on both sides of the rule that gives them the resident
form (256 and 1024 row tiles, rows of 4, 32 and 40 blocks, 16 tokens) against
the CPU oracle: ragged last tiles, rows of one block, tails of 1-3 blocks, rows
that two token groups no longer fit, at the edges of the 16-token groups."""
import numpy as np
import pytest

from llm_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qt", [synth.Q4_0, synth.Q4_1, synth.Q8_0])
@pytest.mark.parametrize("rows,k", [(40, 32), (100, 128), (4080, 896), (4081, 896), (4100, 160), (4090, 1024),
                                    (4096, 1056), (16368, 96), (16369, 160), (16384, 1280), (16390, 1312),
                                    (16384, 2592)])
def test_tall_products(gpu, qt, rows, k):
    from llm_amd import kernels
    from oracle import cpuref
    rng = np.random.default_rng([qt, rows, k])
    raw = synth.quant_blocks(qt, rows, k, rng)
    m = kernels.QMat(qt, rows, k, raw)
    x = rng.standard_normal((64, k), dtype=np.float32)
    x[3] *= 1e-20
    x[4] = 0
    y0 = rng.standard_normal((64, rows), dtype=np.float32)
    want = np.stack([cpuref.matvec(qt, raw, rows, k, x[t]) for t in range(64)])
    for n in (5, 16, 17, 33, 64):
        print(f"type {qt} {rows}x{k}, {n} tokens", flush=True)
        y = m.gemv(x[:n])
        for t in range(n):  # f32 sums of k products in another order: sqrt(k) 2^-24, about 3e-6 at the longest
            assert np.max(np.abs(y[t] - want[t])) <= 1e-5 * np.max(np.abs(want[t])), t
        z = m.gemv(x[:n], y0[:n], accumulate=True)
        assert np.array_equal(z, y0[:n] + y)  # the residual is added to the same product
    m.close()
