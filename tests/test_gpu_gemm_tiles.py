"""The GEMM's launch shapes (row-blocks and operand blocks a wave, waves along n, K slices) at their edges, for both
operand forms: FP32 rows (two f16 parts) and BF16 rows (one part, exact for BF16 values), against the FP64 closed form.

Bar: max |err| / RMS <= 3e-5, as tests/test_gpu_gemm.py: K <= 1040 FP32 additions of exact products of 22-bit (or
exact BF16) activations, with about 1e-7 of the RMS per rounding."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = ["4,8,4,1", "4,6,4,1", "4,4,4,1", "4,4,4,2", "3,4,4,2", "2,4,4,2", "4,2,4,2", "2,2,4,2", "1,4,4,2", "1,2,4,2",
          "1,2,4,4", "1,2,2,4", None]


def run(hip, pkg, wl, ws, m, k, bf16, rng, y_offset=0):
    bits = wl.f32_to_bf16(rng.standard_normal((m, k)).astype(np.float32))
    x = wl.bf16_to_f32(bits) if bf16 else rng.standard_normal((m, k)).astype(np.float32)
    dx = hip.array(bits if bf16 else x)
    total = m * sum(w[0].shape[0] for w in ws)
    dy = hip.array(np.full(y_offset + total + 4, 7.0, np.float32))
    hip.matmul_dev([pkg.Weight(*w) for w in ws], dx, pkg.X_BF16 if bf16 else pkg.X_F32, m, dy, y_offset)
    y = dy.numpy()
    dx.free()
    dy.free()
    assert (y[:y_offset] == 7).all() and (y[y_offset + total:] == 7).all()   # nothing outside the outputs
    off = y_offset
    for w in ws:
        n = w[0].shape[0]
        exact = x.astype(np.float64) @ wl.decode_nvfp4(*w).astype(np.float64).T
        got = y[off:off + m * n].reshape(m, n)
        err = np.max(np.abs(got - exact)) / np.sqrt(np.mean(exact ** 2))
        assert err <= 3e-5, (n, err)
        off += m * n


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("shape", SHAPES)
def test_shapes_at_their_edges(hip, pkg, wl, monkeypatch, shape, bf16):
    if shape:
        monkeypatch.setenv("XTG_GEMM_SHAPE", shape)
    rng = np.random.default_rng(31)
    # one k-tile (fewer than the slices), a partial last one, 9 tiles over 2 and 4 slices; odd outputs (no float4
    # stores), a partial row-block, more than one n-tile; row counts around a group, a 16-row block and an m-tile
    for ns, k, ms in (([129], 1040, (9, 33, 130)), ([260, 68], 128, (16, 65)), ([17, 512, 5], 272, (15, 17))):
        ws = [wl.nvfp4_weight(rng, n, k) for n in ns]
        for m in ms:
            run(hip, pkg, wl, ws, m, k, bf16, rng, y_offset=m % 3)


@pytest.mark.parametrize("m", [9, 16, 17, 100])
def test_bf16_rows_of_every_magnitude(hip, pkg, wl, m):
    """Rows of very different sizes, with values 2^-30 of the row's largest, zeros and a zero row."""
    rng = np.random.default_rng(m)
    k = 512
    x = rng.standard_normal((m, k)).astype(np.float32) * np.exp2(rng.integers(-30, 1, (m, k))).astype(np.float32)
    x *= np.exp2(rng.integers(-60, 60, (m, 1))).astype(np.float32)
    x[rng.random((m, k)) < 0.1] = 0
    x[m // 2] = 0
    bits = wl.f32_to_bf16(x)
    w = wl.nvfp4_weight(rng, 200, k)
    dx, dy = hip.array(bits), hip.array(shape=(m, 200))
    hip.matmul_dev([pkg.Weight(*w)], dx, pkg.X_BF16, m, dy)
    y = dy.numpy().astype(np.float64)
    exact = wl.bf16_to_f32(bits).astype(np.float64) @ wl.decode_nvfp4(*w).astype(np.float64).T
    rms = np.sqrt(np.mean(exact ** 2, axis=1, keepdims=True))
    assert (y[m // 2] == 0).all()
    assert np.max(np.abs(y - exact) / np.where(rms > 0, rms, 1)) <= 3e-5
