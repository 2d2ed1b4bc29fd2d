"""The tanh-GELU of the gate/up products (gelu_mul) value by value through af_ffn_run: gate values that are exact
fp16 scales, up 1, and a down projection that picks one activation per output."""
import numpy as np
import pytest

import oracle
from tests.test_gpu_ops import run_ffn

pytestmark = pytest.mark.gpu
H, I = 32, 1024  # block r of the 1,024 activations holds one, for output r


def one_weight(rows, columns, at):
    """Q4_0 matrix of zeros but for row: (column, scale, code)."""
    m = np.zeros((rows, columns // 32, 18), np.uint8)
    m[:, :, 2:] = 0x88
    for r, (c, d, n) in at.items():
        b, j = c // 32, c % 32
        m[r, b, :2] = np.frombuffer(np.float16(d).tobytes(), np.uint8)
        m[r, b, 2 + j % 16] = (0x80 | n) if j < 16 else (n << 4 | 0x08)
    return m.ravel()


def gelu(values):
    """Outputs of the FFN for up to 31 gate values (rows 1 on: x is zero there)."""
    x = np.zeros(H, np.float32)
    x[0] = 1.0
    pre = np.zeros(H, np.float32)
    w = np.float32(np.sqrt(1.0 / H + 1e-6))
    while np.float32(oracle.rmsnorm(np.where(np.arange(H) == 0, w, 0), 1e-6, x)[0]) < 1.0:
        w = np.nextafter(w, np.float32(1.0))
    pre[0] = w  # the normed input is 1 in channel 0 exactly
    assert np.float32(oracle.rmsnorm(pre, 1e-6, x)[0]) == 1.0
    gate = one_weight(I, H, {32 * (r + 1): (0, v, 9) for r, v in enumerate(values)})
    up = one_weight(I, H, {32 * (r + 1): (0, 1.0, 9) for r in range(len(values))})
    down = one_weight(H, I, {r + 1: (32 * (r + 1), 1.0, 9) for r in range(len(values))})
    return run_ffn(pre, gate, up, down, H, I, x)[1:len(values) + 1]


def exact(v):
    """0.5 v (1 + tanh z) without its cancellation and v times its derivative, in extended precision."""
    v = v.astype(np.longdouble)
    c = np.sqrt(np.longdouble(2) / np.longdouble("3.14159265358979323846264338327950288"))
    z, dz = c * (v + np.longdouble(0.044715) * v ** 3), c * (1 + 3 * np.longdouble(0.044715) * v ** 2)
    with np.errstate(over="ignore", invalid="ignore"):
        e = np.exp(-2 * z)
        f = v / (1 + e)
        return f, np.nan_to_num(f * (1 + 2 * v * dz * e / (1 + e)))


def test_gelu_values():
    """Magnitudes from 2^-14 to 65,504 of both signs, with the range where the result leaves the floats (gates below
    about -10) and both saturations: within one ulp of the value plus what one ulp of the gate makes (the gate is a
    float sum; 2^-126 absolute, the smallest normal float, below which the digits of the down projection's
    input end)."""
    mag = np.concatenate([np.exp2(np.linspace(-14, 15.99, 180)), np.linspace(0.05, 14, 190)]).astype(np.float16)
    values = np.concatenate([mag, -mag, np.float16([0.0, 65504.0, -65504.0])])
    got = np.concatenate([gelu(values[i:i + 31]) for i in range(0, values.size, 31)])
    ref, slope = exact(values)
    err = np.abs(got.astype(np.longdouble) - ref)
    bound = np.maximum((np.abs(ref) + np.abs(slope)) * 2.0 ** -23, 2.0 ** -126)
    worst = (err / bound).argmax()
    print(f"worst {float(err[worst] / bound[worst]):.3f} of the bound at gate {values[worst]}", flush=True)
    assert (err <= bound).all(), (values[worst], got[worst], ref[worst])
    assert got[values == -65504.0] == 0.0 and got[values == 65504.0] == 65504.0
