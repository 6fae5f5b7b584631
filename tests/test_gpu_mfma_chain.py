"""The float32 matrix instructions are chains of fmas in the order of k, each
rounded to nearest even, subnormals, infinities and signed zeros included: the
ground on which the prompt attention (K = 4) and the outer products of the
batched kernels (K = 1) have the reference's bits."""
import ctypes as C
import ctypes.util

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

fmaf = C.CDLL(ctypes.util.find_library("m") or "libm.so.6").fmaf
fmaf.restype, fmaf.argtypes = C.c_float, [C.c_float] * 3


def values(rng, shape, kind):
    v = rng.standard_normal(shape).astype(np.float32)
    if kind == "scaled":  # products and sums over the whole range, under- and overflow too
        with np.errstate(over="ignore", under="ignore"):
            v = np.ldexp(v, rng.integers(-90, 70, shape)).astype(np.float32)
    elif kind == "subnormal":  # subnormal operands and results
        v = (rng.integers(0, 1 << 23, shape, dtype=np.uint32) |
             (rng.integers(0, 2, shape, dtype=np.uint32) << np.uint32(31))).view(np.float32).copy()
        big = rng.random(shape) < 0.5
        v[big] = rng.standard_normal(int(big.sum())).astype(np.float32)
    elif kind == "special":
        v[rng.random(shape) < 0.3] = 0.0
        v[rng.random(shape) < 0.2] = -0.0
        v[rng.random(shape) < 0.03] = np.inf
        v[rng.random(shape) < 0.03] = -np.inf
        v[rng.random(shape) < 0.01] = np.nan
    return v


@pytest.mark.parametrize("kind", ["normal", "scaled", "subnormal", "special"])
@pytest.mark.parametrize("k", [1, 4])
def test_mfma_is_an_fma_chain(hip, k, kind):
    import torch
    from gopherllm_amd import build
    n, blocks = 16, 4 // k
    rng = np.random.default_rng([k, len(kind)])
    a, b = values(rng, (n, 4, 16), kind), values(rng, (n, 4, 16), kind)
    c = values(rng, (n, blocks, 16, 16), kind)  # [tile][block][row][column]
    # registers: lane (g, c) holds rows 4g + i of column c, block after block
    creg = np.ascontiguousarray(c.reshape(n, blocks, 4, 4, 16).transpose(0, 2, 4, 1, 3)).reshape(n, 64, 4 * blocks)
    dev = [torch.from_numpy(v).cuda() for v in (a, b, creg)]
    d = torch.zeros_like(dev[2])
    fn = C.CDLL(build.PROBE_LIB).gllm_probe_mfma_f32
    fn.argtypes = [C.c_int] + [C.c_void_p] * 4 + [C.c_int, C.c_void_p]
    assert fn(k, *(t.data_ptr() for t in dev), d.data_ptr(), n, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    got = d.cpu().numpy().reshape(n, 4, 16, blocks, 4).transpose(0, 3, 1, 4, 2).reshape(n, blocks, 16, 16)
    want = np.empty_like(c)
    for t, j, r, col in np.ndindex(*c.shape):
        v = c[t, j, r, col]
        for g in range(k):
            v = fmaf(a[t, j * k + g, r], b[t, j * k + g, col], v)
        want[t, j, r, col] = v
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    bad = np.argwhere((got.view(np.uint32) != want.view(np.uint32)) & ~nan)
    assert not len(bad), (len(bad), got[tuple(bad[0])], want[tuple(bad[0])])
    if kind == "subnormal":
        assert np.any((np.abs(want) < np.finfo(np.float32).tiny) & (want != 0))
