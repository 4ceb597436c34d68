"""GPU kernels at the sizes where their variants meet: edges of tiles, remainders, the smallest and
largest size of a dispatch rule, against NumPy or the oracle."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from msamd import gpu as G
    G.lib()
    return G


def dev(a, dt):
    return torch.tensor(np.ascontiguousarray(a), dtype=dt, device="cuda")


def host(t):
    return t.detach().cpu().double().numpy()


@pytest.mark.parametrize("n,frames", [(2, 3), (4, 1), (64, 5), (128, 2), (256, 3)])
@pytest.mark.parametrize("code", [0, 1])
def test_normalize_ranks(gpu, n, frames, code):
    """The radix-selected bounds are the sorted image's elements: images below, at and above one
    workgroup's chunk, few distinct values, values of both signs over many binades, constant images,
    infinities. The result then repeats the definition's operations in FP64, so it is exact up to the
    rounding to the storage type."""
    rng = np.random.default_rng(n + frames)
    dt = gpu.torch_dtype(code)
    np_dt = np.float64 if code else np.float32
    kinds = [rng.poisson(3.0, (n, n)) / 200.0, rng.normal(size=(n, n)) * 10.0 ** rng.integers(-20, 20, (n, n)),
             np.full((n, n), -2.5), rng.random((n, n)) - 0.5]
    src = np.stack([kinds[(k + n) % 4] for k in range(frames)]).astype(np_dt)
    if n >= 64:
        src[-1, 0, 0], src[-1, 1, 1] = np.inf, -np.inf
    for pct, zero in ((0.15, True), (30.0, False), (200.0, True), (0.0, True), (-1.0, True), (-1.0, False)):
        out = gpu.normalize(dev(src, dt), pct, zero).cpu().numpy()
        for k in range(frames):
            v, s = src[k].astype(np.float64), np.sort(src[k].ravel()).astype(np.float64)
            m = s.size - 1
            with np.errstate(invalid="ignore", over="ignore"):
                if pct >= 0:
                    lo, hi = s[int(pct / 200 * m)], s[int((1 - pct / 200) * m)]
                    v = np.where(v < lo, lo, np.where(v > hi, hi, v)) - lo
                    top = hi - lo
                else:
                    lo, top = s[0], s[-1]
                    if lo < 0 or zero:
                        v, top = v - lo, top - lo
                want = (v / top if top != 0 else v).astype(np_dt)
            assert np.array_equal(out[k], want, equal_nan=True), (k, pct, zero)
