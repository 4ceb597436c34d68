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


@pytest.mark.parametrize("n,frames", [(2, 3), (4, 1), (64, 5), (128, 2), (256, 3), (8, 2), (32, 3), (512, 5)])
@pytest.mark.parametrize("code", [0, 1])
def test_normalize_ranks(gpu, n, frames, code):
    """The radix-selected bounds are the sorted image's elements: images below, at and above one
    workgroup's chunk (one launch up to 64^2, above it 8 or 32 pixels per thread), few distinct values, values of both signs over many binades, constant images,
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


def test_normalize_many_small_images(gpu):
    """More images than one launch takes (2^20 workgroups): the ends of the launches and of the whole are what
    they are alone."""
    img = torch.randn((1 << 22) + 3, 2, 2, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    out = gpu.normalize(img.clone(), 0.15)
    for k in (0, (1 << 20) - 1, 1 << 20, 1 << 21, (1 << 22) - 1, 1 << 22, (1 << 22) + 2):
        assert torch.equal(out[k:k + 1], gpu.normalize(img[k:k + 1].clone(), 0.15))


@pytest.mark.parametrize("frames", [1, 2, 3, 4, 5, 7, 8, 9, 16, 17, 31, 32, 33, 63, 64, 65])
@pytest.mark.parametrize("code", [0, 1])
def test_series_stats_networks(gpu, frames, code):
    """Every length around the sorting networks' sizes and the counting kernel beyond them, on a pixel
    count that is no multiple of a workgroup: ties, missing samples, -Inf; the statistics are selections
    and one FP64 sum in frame order, so count and median are exact."""
    n = 16 if frames != 33 else 8
    rng = np.random.default_rng(100 + frames)
    dt = gpu.torch_dtype(code)
    st = rng.normal(size=(frames, n, n))
    st = np.round(st * 4) / 4 if frames % 3 == 0 else st
    st[rng.random(st.shape) < 0.25] = np.inf
    st[:, 0, 0] = np.inf
    st[frames // 2, 1, 1] = -np.inf
    st = st.astype(np.float64 if code else np.float32)
    t = torch.tensor(st, device="cuda")
    mean, count, med = (host(x) for x in gpu.series_stats(t, 0.375))
    have = st != np.inf
    c = have.sum(0)
    assert np.array_equal(count, c)
    s = np.sort(st.astype(np.float64), axis=0)
    for y in range(n):
        for x in range(n):
            k = c[y, x]
            want = 0.375 if k == 0 else (s[k // 2, y, x] if k % 2 else (s[k // 2 - 1, y, x] + s[k // 2, y, x]) / 2)
            assert med[y, x] == (want if code else np.float64(np.float32(want)))
            acc = 0.0
            for f in range(frames):
                acc += float(st[f, y, x]) if have[f, y, x] else 0.0
            want = acc / k if k else 0.375
            assert mean[y, x] == (want if code else np.float64(np.float32(want)))


@pytest.mark.parametrize("n,count", [(2, 3), (16, 2), (32, 1), (64, 3), (512, 1)])
@pytest.mark.parametrize("code", [0, 1])
def test_warp_modes(gpu, n, count, code):
    """Images below, at and above one workgroup's pixels, every mode, one field per image and one
    shared, displacements that leave the grid, land on its border and are not finite. The kernel's FP64
    operations are repeated in their order: exact up to the rounding to the storage type."""
    rng = np.random.default_rng(n)
    np_dt = np.float64 if code else np.float32
    dt = gpu.torch_dtype(code)
    img = rng.normal(size=(count, n, n)).astype(np_dt)
    phi = (rng.normal(size=(count, 2, n, n)) * 3 / (n - 1)).astype(np_dt)
    phi[:, :, 0, :] = 0
    phi[0, 0, 1, 0], phi[0, 1, 1, 1], phi[0, 0, 0, 1] = np.inf, -np.inf, np.nan
    h, hi = 1.0 / (n - 1), float(n - 1)
    yy, xx = np.mgrid[0:n, 0:n]
    for shared in (False, True):
        p = phi[0] if shared else phi
        for mode, nearest in ((0, False), (0, True), (1, False), (2, False)):
            got = gpu.warp(dev(img, dt), dev(p, dt), mode, 0.75, nearest).cpu().numpy()
            for k in range(count):
                f = (p if shared else p[k]).astype(np.float64)
                with np.errstate(invalid="ignore"):
                    X, Y = xx + f[0] / h, yy + f[1] / h
                    if mode == 1:
                        X, Y = (np.where(c < 0, 0, np.where(c > hi, hi, c)) for c in (X, Y))
                        inside = np.ones((n, n), bool)
                    else:
                        inside = ~((X < 0) | (X > hi) | (Y < 0) | (Y > hi))
                        if mode == 0:
                            inside &= ~(np.isnan(X) | np.isnan(Y))
                        if nearest:
                            X, Y = np.floor(X + 0.5), np.floor(Y + 0.5)
                    X, Y = np.where(np.isnan(X), 0, X), np.where(np.isnan(Y), 0, Y)
                    i, j = (np.clip(np.trunc(np.clip(c, -1, n)), 0, n - 2).astype(int) for c in (X, Y))
                    X, Y = X - i, Y - j
                    v = [img[k][b, a].astype(np.float64) for b in (j, j + 1) for a in (i, i + 1)]
                    r0 = (1 - X) * v[0] + X * v[1]
                    r1 = (1 - X) * (1 - Y) * v[0] + X * (1 - Y) * v[1] + (1 - X) * Y * v[2] + X * Y * v[3]
                    want = np.where(inside, np.where(Y == 0, r0, r1), np.nan if mode == 2 else 0.75).astype(np_dt)
                assert np.array_equal(got[k], want, equal_nan=True), (shared, mode, nearest, k)


@pytest.mark.parametrize("scales,base,H,W", [(4, 32, 256, 256), (2, 64, 128, 256)])
def test_unet_tile_choice(gpu, scales, base, H, W):
    """The convolutions' tiles depend on the amount of work; their sums run in one order, so an image's
    prediction is the same bits alone as inside a batch of eight."""
    net = gpu.UNet(scales, base, seed=2)
    x = torch.rand((8, 2, H, W), device="cuda")
    whole = net.forward(x)
    for k in (0, 7):
        assert torch.equal(net.forward(x[k:k + 1].contiguous())[0], whole[k])
    net.close()


@pytest.mark.parametrize("scales,base,B,H,W", [(1, 32, 3, 32, 96), (2, 64, 1, 64, 128), (2, 128, 1, 64, 64),
                                               (2, 256, 1, 64, 64)])
def test_unet_widths(gpu, scales, base, B, H, W):
    """Every source of an activation's gradient (no pooling at one scale), the convolutions' channel
    counts up to those whose input tile fits LDS (384) and beyond (512, 768), on one tile of rows and
    columns and on several: against the CPU network, within four times the difference between FP64 and
    FP32 accumulation of the same BF16 operands."""
    import unet_ref as U
    rng = np.random.default_rng(base)
    x = rng.random((B, 2, H, W)).astype(np.float32)
    t = (2.0 * rng.standard_normal((B, 2, H, W))).astype(np.float32)
    net = gpu.UNet(scales, base, seed=3)
    p = net.get_params().astype(np.float64)
    out = host(net.forward(dev(x, torch.float32)))
    _, g = net.gradient(dev(x, torch.float32), dev(t, torch.float32), want_grad=True)
    net.close()

    def gap(a, b):
        return np.linalg.norm(a - b) / np.linalg.norm(b)

    ref, _ = U.forward(p, x.astype(np.float64), scales, base)
    alt, _ = U.forward(p, x.astype(np.float64), scales, base, acc32=True)
    assert gap(out, ref) < max(1e-3, 4 * gap(alt, ref))
    _, ref_g, _ = U.loss_and_grad(p, x.astype(np.float64), t.astype(np.float64), scales, base)
    _, alt_g, _ = U.loss_and_grad(p, x.astype(np.float64), t.astype(np.float64), scales, base, acc32=True)
    for c in U.graph(scales, base)[1]:
        for a, k in ((c["woff"], 9 * c["cout"] * (c["cin1"] + c["cin2"])), (c["boff"], c["cout"])):
            s = slice(a, a + k)
            assert gap(g[s], ref_g[s]) < max(1e-2, 4 * gap(alt_g[s], ref_g[s])), a


def test_unet_gradient_of_a_batch(gpu):
    """A batch's convolutions take larger tiles than an image's (16 images of 256^2 every FP32-output tile of
    32 to 256 channels, among them those that no single image here reaches). Its loss is the mean of the
    images', 1/16 of their gradients an exact scaling, and every sum but those over pixels runs in one order,
    so its gradient is the mean of the images' but for the FP32 sums over up to 2^20 pixels: their terms have
    random signs (random targets), so about 2^-24 sqrt(2^20) = 6e-5 of the result, 3e-4 allowed."""
    import unet_ref as U
    net = gpu.UNet(4, 32, seed=4)
    g = torch.Generator(device="cuda").manual_seed(9)
    x = torch.rand((16, 2, 256, 256), device="cuda", generator=g)
    t = 2.0 * torch.randn((16, 2, 256, 256), device="cuda", generator=g)
    loss, got = net.gradient(x, t, want_grad=True)
    one = [net.gradient(x[k:k + 1].contiguous(), t[k:k + 1].contiguous(), want_grad=True) for k in range(16)]
    net.close()
    want = np.mean([np.asarray(o[1], np.float64) for o in one], axis=0)
    assert abs(loss - np.mean([o[0] for o in one])) <= 1e-12 * loss
    _, convs, _, head, total = U.graph(4, 32)
    parts = [(c["woff"], 9 * c["cout"] * (c["cin1"] + c["cin2"])) for c in convs] + [(c["boff"], c["cout"]) for c in convs]
    for a, k in parts + [(head["woff"], total - head["woff"])]:
        assert np.linalg.norm(got[a:a + k] - want[a:a + k]) <= 3e-4 * np.linalg.norm(want[a:a + k]), a


@pytest.mark.parametrize("n", [2, 4, 16, 64])
@pytest.mark.parametrize("pixels", [0.0, 0.4, 6.0])
def test_compose_borders(gpu, n, pixels):
    """No undefined node, a few, and whole borders and corners of them (every form of a stiffness row),
    from a start value of its own: FP64 fields against the oracle, which runs the same recurrence."""
    rng = np.random.default_rng(n)
    h = 1.0 / (n - 1)
    y, x = np.mgrid[0:n, 0:n] / n
    p1 = 0.3 * h * rng.normal(size=(2, n, n))
    p2 = pixels * h * np.stack([np.sin(3 * x + y) - 0.3, np.cos(2 * y - x) - 0.4])
    start = 0.2 * h * rng.normal(size=(2, n, n))
    got = host(gpu.compose(dev(p1, torch.float64), dev(p2, torch.float64), dev(start, torch.float64)))
    want = O.compose(p1, p2, start)
    # both stop at |residual|^2 < 1e-16; rounding moves the iterates by far less than what that leaves
    assert np.abs(got - want).max() < 1e-10 * max(np.abs(want).max(), h)


@pytest.mark.parametrize("n", [2, 4, 64, 128, 256, 512, 1024, 2048])
def test_xshift_row_lengths(gpu, n):
    """Every thread count and run length of the row kernels, displacements that leave the row at both
    ends, a row that starts with NaN (left out): FP64 fields against the oracle. Rounding: sums of n
    terms in another order, 1e-16 n at worst relative to terms of the result's size."""
    rng = np.random.default_rng(n)
    x = np.arange(n) / n
    R = 1 + np.cumsum(rng.normal(size=(n, n)), axis=1) / n
    T = np.roll(R, 1, axis=1) + 0.02 * rng.normal(size=(n, n))
    phi = (3.0 * np.sin(7 * x[None, :] + np.arange(n)[:, None] / n) + 0.3 * rng.normal(size=(n, n))) / (n - 1)
    if n >= 64:
        R[n // 2, 0] = np.nan
    args = (dev(R[None], torch.float64), dev(T[None], torch.float64),
            dev(np.stack([phi, np.zeros_like(phi)])[None], torch.float64))
    ed, er = gpu.xshift_energy(*args, 0.7)
    g = host(gpu.xshift_gradient(*args, 5.0, 0.7))[0]
    oe, orr = O.xshift_energy(R, T, phi, 0.7)
    og = O.xshift_gradient(R, T, phi, 0.7, 5.0)
    tol = 2e-16 * 8 * n
    assert abs(ed[0] - oe) <= max(tol, 1e-14) * max(abs(oe), 1.0)
    assert abs(er[0] - orr) <= max(tol, 1e-14) * abs(orr)
    assert np.abs(g[0] - og).max() <= max(100 * tol, 1e-12) * np.abs(og).max()
    assert (g[1] == 0).all()


@pytest.mark.parametrize("n,pairs", [(2, 1 << 19), (4, 1 << 17), (64, 513), (128, 128), (512, 8), (1024, 3)])
def test_f32_gradient_runs_are_the_tiles(gpu, n, pairs):
    """The FP32 SSD gradient of 2^21 nodes and more, from 512^2 on in element runs of whole waves, repeats the
    operations and order of smaller launches' tiles: the same bits, with positions inside, on and far outside
    the domain and a NaN."""
    g = torch.Generator(device="cuda").manual_seed(n)
    R, T = (torch.rand(pairs, n, n, device="cuda", generator=g) for _ in range(2))
    phi = torch.randn(pairs, 2, n, n, device="cuda", generator=g) * (4.0 / n)
    phi[1] = 0.0
    phi[2 % pairs, 0, n // 2, n // 3] = 1e30
    phi[0, 1, n - 1, 0] = float("nan")
    whole = gpu.gradient(R, T, phi, 50.0)
    step = max(1, ((1 << 21) - 1) // (n * n))
    for a in range(0, pairs, step):
        part = gpu.gradient(R[a:a + step].contiguous(), T[a:a + step].contiguous(), phi[a:a + step].contiguous(), 50.0)
        ref = whole[a:a + step]
        assert torch.equal(part.isnan(), ref.isnan())
        # 0 == -0, which the bits tell apart: compared where both are numbers and not zero, zeros as zeros
        same = (part.view(torch.int32) == ref.contiguous().view(torch.int32)) | part.isnan() | ((part == 0) & (ref == 0))
        assert same.all()


def test_f32_gradient_above_4096(gpu):
    """Above 4096^2 the gather offsets are integers. Smooth images (period 400 px or more): the FP32 differences
    of neighbouring values carry 2^-24 / (2 pi / 400) = 4e-6 relative, so 2e-5 in L2 against the FP64 pass on
    the same stored values."""
    n = 8192
    y = torch.linspace(0, 1, n, device="cuda", dtype=torch.float64)[:, None]
    x = torch.linspace(0, 1, n, device="cuda", dtype=torch.float64)[None, :]
    R = (0.5 + 0.4 * torch.sin(100 * x + 60 * y)).float()[None]
    T = (0.5 + 0.4 * torch.cos(90 * x - 110 * y)).float()[None]
    phi = torch.stack([1e-3 * torch.sin(9 * x + 4 * y), 1e-3 * torch.cos(5 * x - 8 * y)]).float()[None]
    a = gpu.gradient(R, T, phi, 0.0).double()
    b = gpu.gradient(R.double(), T.double(), phi.double(), 0.0)
    assert ((a - b).norm() / b.norm()).item() < 2e-5


@pytest.mark.parametrize("op", ["ncc", "compose", "xshift"])
def test_displacements_beyond_the_range(gpu, op):
    """Finite displacements whose value in pixels overflows FP64 (from 2.9e306 domain units on, at 63 pixels a
    unit; the kernels divide by a corrected reciprocal) and infinite ones are positions beyond the grid as any
    other: the data terms and the composition are those of a displacement of 2e4 pixels, bit for bit (weight 0
    on the regulariser, whose own value overflows)."""
    n, h = 64, 1.0 / 63
    rng = np.random.default_rng(11)
    R, T = 1 + np.cumsum(rng.normal(size=(2, 1, n, n)), axis=3) / n
    base = 0.4 * h * rng.normal(size=(2, n, n))

    def fields(huge):
        p = base.copy()
        for k, (y, x) in enumerate(((5, 9), (20, 3), (33, 50), (62, 62), (0, 30), (41, 0))):  # no shared element
            p[k % 2 if op != "xshift" else 0, y, x] = huge if k < 3 else -huge
        return dev(p[None], torch.float64)

    a = (dev(R, torch.float64), dev(T, torch.float64))

    def run(huge, gradient):
        p = fields(huge)
        if op == "ncc":
            return [gpu.ncc_energy(*a, p)[0]] + ([host(gpu.ncc_gradient(*a, p, 0.0))] if gradient else [])
        if op == "xshift":
            return [gpu.xshift_energy(*a, p, 0.7)[0]] + ([host(gpu.xshift_gradient(*a, p, 0.0, 0.7))] if gradient else [])
        return [host(gpu.compose(dev(base, torch.float64), p[0]))]

    for huge in (3e306, 5e306, 1e307, 1.7e308, np.inf):  # just beyond 2^1024 pixels, far beyond
        gradient = huge <= 1e307  # 0 times the stiffness row of the larger ones is NaN
        for got, want in zip(run(huge, gradient), run(2e4 * h, gradient)):
            assert np.isfinite(want).all() and np.array_equal(got, want)


@pytest.mark.parametrize("n", [2, 4, 8, 16, 32, 64])
def test_f64_coarse_workgroups(gpu, n):
    """The FP64 coarse V-cycle's workgroup depends on the level and, at 32^2, on the number of fields (more than
    256 take narrower ones); the operations and the scalar products' sums do not: fields smoothed and levels
    solved in a batch of 129 pairs are those of small batches bit for bit."""
    g = torch.Generator(device="cuda").manual_seed(n)
    phi = torch.randn(129, 2, n, n, device="cuda", generator=g, dtype=torch.float64)
    whole = gpu.h1_smooth(phi, 0.125)
    for a in (0, 64, 128):
        assert torch.equal(gpu.h1_smooth(phi[a:a + 64].contiguous(), 0.125), whole[a:a + 64])
    if n < 8:
        return
    R = torch.rand(129, n, n, device="cuda", generator=g, dtype=torch.float64)
    T = 0.6 * R + 0.4 * R.roll(1, 2)
    out = []
    for a, b in ((0, 129), (0, 2), (127, 129)):
        c = gpu.Context(n.bit_length() - 1, b - a, gpu.F64)
        c.set_images_device(R[a:b].contiguous(), T[a:b].contiguous())
        c.set_deformations_device(torch.zeros(b - a, 2, n, n, device="cuda", dtype=torch.float64))
        e = np.array(c.solve_level(n.bit_length() - 1, 10.0, 5, -1.0)[0])
        f = torch.empty(b - a, 2, n, n, device="cuda", dtype=torch.float64)
        c.get_deformations_device(f)
        c.close()
        out.append((e, f))
    for (e, f), (a, b) in zip(out[1:], ((0, 2), (127, 129))):
        assert np.array_equal(e, out[0][0][a:b]) and torch.equal(f, out[0][1][a:b])


def test_energies_from_many_threads(gpu):
    """The energies' results pass through pinned blocks that calls borrow and give back: threads that come and go,
    with batches of different sizes and the blocks freed in between, get what one thread gets."""
    import threading
    g = torch.Generator(device="cuda").manual_seed(3)
    work = []
    for k, (n, pairs) in enumerate(((16, 1), (8, 700), (32, 3), (64, 2), (4, 3000), (128, 1))):
        R, T = (torch.rand(pairs, n, n, device="cuda", generator=g) for _ in range(2))
        phi = torch.randn(pairs, 2, n, n, device="cuda", generator=g) * (1.0 / n)
        work.append((R, T, phi, gpu.energy(R, T, phi)))
    torch.cuda.synchronize()
    wrong = []

    def run(k):
        for r in range(10):
            R, T, phi, want = work[(k + r) % len(work)]
            got = gpu.energy(R, T, phi)
            if not all(np.array_equal(a, b) for a, b in zip(got, want)):
                wrong.append((k, r))
            if k == 0 and r == 5:
                gpu.release_cache()

    for _ in range(2):
        threads = [threading.Thread(target=run, args=(k,)) for k in range(8)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    assert not wrong


def shortest(fn, calls=25):
    """The shortest of some calls, in seconds (every entry point waits for its result)."""
    import time
    best = 1e9
    for _ in range(calls):
        torch.cuda.synchronize()
        a = time.perf_counter()
        fn()
        torch.cuda.synchronize()
        best = min(best, time.perf_counter() - a)
    return best


def test_many_small_fields_keep_the_rate(gpu):
    """8192 pairs of 8^2 FP64 fields are 64 workgroups a compute unit of one wave: 2 times a single pair's call,
    whose launch dominates (16 times where every field took 1024 threads); 5 allowed."""
    phi = torch.randn(8192, 2, 8, 8, device="cuda", dtype=torch.float64)
    one = phi[:1].contiguous()
    assert shortest(lambda: gpu.h1_smooth(phi, 0.125)) < 5 * shortest(lambda: gpu.h1_smooth(one, 0.125))


def test_many_small_pairs_keep_the_rate(gpu):
    """The FP32 SSD gradient of 4096 pairs of 32^2 in tiles that fit them takes as long as that of one pair of
    2048^2, the same number of nodes (1.8 times in runs of 63 columns); 1.4 allowed."""
    def inputs(n, pairs):
        R, T = (torch.rand(pairs, n, n, device="cuda") for _ in range(2))
        return R, T, torch.randn(pairs, 2, n, n, device="cuda") * (1.5 / n), 10.0
    small, large = inputs(32, 4096), inputs(2048, 1)
    assert shortest(lambda: gpu.gradient(*small)) < 1.4 * shortest(lambda: gpu.gradient(*large))


@pytest.mark.parametrize("n,count", [(2, 1 << 17), (8, 8193), (64, 129), (256, 9), (512, 2)])
@pytest.mark.parametrize("code", [0, 1])
def test_warp_runs(gpu, n, count, code):
    """From 2^19 pixels on a thread takes four pixels of a column; fewer pixels go one by one, with the same
    operations: images of a large launch are those of small ones bit for bit, on grids below, at and above a
    tile's 256 columns, every mode, a field per image and a shared one, with positions that are not finite."""
    dt = gpu.torch_dtype(code)
    g = torch.Generator(device="cuda").manual_seed(n)
    img = torch.rand(count, n, n, device="cuda", generator=g, dtype=dt)
    phi = torch.randn(count, 2, n, n, device="cuda", generator=g, dtype=dt) * (2.0 / n)
    phi[:, 0, 0, 0], phi[:, 1, 1, 1] = float("nan"), float("-inf")
    some = sorted({0, count // 2, count - 1})
    for mode, nearest in ((0, False), (0, True), (1, False), (2, False)):
        whole = gpu.warp(img, phi, mode, 0.75, nearest)
        shared = gpu.warp(img, phi[0].contiguous(), mode, 0.75, nearest)
        for k in some:
            one = img[k:k + 1].contiguous()
            for got, want in ((whole, gpu.warp(one, phi[k:k + 1].contiguous(), mode, 0.75, nearest)),
                              (shared, gpu.warp(one, phi[0].contiguous(), mode, 0.75, nearest))):
                assert torch.equal(got[k].isnan(), want[0].isnan())
                assert torch.equal(got[k].nan_to_num(9.0), want[0].nan_to_num(9.0))


def test_warp_of_noisy_fields_keeps_the_rate(gpu):
    """Neighbouring rows' gathers share cache lines: a warp of FP64 images by a field with 1.5 pixels of noise takes
    about 1.15 times that of a zero field (1.8 times with four distant pixels per thread); 1.5 allowed."""
    img = torch.rand(31, 1024, 1024, device="cuda", dtype=torch.float64)
    phi = torch.randn(31, 2, 1024, 1024, device="cuda", dtype=torch.float64) * (1.5 / 1024)
    still = torch.zeros_like(phi)
    assert shortest(lambda: gpu.warp(img, phi)) < 1.5 * shortest(lambda: gpu.warp(img, still))


def test_normalize_of_a_small_image_is_one_launch(gpu):
    """An FP64 image of 16^2 is normalised in about 1.2 times the time of its warp, one launch each (2.5 times in
    eight launches); 1.8 allowed."""
    img = torch.rand(1, 16, 16, device="cuda", dtype=torch.float64)
    phi = torch.zeros(1, 2, 16, 16, device="cuda", dtype=torch.float64)
    assert shortest(lambda: gpu.normalize(img, 0.15)) < 1.8 * shortest(lambda: gpu.warp(img, phi))


def test_unet_of_wide_layers_keeps_the_rate(gpu):
    """One image through 256 to 2048 channels is 8 times the operations of 8 images through 32 to 256, and takes 7
    times as long (15 times where a step of the wide layers waited for its own loads); 10 allowed."""
    wide, narrow = gpu.UNet(4, 256, seed=1), gpu.UNet(4, 32, seed=1)
    x = torch.rand(8, 2, 256, 256, device="cuda")
    one = x[:1].contiguous()
    assert shortest(lambda: wide.forward(one)) < 10 * shortest(lambda: narrow.forward(x))
    wide.close()
    narrow.close()


def test_statistics_of_one_frame_keep_the_rate(gpu):
    """The statistics of one frame read and write what the warp of it does, and take 0.85 times its time at 2048^2
    (1.3 times with its one sample padded to 8); 1.1 allowed."""
    img = torch.rand(1, 2048, 2048, device="cuda")
    phi = torch.zeros(1, 2, 2048, 2048, device="cuda")
    assert shortest(lambda: gpu.series_stats(img, 0.0), 60) < 1.1 * shortest(lambda: gpu.warp(img, phi), 60)
