"""The split-x product over LDS-shared tiles (prompts of Q4_K, Q2_K, Q6_K and
IQ2_XXS) against the f64 product of the oracle's weights, at the edges of its
tiles: rows and tokens past whole tiles, one block of k, odd block counts (one k
slice of the workgroup then ends early), k slices over workgroups, blocks whose
scale is zero, and non-finite x."""
import numpy as np
import pytest

from test_gpu_parity import make_weights, upload_w

pytestmark = pytest.mark.gpu

# x is kept to 2^-22 of each value, and a sum is at most 40 roundings to f32 per
# block of 256 and one per block and slice; rounding errors of random sign over
# them stay under 16 ulp (2^-20) of the output's norm
REL = 2.0 ** -20

# (type, rows, k, tokens): shapes at which the planner takes the shared tiles (held
# to that by test_shapes_take_the_shared_tiles), whole and in 2 to 8 k slices; Q6_K
# also below 8 blocks of k, where it takes one product more
SHAPES = [("Q4_K", 641, 256, 2000), ("Q4_K", 1000, 4352, 1000), ("Q4_K", 513, 8192, 501), ("Q4_K", 777, 768, 4000),
          ("Q4_K", 3000, 2304, 449), ("Q4_K", 700, 4352, 1500), ("Q2_K", 641, 256, 2000),
          ("Q2_K", 513, 8192, 501), ("Q2_K", 777, 768, 4000),
          ("Q6_K", 1500, 256, 777), ("Q6_K", 777, 768, 1000), ("Q6_K", 513, 2304, 1000), ("Q6_K", 1000, 8192, 65),
          ("IQ2_XXS", 777, 256, 2000), ("IQ2_XXS", 513, 4352, 501), ("Q2_K", 1000, 4352, 1000),
          ("Q6_K", 513, 2048, 1000)]


def product(orc, tname, gguf, n, x, rows, k):
    w = orc.dequant(orc.NAMES[tname], gguf, n).astype(np.float64).reshape(rows, k)
    return x.astype(np.float64).reshape(-1, k) @ w.T


def run(ctx, t, wb, x, rows, k, tokens):
    xb, yb = ctx.upload(x), ctx.alloc(tokens * rows * 4)
    ctx.qmatmul(t, wb, xb, yb, rows, k, tokens)
    y = yb.read(np.float32).reshape(tokens, rows)
    ctx.qmatmul(t, wb, xb, yb, rows, k, tokens)
    again = yb.read(np.float32).reshape(tokens, rows)
    xb.free(); yb.free()
    assert np.array_equal(y.view(np.uint32), again.view(np.uint32))   # whatever the order of arrival
    return y


def test_shapes_take_the_shared_tiles(eff):
    plans = [eff.split_plan(*s) for s in SHAPES]
    assert all(p["shared"] for p in plans)
    assert {1, 2, 3, 6, 8} <= {p["slices"] for p in plans}
    assert not any(eff.split_plan(*s, 1)["shared"] for s in SHAPES)


@pytest.mark.parametrize("tname,rows,k,tokens", SHAPES)
def test_shared_tiles_vs_f64(ctx, eff, orc, tname, rows, k, tokens):
    t, data, gguf, n = make_weights(eff, tname, rows, k, 71)
    x = eff.fill_normal(72, 1.0, tokens * k)
    if tname in ("Q4_K", "Q2_K"):   # every fifth block: scale 0, its minima stay
        b = data.reshape(n, -1)
        b[::5, (0, 1) if tname == "Q4_K" else (80, 81)] = 0
    wb = ctx.upload(data)
    y = run(ctx, t, wb, x, rows, k, tokens)
    ref = product(orc, tname, gguf, n, x, rows, k)
    rel = np.linalg.norm(y - ref) / np.linalg.norm(ref)
    print(f"shared tiles {tname} {rows}x{k} M={tokens}: rel_l2={rel:.2e}", flush=True)
    assert rel <= REL
    # no row or token is off by itself (a tile's edge)
    err, scale = np.abs(y - ref), np.sqrt(np.mean(ref * ref))
    assert err.max() <= 16 * REL * scale
    # a forced configuration runs the other kernel: other sums, the same product
    try:
        ctx.set_option(eff.OPT_SPLIT_CONFIG, 1)
        other = run(ctx, t, wb, x, rows, k, tokens)
    finally:
        ctx.set_option(eff.OPT_SPLIT_CONFIG, 0)
    if k > 256:   # (over one block IQ2_XXS is summed alike)
        assert not np.array_equal(y.view(np.uint32), other.view(np.uint32))
    assert np.linalg.norm(other - ref) <= REL * np.linalg.norm(ref)
    # prepared x: the same bits
    nb, _ = ctx.qmatmul_x_layout(t, rows, k, tokens)
    xb, xp, yb = ctx.upload(x), ctx.alloc(nb), ctx.alloc(tokens * rows * 4)
    ctx.qmatmul_prepare_x(t, xb, xp, rows, k, tokens)
    ctx.qmatmul_prepared(t, wb, xp, yb, rows, k, tokens)
    assert np.array_equal(yb.read(np.uint32), y.view(np.uint32).ravel())
    for b in (wb, xb, xp, yb):
        b.free()


@pytest.mark.parametrize("tname,rows,k,tokens", [SHAPES[1], SHAPES[3], SHAPES[10], SHAPES[14]])
def test_shared_tiles_range_and_non_finite(ctx, eff, orc, tname, rows, k, tokens):
    """x of mixed magnitudes (blocks of 1e-20 to 1e20), and tokens holding an
    infinity or a NaN, whose outputs become non-finite and no other's."""
    t, data, gguf, n = make_weights(eff, tname, rows, k, 81)
    x = eff.fill_normal(82, 1.0, tokens * k).reshape(tokens, k)
    x[0:4] *= 1e-20
    x[4:8] *= 1e20
    x[70, :256] *= 1e-3
    x[70, 300 % k] *= 1e4
    bad = x.copy()
    bad[9, 5], bad[tokens - 1, k - 1] = np.inf, np.nan
    wb = ctx.upload(data)
    y = run(ctx, t, wb, bad, rows, k, tokens)
    ref = product(orc, tname, gguf, n, x, rows, k)
    good = np.ones(tokens, bool)
    good[[9, tokens - 1]] = False
    assert not np.isfinite(y[~good]).any() and np.isfinite(y[good]).all()
    rel = np.linalg.norm(y - ref, axis=1)[good] / np.linalg.norm(ref, axis=1)[good]
    assert rel.max() <= 2 * REL
    wb.free()


# weights of one sign and of both: Q4_K and Q2_K then hold no minima, or minima only
WEIGHTS = {"normal": lambda z, e: z, "abs": lambda z, e: np.abs(z), "exp3": lambda z, e: e ** 3,
           "neg": lambda z, e: -np.abs(z)}
PROMPTS = [(1000, 512, 777), (1024, 2048, 1000), (513, 8192, 501)]


@pytest.mark.parametrize("tname,rows,k,tokens", [(t, *s) for t in ("Q4_K", "Q2_K", "Q6_K") for s in PROMPTS])
@pytest.mark.parametrize("positive_x", [False, True])
def test_error_no_larger_than_the_other_kernels(ctx, eff, orc, tname, rows, k, tokens, positive_x):
    """Relative L2 error against 64 bits beside that of the kernel whose waves read x
    by themselves, for weights of both signs and of one. The two add the same terms in
    another order, which by itself moves the error by up to 2%: 1.05 of it at most."""
    assert eff.split_plan(tname, rows, k, tokens)["shared"]
    t = eff.TYPES[tname]
    x = eff.fill_normal(76, 1.0, tokens * k)
    x = np.abs(x) if positive_x else x
    z = eff.fill_normal(75, 0.02, rows * k)
    e = np.abs(eff.fill_normal(77, 0.2, rows * k))
    for kind, f in WEIGHTS.items():
        data = eff.quantize(t, np.ascontiguousarray(f(z, e), np.float32))
        ref = product(orc, tname, data, rows * k // 256, x, rows, k)
        wb = ctx.upload(data)
        err = []
        try:
            for cfg in (0, 1):
                ctx.set_option(eff.OPT_SPLIT_CONFIG, cfg)
                err.append(np.linalg.norm(run(ctx, t, wb, x, rows, k, tokens) - ref) / np.linalg.norm(ref))
        finally:
            ctx.set_option(eff.OPT_SPLIT_CONFIG, 0)
            wb.free()
        print(f"{tname} {rows}x{k} M={tokens} {kind}: {err[0]:.3e} beside {err[1]:.3e}", flush=True)
        assert err[0] <= 1.05 * err[1], kind


@pytest.mark.parametrize("tname", ["Q4_K", "Q2_K"])
def test_zero_weights_give_zero(ctx, eff, tname):
    """Blocks whose quants and minima are zero, at scales that are not: every output
    is 0, as the sums of the weights themselves are."""
    rows, k, tokens = 1000, 512, 777
    assert eff.split_plan(tname, rows, k, tokens)["shared"]
    data = np.zeros((rows * k // 256, 144 if tname == "Q4_K" else 84), np.uint8)
    if tname == "Q4_K":
        data[:, 1], data[:, 3], data[:, 4:8] = 0x20, 0x20, 63      # d, dmin and the first scales
    else:
        data[:, :16], data[:, 81], data[:, 83] = 15, 0x20, 0x20
    wb = ctx.upload(data)
    assert not run(ctx, eff.TYPES[tname], wb, eff.fill_normal(5, 1.0, tokens * k), rows, k, tokens).any()
    wb.free()


def test_recorded_before_any_eager_call_gives_the_eager_bits(eff, orc):
    """A shape whose shared tiles take k slices, recorded in a context in which no
    eager call has taken them: the recording runs the same kernel, gives the bits of
    the eager calls that follow, and replays them unchanged among other products."""
    rows, k, tokens = 2048, 8192, 300
    with eff.Context(0) as ctx:
        t, data, gguf, n = make_weights(eff, "Q6_K", rows, k, 97)
        assert eff.split_plan(t, rows, k, tokens)["shared"] and eff.split_plan(t, rows, k, tokens)["slices"] > 1
        x = eff.fill_normal(98, 1.0, tokens * k)
        ref = product(orc, "Q6_K", gguf, n, x, rows, k)
        wb, xb, yb = ctx.upload(data), ctx.upload(x), ctx.alloc(tokens * rows * 4)
        nb, _ = ctx.qmatmul_x_layout(t, rows, k, tokens)
        xp = ctx.alloc(nb)
        ctx.qmatmul_prepare_x(t, xb, xp, rows, k, tokens)
        ctx.set_option(eff.OPT_SPLIT_CONFIG, 1)
        ctx.qmatmul(t, wb, xb, yb, rows, k, tokens)      # sizes the x scratch, by the other kernel
        plain = yb.read(np.uint32)
        ctx.set_option(eff.OPT_SPLIT_CONFIG, 0)

        def record(prepared):
            ctx.graph_begin()
            if prepared:
                ctx.qmatmul_prepared(t, wb, xp, yb, rows, k, tokens)
            else:
                ctx.qmatmul(t, wb, xb, yb, rows, k, tokens)
            return ctx.graph_end()

        graphs = [record(False), record(True)]
        got = []
        for g in graphs:
            yb.write(np.zeros(tokens * rows, np.float32))
            g.launch()
            got.append(yb.read(np.uint32))
        ctx.qmatmul(t, wb, xb, yb, rows, k, tokens)
        eager = yb.read(np.uint32)
        assert not np.array_equal(eager, plain)
        assert np.linalg.norm(eager.view(np.float32).reshape(tokens, rows) - ref) <= REL * np.linalg.norm(ref)
        for y in got:
            assert np.array_equal(y, eager)
        graphs += [record(False), record(True)]
        for _ in range(2):
            ctx.qmatmul(t, wb, xb, yb, rows, k, 129)
            for g in graphs:
                yb.write(np.zeros(tokens * rows, np.float32))
                g.launch()
                assert np.array_equal(yb.read(np.uint32), eager)
        for g in graphs:
            g.destroy()
        for b in (wb, xb, yb, xp):
            b.free()


def test_forced_slices_leave_a_recording_its_buffer(eff, orc):
    """A recording of the sliced shared tiles, then eager calls whose forced slice
    count needs more than the slices' buffer holds (512 tiles x 8): they run the
    other kernel, and the recording replays its bits."""
    with eff.Context(0) as ctx:
        small, big = ("Q6_K", 2048, 8192, 300), ("Q4_K", 8192, 2048, 512)
        assert eff.split_plan(*small)["shared"] and eff.split_plan(*small)["slices"] > 1
        assert not eff.split_plan(*big, 0, 8)["shared"]
        st = []
        for tname, rows, k, tokens in (small, big):
            t, data, gguf, n = make_weights(eff, tname, rows, k, 97)
            x = eff.fill_normal(98, 1.0, tokens * k)
            st.append((t, ctx.upload(data), ctx.upload(x), ctx.alloc(tokens * rows * 4),
                       product(orc, tname, gguf, n, x, rows, k)))
        t, wb, xb, yb, ref = st[0]
        t2, wb2, xb2, yb2, ref2 = st[1]
        ctx.qmatmul(t2, wb2, xb2, yb2, *big[1:])
        ctx.qmatmul(t, wb, xb, yb, *small[1:])
        want = yb.read(np.uint32)
        assert np.linalg.norm(want.view(np.float32).reshape(ref.shape) - ref) <= REL * np.linalg.norm(ref)
        ctx.graph_begin()
        ctx.qmatmul(t, wb, xb, yb, *small[1:])
        g = ctx.graph_end()
        ctx.set_option(eff.OPT_SPLIT_SLICES, 8)
        for _ in range(2):
            ctx.qmatmul(t2, wb2, xb2, yb2, *big[1:])
            y2 = yb2.read(np.float32).reshape(ref2.shape)
            assert np.linalg.norm(y2 - ref2) <= REL * np.linalg.norm(ref2)
            yb.write(np.zeros(yb.size // 4, np.float32))
            g.launch()
            assert np.array_equal(yb.read(np.uint32), want)
        g.destroy()
        for _, *bufs, _ in st:
            for b in bufs:
                b.free()


@pytest.mark.parametrize("tname", ["Q4_K", "Q2_K", "IQ2_XXS"])
@pytest.mark.parametrize("tokens", [33, 48, 64, 65, 96, 129])
def test_three_token_tiles(ctx, eff, orc, tname, tokens):
    """Token counts that three tiles of 16 per wave fit better than four (33-48,
    65-96, 129-144; 64 takes four), in both workgroup shapes and from a prepared x."""
    rows, k = 77, 1280
    t, data, gguf, n = make_weights(eff, tname, rows, k, 91)
    x = eff.fill_normal(92, 1.0, tokens * k)
    ref = product(orc, tname, gguf, n, x, rows, k)
    wb = ctx.upload(data)
    try:
        for cfg in (0, 1, 2):
            ctx.set_option(eff.OPT_SPLIT_CONFIG, cfg)
            y = run(ctx, t, wb, x, rows, k, tokens)
            assert np.linalg.norm(y - ref) <= REL * np.linalg.norm(ref), cfg
            assert np.abs(y - ref).max() <= 16 * REL * np.sqrt(np.mean(ref * ref)), cfg
            nb, _ = ctx.qmatmul_x_layout(t, rows, k, tokens)
            xb, xp, yb = ctx.upload(x), ctx.alloc(nb), ctx.alloc(tokens * rows * 4)
            ctx.qmatmul_prepare_x(t, xb, xp, rows, k, tokens)
            ctx.qmatmul_prepared(t, wb, xp, yb, rows, k, tokens)
            assert np.array_equal(yb.read(np.uint32), y.view(np.uint32).ravel())
            for b in (xb, xp, yb):
                b.free()
    finally:
        ctx.set_option(eff.OPT_SPLIT_CONFIG, 0)
    wb.free()


@pytest.mark.parametrize("tname", ["Q8_0", "Q8_0R", "Q6_K"])
@pytest.mark.parametrize("rows,k,tokens", [(2048, 8192, 8), (77, 8192, 7), (1000, 4608, 8), (130, 16384, 5)])
def test_one_launch_in_k_slices(ctx, eff, orc, tname, rows, k, tokens):
    """5-8 tokens where the int8 GEMVs do not run: x prepared inside the product
    (whose workgroups take slices of k), with the bits of the two-launch form."""
    t, data, gguf, n = make_weights(eff, tname, rows, k, 95)
    x = eff.fill_normal(96, 1.0, tokens * k)
    x[:256] *= 1e-3
    x[k:k + 256] *= 1e6
    wb = upload_w(ctx, eff, tname, data, n)
    assert not eff.split_plan(t, rows, k, tokens)["prepares_x"]
    before = ctx.stats()
    y = run(ctx, t, wb, x, rows, k, tokens)
    assert ctx.stats()["split"] == before["split"] + 2
    assert ctx.stats()["split_x"] == before["split_x"]      # no preparation of its own: one launch
    ref = product(orc, "Q8_0" if tname == "Q8_0R" else tname, gguf, n, x, rows, k)
    assert (np.linalg.norm(y - ref, axis=1) <= REL * np.linalg.norm(ref, axis=1)).all()
    nb, _ = ctx.qmatmul_x_layout(t, rows, k, tokens)
    xb, xp, yb = ctx.upload(x), ctx.alloc(nb), ctx.alloc(tokens * rows * 4)
    ctx.qmatmul_prepare_x(t, xb, xp, rows, k, tokens)
    ctx.qmatmul_prepared(t, wb, xp, yb, rows, k, tokens)
    assert ctx.stats()["split_x"] == before["split_x"] + 1
    assert np.array_equal(yb.read(np.uint32), y.view(np.uint32).ravel())
    for b in (wb, xb, xp, yb):
        b.free()
