"""Products on the matrix cores (Q4_0, Q8_0, Q6_K, BF16, and Q4_K) against
float64 products of the same dequantized weights, at the sizes where their
tiles, steps and parts end.

The bound: a result is a sum of cols products, each of an exact weight and an
activation kept to 23 bits (2^-23 of it: two of the last term's 2^-24), summed
in f32.  Sums of at most 64 products round inside a block, then a sum of at most
cols/16 block sums: every rounding is at most 2^-24 of a partial sum, itself at
most Σ|w||x|.  So (64 + cols/16 + 4) · 2^-24 · Σ|w||x| holds for any order of
summation."""
import numpy as np
import pytest

import oracle as O
from dwim_amd import device as D

pytestmark = pytest.mark.gpu

FORMATS = {"q4_0": (D.Q4_0, 32), "q8_0": (D.Q8_0, 32), "q6_k": (D.Q6_K, 256), "bf16": (D.BF16, 8)}
OFMT = {D.BF16: O.BF16, D.Q4_0: O.Q4_0, D.Q8_0: O.Q8_0, D.Q6_K: O.Q6_K}


@pytest.fixture(scope="module")
def gpu():
    g = D.Hip(0)
    yield g
    g.close()


def weight(name, rows, cols, seed):
    fmt = FORMATS[name][0]
    rng = O.Rng(seed)
    if name == "q6_k":
        w = O.Weight.quantized(O.Q6_K, (rng.floats(rows * cols) * 0.05).reshape(rows, cols))
    else:
        w = {"q4_0": rng.q4_0, "q8_0": rng.q8_0, "bf16": rng.bf16}[name](rows, cols)
    return D.Tensor(fmt, rows, cols, w.quants, w.scales), w.dequantize().reshape(rows, cols).astype(np.float64)


def check(got, w, x, base=0.0):
    n = x.shape[0]
    got = got.reshape(n, -1).astype(np.float64)
    want = x.astype(np.float64) @ w.T + base
    size = np.abs(x).astype(np.float64) @ np.abs(w).T + np.abs(base)
    bound = (64 + w.shape[1] / 16 + 4) * 2.0 ** -24 * size + 1e-37
    over = np.abs(got - want) > bound
    assert not over.any(), f"{over.sum()} of {over.size}, first at {np.argwhere(over)[0]}: " \
                           f"{got[over][0]} for {want[over][0]}, {np.abs(got - want)[over].max() / bound[over].max():.1f} bounds"


# rows at the ends of runs of 16, 32, 64, 128 and 256; tokens at those of every
# kernel's tiles (1, 2, 4, 8, 16, 32, 64, then 128); columns of whole and part
# steps of 64 and units of 128, one run and several
SIZES = [(1, 0, 1), (15, 4, 1), (17, 20, 1), (33, 45, 1), (5, 3, 2), (130, 30, 3), (64, 1, 4), (300, 90, 4), (1, 0, 5), (64, 20, 8),
         (33, 34, 9), (257, 7, 16), (31, 1, 17), (100, 18, 32), (33, 0, 33), (65, 2, 64), (520, 9, 50), (256, 5, 65),
         (257, 3, 127), (130, 4, 129), (520, 9, 300)]


@pytest.mark.parametrize("name", list(FORMATS))
@pytest.mark.parametrize("rows,more,n", SIZES)
def test_matmul_and_add_at_the_edges(gpu, name, rows, more, n):
    block = FORMATS[name][1]
    cols = block * (more + 1) if block >= 32 else 8 * (4 * more + 3)
    t, w = weight(name, rows, cols, rows + cols)
    gw = gpu.upload(t)
    x = O.Rng(n).floats(n * cols).reshape(n, cols)
    gx, out = gpu.buffer(x), gpu.alloc(n * rows)
    gpu.matmul(out, gw, gx)
    first = gpu.read(out)
    check(first, w, x)
    gpu.matmul(out, gw, gx)
    assert first.tobytes() == gpu.read(out).tobytes()
    base = O.Rng(n + 1).floats(n * rows)
    acc = gpu.buffer(base)
    gpu.matmul_add(acc, gw, gx, gpu.alloc(n * rows))
    check(gpu.read(acc), w, x, base.reshape(n, rows).astype(np.float64))


@pytest.mark.parametrize("name", list(FORMATS))
@pytest.mark.parametrize("rows,cols,n", [(15, 512, 1), (96, 2304, 1), (40, 768, 3), (96, 256, 5), (129, 512, 40), (300, 1280, 130)])
def test_swiglu_pair(gpu, name, rows, cols, n):
    (tg, wg), (tu, wu) = weight(name, rows, cols, 7), weight(name, rows, cols, 8)
    x = O.Rng(n).floats(n * cols).reshape(n, cols)
    out, scratch = gpu.alloc(n * rows), gpu.alloc(n * rows)
    gpu.swiglu(out, gpu.upload(tg), gpu.upload(tu), gpu.buffer(x), scratch)
    x64 = x.astype(np.float64)
    g, u = x64 @ wg.T, x64 @ wu.T
    sg, su = np.abs(x64) @ np.abs(wg).T, np.abs(x64) @ np.abs(wu).T
    want = g / (1 + np.exp(-g)) * u
    e = (64 + cols / 16 + 4) * 2.0 ** -24
    # |silu'| <= 1.1, |silu(g)| <= |g|; and the sigmoid's own few roundings
    bound = 1.1 * e * sg * np.abs(u) + np.abs(g) * e * su + 1.1 * e * e * sg * su + 2.0 ** -20 * np.abs(want) + 1e-37
    assert (np.abs(gpu.read(out).reshape(n, rows) - want) <= bound).all()


@pytest.mark.parametrize("name,n", [("q6_k", 33), ("q6_k", 64), ("bf16", 17), ("bf16", 32)])
@pytest.mark.parametrize("rows,cols", [(8192, 1280), (8193, 1280)])
def test_both_sides_of_many_rows(gpu, name, n, rows, cols):
    """The few-token kernel and the batch kernel where matrices of many rows change
    from the one to the other."""
    t, w = weight(name, rows, cols, 9)
    x, base = O.Rng(n).floats(n * cols).reshape(n, cols), O.Rng(n + 1).floats(n * rows)
    acc = gpu.buffer(base)
    gpu.matmul_add(acc, gpu.upload(t), gpu.buffer(x), gpu.alloc(n * rows))
    check(gpu.read(acc), w, x, base.reshape(n, rows).astype(np.float64))


@pytest.mark.parametrize("name", ["q4_0", "q8_0"])
@pytest.mark.parametrize("rows,cols,n", [(5461, 1024, 3), (5462, 1024, 3), (4096, 1024, 4), (4097, 992, 4), (16, 32, 2), (9000, 160, 2),
                                         (2048, 2048, 2), (2049, 2048, 2), (37, 1056, 2), (50, 2080, 2), (17, 1056, 3),
                                         (1, 2080, 1), (18, 4096, 1), (1023, 2176, 1), (1025, 2176, 1), (7, 17408, 1), (30, 16416, 1),
                                         (1024, 2080, 2), (5, 5120, 3), (97, 2336, 4), (1025, 2080, 4)])
def test_few_tokens_of_few_units(gpu, name, rows, cols, n):
    """Both sides of the rules that take two to four tokens over short rows, and up
    to four over few long ones, to the vector ALUs; whole and part units, one wave to 16."""
    t, w = weight(name, rows, cols, 9)
    x, base = O.Rng(n).floats(n * cols).reshape(n, cols), O.Rng(n + 1).floats(n * rows)
    gw, gx, out, acc = gpu.upload(t), gpu.buffer(x), gpu.alloc(n * rows), gpu.buffer(base)
    gpu.matmul(out, gw, gx)
    check(gpu.read(out), w, x)
    gpu.matmul_add(acc, gw, gx, gpu.alloc(n * rows))
    check(gpu.read(acc), w, x, base.reshape(n, rows).astype(np.float64))


@pytest.mark.parametrize("rows,cols", [(16383, 24), (16384, 520), (16387, 40)])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5])
def test_bf16_of_many_rows(gpu, rows, cols, n):
    """The vector kernel's rows a group (1, 2 and 4) and lanes a group (4, 8 and
    64) where they change, and 5 tokens past it; an add and a pair."""
    (t, w), (tu, wu) = weight("bf16", rows, cols, 3), weight("bf16", rows, cols, 4)
    x = O.Rng(n).floats(n * cols).reshape(n, cols)
    base = O.Rng(n + 1).floats(n * rows)
    gw, gx, acc, out = gpu.upload(t), gpu.buffer(x), gpu.buffer(base), gpu.alloc(n * rows)
    gpu.matmul_add(acc, gw, gx, gpu.alloc(n * rows))
    check(gpu.read(acc), w, x, base.reshape(n, rows).astype(np.float64))
    gpu.swiglu(out, gw, gpu.upload(tu), gx, gpu.alloc(n * rows))
    g, u = x.astype(np.float64) @ w.T, x.astype(np.float64) @ wu.T
    sg, su = np.abs(x) @ np.abs(w).T, np.abs(x) @ np.abs(wu).T
    e = (64 + cols / 16 + 4) * 2.0 ** -24
    want = g / (1 + np.exp(-g)) * u
    bound = 1.1 * e * sg * np.abs(u) + np.abs(g) * e * su + 1.1 * e * e * sg * su + 2.0 ** -20 * np.abs(want) + 1e-37
    assert (np.abs(gpu.read(out).reshape(n, rows) - want) <= bound).all()


@pytest.mark.parametrize("name", list(FORMATS))
@pytest.mark.parametrize("n", [1, 2, 4, 5, 16, 40, 65, 130])
def test_activations_of_any_size(gpu, name, n):
    """Rows far beyond f16's range on either side, of zeros, of an outlier
    among tiny values; then infinities and NaN, which stay in their tokens."""
    rows, cols = 70, 512
    t, w = weight(name, rows, cols, 5)
    gw = gpu.upload(t)
    r = np.random.default_rng(n)
    rows_of = [r.normal(0, 1, cols) * 1e30, r.normal(0, 1, cols) * 1e-30, np.zeros(cols),
               np.where(np.arange(cols) == 77, 3e4, r.normal(0, 1e-3, cols)), r.normal(0, 1, cols) * 10.0 ** r.uniform(-9, 9, cols)]
    for shift in range(len(rows_of)):
        x = np.stack([rows_of[(t + shift) % len(rows_of)] for t in range(n)]).astype(np.float32)
        out = gpu.alloc(n * rows)
        gpu.matmul(out, gw, gpu.buffer(x))
        check(gpu.read(out), w, x)
    if name == "q6_k" and n < 16:
        return  # int8 planes, whose scale is a group's largest value: an infinity's results are NaN
    x = r.normal(0, 1, (n, cols)).astype(np.float32)
    x[0, 3], clean = np.inf, x.copy()
    if n > 1:
        x[1, 100] = np.nan
    if n > 2:
        x[2, 40] = -np.inf
    out = gpu.alloc(n * rows)
    gpu.matmul(out, gw, gpu.buffer(x))
    got = gpu.read(out).reshape(n, rows)
    with np.errstate(invalid="ignore"):
        assert np.array_equal(got[0], np.where(w[:, 3] == 0, np.nan, np.inf * w[:, 3]).astype(np.float32), equal_nan=True)
        if n > 1:
            assert np.isnan(got[1]).all()
        if n > 2:
            assert np.array_equal(got[2], np.where(w[:, 40] == 0, np.nan, -np.inf * w[:, 40]).astype(np.float32), equal_nan=True)
    if n > 3:
        check(got[3:], w, clean[3:])


def errors(gpu, name, rows, cols, n, seed):
    """results less the true ones, over the true ones' root mean square
    (an add to zeros: Q6_K's plain products of few tokens run on int8 planes)"""
    t, w = weight(name, rows, cols, seed)
    x = np.random.default_rng(seed).standard_normal((n, cols), dtype=np.float32)
    out = gpu.buffer(np.zeros(n * rows, np.float32))
    gpu.matmul_add(out, gpu.upload(t), gpu.buffer(x), gpu.alloc(n * rows))
    want = x.astype(np.float64) @ w.T
    return (gpu.read(out).reshape(n, rows) - want) / np.sqrt((want ** 2).mean())


FEW, BATCH = [1, 2, 5, 16], [40, 130]  # tokens through the one kernel and the other


@pytest.mark.parametrize("name", list(FORMATS))
@pytest.mark.parametrize("n", FEW + BATCH)
def test_products_err_up_as_often_as_down(gpu, name, n):
    """The matrix cores' sums round down.  Unless that is made up for, the mean
    error over 5120 columns is 4e-8 to 8e-8 of the results' size, where that of
    unbiased errors of 1.2e-7 over 2048 rows and n tokens is under
    1.2e-7 / sqrt(2048 n) (here: five times that)."""
    err = errors(gpu, name, 2048, 5120, n, 11)
    assert abs(err.mean()) <= 5 * 1.2e-7 / np.sqrt(err.size)


@pytest.mark.parametrize("name", list(FORMATS))
@pytest.mark.parametrize("n", FEW + BATCH)
def test_long_rows_round_no_more_than_f32_sums(gpu, name, n):
    """17408 columns.  A chain of k sums that grow to the result's size has
    k/2 · u² of error, u = 2^-24 · 0.42 (the mean square of a rounding): 8 block
    sums a unit, at most 34 units a run of columns, 8 runs, and about 8 inside
    the blocks, 29 u² = (1.35e-7)².  On the vector ALUs it was 1.3e-7 (bf16 1.4e-7),
    with every block's sum joining the row's (and rounding down) 1.7e-7 to 2.7e-7."""
    err = errors(gpu, name, 512, 17408, n, 12)
    assert np.sqrt((err ** 2).mean()) <= 1.5e-7


@pytest.mark.parametrize("name", list(FORMATS))
@pytest.mark.parametrize("n", [1, 20, 65, 130])
def test_an_outlier_does_not_cost_other_columns_their_bits(gpu, name, n):
    """A value 1e10 times the others, under weights that are 0 from there to
    column 512 (as far as an activation's parts may share its scale): the results are the
    other columns', within the bound of their own sizes."""
    rows, cols = 70, 2304
    fmt = FORMATS[name][0]
    rng = O.Rng(3)
    if name == "q6_k":
        vals = (rng.floats(rows * cols) * 0.05).reshape(rows, cols)
        vals[:, :512] = 0
        w = O.Weight.quantized(O.Q6_K, vals)
    else:
        w = {"q4_0": rng.q4_0, "q8_0": rng.q8_0, "bf16": rng.bf16}[name](rows, cols)
        (w.quants if name == "bf16" else w.scales).reshape(rows, -1)[:, :512 if name == "bf16" else 16] = 0
    x = np.random.default_rng(n).standard_normal((n, cols), dtype=np.float32)
    x[:, 7] = 1e10
    out = gpu.buffer(np.zeros(n * rows, np.float32))
    gpu.matmul_add(out, gpu.upload(D.Tensor(fmt, rows, cols, w.quants, w.scales)), gpu.buffer(x), gpu.alloc(n * rows))
    check(gpu.read(out), w.dequantize().reshape(rows, cols).astype(np.float64), x)


@pytest.mark.parametrize("name", list(FORMATS))
def test_whole_rounds_of_tiles_and_a_second_launch(gpu, name):
    """9 × 64 tiles of 4096 tokens, 512 of them whole (two to each of 256 CUs) and 64 in
    parts, then 33 tokens more in a launch of their own; a product and a pair.
    5120 columns: at most 32 roundings a run of 512 (Q6_K 16 of 256), 10 (20) of
    the totals, about 8 inside the blocks: 22 u² = (1.2e-7)² (see above)."""
    n, cols = 4096 + 33, 5120
    x = np.random.default_rng(5).standard_normal((n, cols), dtype=np.float32)
    some = np.unique(np.concatenate([np.arange(0, n, 97), [63, 64, 3583, 3584, 4095, 4096, n - 1]]))
    gx, xs = gpu.buffer(x), x[some].astype(np.float64)
    t, w = weight(name, 2304, cols, 6)
    out = gpu.alloc(n * 2304)
    gpu.matmul(out, gpu.upload(t), gx)
    got = gpu.read(out).reshape(n, -1)[some]
    check(got, w, x[some])
    want = xs @ w.T
    assert np.linalg.norm(got - want) <= 1.4e-7 * np.linalg.norm(want)
    (tg, wg), (tu, wu) = weight(name, 1152, cols, 7), weight(name, 1152, cols, 8)
    out = gpu.alloc(n * 1152)
    gpu.swiglu(out, gpu.upload(tg), gpu.upload(tu), gx, gpu.alloc(n * 1152))
    g, u = xs @ wg.T, xs @ wu.T
    sg, su = np.abs(xs) @ np.abs(wg).T, np.abs(xs) @ np.abs(wu).T
    with np.errstate(over="ignore"):
        want = g / (1 + np.exp(-g)) * u
    e = (64 + cols / 16 + 4) * 2.0 ** -24
    bound = 1.1 * e * sg * np.abs(u) + np.abs(g) * e * su + 1.1 * e * e * sg * su + 2.0 ** -20 * np.abs(want) + 1e-37
    assert (np.abs(gpu.read(out).reshape(n, -1)[some] - want) <= bound).all()


@pytest.mark.parametrize("rows,cols", [(1, 256), (17, 512), (40, 1280), (64, 1536), (100, 2304), (8200, 1280), (33, 5120), (50, 20480)])
def test_q4_k_one_token_converts_its_activations(gpu, rows, cols):
    """One token through Q4_K (the planes made by each wave for its own 1 to 6
    blocks), the SwiGLU pair and the add.  A weight is d·sc·q less dmin·m, each
    at most its block's range, 2·max|w|; activations to 2^-24 of their group's
    largest, sums rounded as above."""
    r = np.random.default_rng(cols + rows)
    def make():
        w = O.Weight.quantized(O.Q4_K, (r.normal(0, 0.05, (rows, cols))).astype(np.float32))
        return gpu.upload(D.Tensor(D.Q4_K, rows, cols, w.quants)), w.dequantize().reshape(rows, cols).astype(np.float64)
    (g, wg), (u, wu) = make(), make()
    x = (r.normal(0, 1, cols) * 10.0 ** r.uniform(-3, 3, cols)).astype(np.float32)
    x64 = x.astype(np.float64)
    reach = np.repeat(np.abs(x64).reshape(-1, 16).max(1), 16)  # a group's error is its largest's
    e = (64 + cols / 16 + 4) * 2.0 ** -24
    def size(w):
        return ((np.abs(w) + 2 * np.abs(w).max()) * reach).sum(1)
    base = r.normal(0, 1, rows).astype(np.float32)
    out = gpu.buffer(base)
    gpu.matmul_add(out, g, gpu.buffer(x), gpu.alloc(rows))
    assert (np.abs(gpu.read(out) - (base + wg @ x64)) <= e * (size(wg) + np.abs(base))).all()
    out, scratch = gpu.alloc(rows), gpu.alloc(rows)
    gpu.swiglu(out, g, u, gpu.buffer(x), scratch)
    a, b = wg @ x64, wu @ x64
    with np.errstate(over="ignore"):
        want = a / (1 + np.exp(-a)) * b
    bound = 1.1 * e * size(wg) * np.abs(b) + np.abs(a) * e * size(wu) + 1.1 * e * e * size(wg) * size(wu) + 2.0 ** -20 * np.abs(want)
    assert (np.abs(gpu.read(out) - want) <= bound + 1e-37).all()


@pytest.mark.parametrize("rows,cols,n", [(1, 256, 5), (33, 512, 8), (100, 5120, 9), (70, 2304, 16), (257, 1280, 17), (2100, 4096, 17),
                                         (40, 17408, 32), (130, 768, 33), (2100, 4096, 40), (2080, 4352, 64), (64, 256, 64)])
def test_q4_k_five_to_sixty_four_tokens(gpu, rows, cols, n):
    """Q4_K through the few-token kernel and the batch kernel's tiles of 32 and
    64 tokens (larger matrices), a plain product, the add and the pair, bounds as
    above."""
    r = np.random.default_rng(cols + rows + n)
    def make():
        w = O.Weight.quantized(O.Q4_K, (r.normal(0, 0.05, (rows, cols))).astype(np.float32))
        return gpu.upload(D.Tensor(D.Q4_K, rows, cols, w.quants)), w.dequantize().reshape(rows, cols).astype(np.float64)
    (g, wg), (u, wu) = make(), make()
    x = r.normal(0, 1, (n, cols)).astype(np.float32)
    x[n // 2] *= 1e30
    x[n - 1] *= 1e-30
    x64, e = x.astype(np.float64), (64 + cols / 16 + 4) * 2.0 ** -24
    def size(w):
        return np.abs(x64) @ (np.abs(w) + 2 * np.abs(w).max()).T
    gx, out, scratch = gpu.buffer(x), gpu.alloc(n * rows), gpu.alloc(n * rows)
    a, b = x64 @ wg.T, x64 @ wu.T
    gpu.matmul(out, g, gx)
    assert (np.abs(gpu.read(out).reshape(n, rows) - a) <= e * size(wg) + 1e-37).all()
    base = r.normal(0, 1, (n, rows)).astype(np.float32)
    acc = gpu.buffer(base)
    gpu.matmul_add(acc, g, gx, scratch)
    assert (np.abs(gpu.read(acc).reshape(n, rows) - (a + base)) <= e * (size(wg) + np.abs(base)) + 1e-37).all()
    gpu.swiglu(out, g, u, gx, scratch)
    got = gpu.read(out).reshape(n, rows)
    with np.errstate(over="ignore"):
        want = a / (1 + np.exp(-a)) * b
    bound = 1.1 * e * size(wg) * np.abs(b) + np.abs(a) * e * size(wu) + 1.1 * e * e * size(wg) * size(wu) + 2.0 ** -20 * np.abs(want)
    fine = np.arange(n) != n // 2  # (that row's products overflow f32)
    assert (np.abs(got - want) <= bound + 1e-37)[fine].all()


@pytest.mark.parametrize("size", [256, 1280, 2560])
@pytest.mark.parametrize("n", [1, 3, 5, 15, 16, 40, 64, 65])
def test_q4_k_products_in_place(gpu, size, n):
    """A square Q4_K product, the add and the pair with the result in the
    input's own buffer, against the same into another buffer.  Where in-place
    calls take another kernel the two differ by both kernels' roundings: the
    bound of a result in the tests above, twice (2^-24 as there, of sums that
    are at most the row's |w||x| and the blocks' ranges)."""
    r = np.random.default_rng(size + n)
    def make():
        w = O.Weight.quantized(O.Q4_K, (r.normal(0, 0.05, (size, size))).astype(np.float32))
        return gpu.upload(D.Tensor(D.Q4_K, size, size, w.quants)), w.dequantize().reshape(size, size).astype(np.float64)
    (g, wg), (u, wu) = make(), make()
    x = r.normal(0, 1, (n, size)).astype(np.float32)
    x64, e = np.abs(x.astype(np.float64)), 2 * (64 + size / 16 + 4) * 2.0 ** -24
    def bound(w):
        return e * (x64 @ (np.abs(w) + 2 * np.abs(w).max()).T)
    def both(op):
        apart, inside, out = gpu.buffer(x.ravel()), gpu.buffer(x.ravel()), gpu.buffer(x.ravel())
        op(out, apart)
        op(inside, inside)
        return gpu.read(out).reshape(n, size).astype(np.float64), gpu.read(inside).reshape(n, size).astype(np.float64)
    want, got = both(lambda o, i: gpu.matmul(o, g, i))
    assert (np.abs(got - want) <= bound(wg)).all()
    scratch = gpu.alloc(n * size)
    want, got = both(lambda o, i: gpu.matmul_add(o, g, i, scratch))
    assert (np.abs(got - want) <= bound(wg) + e * x64).all()
    a, b = np.abs(x.astype(np.float64) @ wg.T), np.abs(x.astype(np.float64) @ wu.T)
    want, got = both(lambda o, i: gpu.swiglu(o, g, u, i, scratch))
    # |silu'| <= 1.1 and |silu(g)| <= |g|
    assert (np.abs(got - want) <= 1.1 * bound(wg) * (b + bound(wu)) + a * bound(wu) + 2.0 ** -20 * np.abs(want)).all()


def q4_k_errors(gpu, rows, cols, n, seed, some):
    """results less the true ones for some of the tokens, over the true ones'
    root mean square"""
    r = np.random.default_rng(seed)
    w = O.Weight.quantized(O.Q4_K, r.standard_normal((rows, cols), dtype=np.float32) * np.float32(0.05))
    x = r.standard_normal((n, cols), dtype=np.float32)
    out = gpu.alloc(n * rows)
    gpu.matmul(out, gpu.upload(D.Tensor(D.Q4_K, rows, cols, w.quants)), gpu.buffer(x))
    want = x[some].astype(np.float64) @ w.dequantize().reshape(rows, cols).astype(np.float64).T
    return (gpu.read(out).reshape(n, rows)[some] - want) / np.sqrt((want ** 2).mean())


def test_q4_k_batches_err_up_as_often_as_down(gpu):
    """As above, for the GEMM of 65 tokens and more, whose unbiased errors are
    under 4e-7 (mean error of plain sums 2.4e-8)."""
    err = q4_k_errors(gpu, 1024, 5120, 130, 21, slice(None))
    assert abs(err.mean()) <= 5 * 4e-7 / np.sqrt(err.size)


def test_q4_k_long_rows_in_whole_tiles(gpu):
    """8 × 32 tiles, a whole round of 256 CUs, 32 blocks a row.  A block is 34
    MFMAs, each two links of a chain (its 16 products come in two eights), and a
    change of units: 32 blocks are N = 2240 roundings at sizes that grow to the
    result's.  In one chain that is N/2 · u² of error (u as above), 8.5e-7, in two
    runs of 16 blocks N/4 · u², 6.0e-7; the line lies between."""
    err = q4_k_errors(gpu, 2048, 8192, 4096, 22, slice(0, 4096, 61))
    assert np.sqrt((err ** 2).mean()) <= 7e-7


@pytest.mark.parametrize("name,cols", [("q8_0", 4096), ("q4_0", 8160), ("q6_k", 5120)])
def test_uploads_of_more_than_a_slab(gpu, name, cols):
    """A matrix goes to the device 64 MB at a time: the rows at the ends of a
    slab, read back, and those of the last tile."""
    fmt = FORMATS[name][0]
    row_bytes = {"q8_0": cols, "q4_0": cols // 2, "q6_k": cols // 256 * 210}[name]
    slab = (64 << 20) // row_bytes // 16 * 16
    rows = slab + 17
    rng = np.random.default_rng(1)
    if name == "q6_k":
        blocks = rng.integers(0, 256, (rows, cols // 256, 210), dtype=np.uint8)
        blocks[..., 208:] = np.frombuffer(np.float16(0.01).tobytes(), np.uint8)
        quants, scales = blocks.ravel(), None
    else:
        quants = rng.integers(0, 256, rows * row_bytes, dtype=np.uint8)
        quants = quants.view(np.int8) if name == "q8_0" else quants
        scales = rng.uniform(0.001, 0.01, rows * cols // 32).astype(np.float16).view(np.uint16)
    gw = gpu.upload(D.Tensor(fmt, rows, cols, quants, scales))
    for r in (0, 15, 16, slab - 1, slab, slab + 15, slab + 16):
        out = gpu.alloc(cols)
        gpu.embed(out, gw, [r])
        one = slice(r * row_bytes, (r + 1) * row_bytes), slice(r * (cols // 32), (r + 1) * (cols // 32))
        want = O.Weight(OFMT[fmt], 1, cols, quants[one[0]], None if scales is None else scales[one[1]]).dequantize()
        assert np.array_equal(gpu.read(out), np.asarray(want, np.float32).ravel()), r
