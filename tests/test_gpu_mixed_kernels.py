"""The mixed-layer decoder's kernels one by one, through the C ABI, against the
plain float64 statement of each mechanism."""
import ctypes

import numpy as np
import pytest
import torch

import mixed_model as mm
import mixer_oracle as mo
import qllm_hip as qh
from kernel_util import BF16, F32, close, on, packed, padded, steps, torch_type

pytestmark = pytest.mark.gpu

# ---- linear --------------------------------------------------------------------


def padded_input(device, x, columns, element):
    out = torch.zeros((x.shape[0], padded(columns, 64)), dtype=torch_type(element), device=device)
    out[:, :x.shape[1]] = on(device, x)
    return out


@pytest.mark.parametrize("element", [F32, BF16])
@pytest.mark.parametrize("batch", [1, 2, 16, 17, 33, 64, 65, 130, 300])
def test_linear_segments_of_every_epilogue(device, element, batch):
    rng = np.random.default_rng(batch)
    shapes = [(70, 200), (33, 90)]
    matrices = [mm.bf16(rng.standard_normal(s) / np.sqrt(s[1])) for s in shapes]
    gate, up = (mm.bf16(rng.standard_normal((45, 200)) / 14) for _ in range(2))
    inputs = [mm.bf16(rng.standard_normal((batch, s[1]))) for s in shapes]
    first = packed(device, [(matrices[0], 0, 1, 0)], 70, 200)
    second = packed(device, [(matrices[1], 0, 1, 0)], 33, 90)
    pair = packed(device, [(gate, 0, 2, 0), (up, 1, 2, 0)], 96, 200)
    x0 = padded_input(device, inputs[0], 200, element)
    x1 = padded_input(device, inputs[1], 90, element)
    base = rng.standard_normal((batch, 36)).astype(np.float32)
    store = torch.full((batch, 72), 7.0, device=device)
    add = on(device, base)
    gated = torch.zeros((batch, 64), dtype=torch_type(element), device=device)
    segments = (qh.LinearSegment * 3)(
        qh.LinearSegment(qh.ptr(first), qh.ptr(x0), qh.ptr(store), 80, 256, 256, 72, 70,
                         qh.LINEAR_STORE, 0, 0),
        qh.LinearSegment(qh.ptr(second), qh.ptr(x1), qh.ptr(add), 48, 128, 128, 36, 33,
                         qh.LINEAR_ADD, 0, 0),
        qh.LinearSegment(qh.ptr(pair), qh.ptr(x0), qh.ptr(gated), 96, 256, 256, 64, 45,
                         qh.LINEAR_GATED, 0, 0))
    qh.call("qllm_linear_batch", segments, 3, batch, element, None)
    torch.cuda.synchronize()
    products = [x.astype(np.float64) @ m.T.astype(np.float64)
                for x, m in zip(inputs, matrices)]
    # bf16 inputs and weights, F32 sums: both modes give the product itself
    close(store[:, :70], products[0], F32, "store")
    assert torch.all(store[:, 70:] == 7.0)
    close(add[:, :33], base[:, :33] + products[1], F32, "add")
    assert np.array_equal(add[:, 33:].cpu().numpy(), base[:, 33:])
    x = inputs[0].astype(np.float64)
    want = mo.gelu_tanh(x @ gate.T.astype(np.float64)) * (x @ up.T.astype(np.float64))
    close(gated[:, :45], want, element, "gated")
    assert torch.all(gated[:, 45:] == 0)


@pytest.mark.parametrize("batch", [1, 16, 17, 33, 64, 65, 200])
def test_linear_takes_all_bits_of_32_bit_inputs(device, batch):
    """Inputs with 24 significant bits over 60 powers of two, the largest finite
    value, infinities and a NaN whose upper half reads as an infinity."""
    rng = np.random.default_rng(batch)
    matrix = mm.bf16(rng.standard_normal((70, 192)) / 14)
    matrix[:, 190] = 0.25
    x = (rng.standard_normal((batch, 192)) * np.exp2(rng.integers(-30, 31, (batch, 192)))
         ).astype(np.float32)
    odd = batch // 2
    special = {0: np.float32(3.4028235e38), 1: np.inf, 2: -np.inf,
               3: np.uint32(0x7f800001).view(np.float32)}.items()
    weights = packed(device, [(matrix, 0, 1, 0)], 70, 192)
    out = torch.zeros((batch, 72), device=device)

    def run(values):
        d_x = padded_input(device, values, 192, F32)
        segment = qh.LinearSegment(qh.ptr(weights), qh.ptr(d_x), qh.ptr(out), 80, 192, 192,
                                   72, 70, qh.LINEAR_STORE, 0, 0)
        qh.call("qllm_linear_batch", ctypes.byref(segment), 1, batch, F32, None)
        return out[:, :70].cpu().numpy().astype(np.float64)

    # every product is exact, every one of the 3 x 192 additions of a sum rounds
    # by at most 2^-24 of the magnitudes' sum, in whatever order
    magnitude = np.abs(x.astype(np.float64)) @ np.abs(matrix.T.astype(np.float64))
    bound = 3 * 192 * 2.0 ** -24 * magnitude
    want = x.astype(np.float64) @ matrix.T.astype(np.float64)
    assert (np.abs(run(x) - want) <= bound).all()
    for _, value in special:
        changed = np.zeros_like(x)
        changed[odd, 190] = value
        with np.errstate(invalid="ignore"):
            expected = changed[odd, 190].astype(np.float64) * 0.25
        got = run(changed)
        assert np.array_equal(got[odd], np.full(70, expected), equal_nan=True)
        assert not np.delete(got, odd, axis=0).any()


@pytest.mark.parametrize("batch", [16, 64, 200])
def test_linear_takes_small_32_bit_inputs(device, batch):
    """One input a row, weights of one: all of 24 significant bits from 2^-110 on,
    below within bf16's smallest step."""
    rng = np.random.default_rng(batch)
    exponents = np.linspace(-149, -96, batch).astype(int)
    values = ((1.0 + rng.integers(0, 1 << 23, batch) * 2.0 ** -23) *
              np.exp2(exponents.astype(np.float64)) *
              rng.choice([-1.0, 1.0], batch)).astype(np.float32)
    x = np.zeros((batch, 64), dtype=np.float32)
    x[np.arange(batch), np.arange(batch) % 64] = values
    weights = packed(device, [(np.ones((16, 64), dtype=np.float32), 0, 1, 0)], 16, 64)
    d_x = padded_input(device, x, 64, F32)
    out = torch.zeros((batch, 16), device=device)
    segment = qh.LinearSegment(qh.ptr(weights), qh.ptr(d_x), qh.ptr(out), 16, 64, 64, 16, 16,
                               qh.LINEAR_STORE, 0, 0)
    qh.call("qllm_linear_batch", ctypes.byref(segment), 1, batch, F32, None)
    got = out.cpu().numpy().astype(np.float64)
    error = np.abs(got - values[:, None].astype(np.float64))
    assert not error[np.abs(values) >= 2.0 ** -110].any()
    assert (error < 2.0 ** -133).all()


@pytest.mark.parametrize("batch", [1, 16, 17, 33, 64, 65, 200, 1000])
@pytest.mark.parametrize("epilogue", ["store", "gated"])
def test_weights_that_are_no_numbers_meet_32_bit_inputs(device, batch, epilogue):
    """Infinite and NaN weights give what a multiply-add gives, whichever parts of
    an input are zero: inputs of one, sixteen and 24 significant bits, zeros,
    infinities."""
    rng = np.random.default_rng(batch)
    rows = 2112 if batch == 1000 else 64     # (the wider form of the tall launch)
    inputs = np.array([1.0, -1.5, 1.0 + 2.0 ** -15, 1.0 + 2.0 ** -23, -3.0e-30, 0.0, np.inf,
                       -np.inf], dtype=np.float32)
    x = np.zeros((batch, 192), dtype=np.float32)
    x[:, 7] = inputs[np.arange(batch) % len(inputs)]
    x[:, 100] = rng.standard_normal(batch)
    matrix = mm.bf16(rng.standard_normal((rows, 192)))
    matrix[:, 7] = np.resize(np.array([np.inf, -np.inf, np.nan, 0.5], dtype=np.float32), rows)
    x[:, 150] = 30.0     # the gate's input, and silu(30) is 30 in 32 bits
    d_x = padded_input(device, x, 192, F32)
    matrix[:, 150] = 0.0
    with np.errstate(invalid="ignore"):
        products = [x[:, k, None].astype(np.float64) * matrix[:, k] for k in (7, 100)]
        want = products[0] + products[1]
    if epilogue == "store":
        weights = packed(device, [(matrix, 0, 1, 0)], rows, 192)
        out = torch.zeros((batch, rows), device=device)
        segment = qh.LinearSegment(qh.ptr(weights), qh.ptr(d_x), qh.ptr(out), rows, 192, 192,
                                   rows, rows, qh.LINEAR_STORE, 0, 0)
    else:
        gate = np.zeros((rows, 192), dtype=np.float32)
        gate[:, 150] = 1.0
        want, products = 30.0 * want, [30.0 * p for p in products]
        want[np.isinf(x[:, 7])] = np.nan      # meets the gate's zeros
        weights = packed(device, [(gate, 0, 2, 0), (matrix, 1, 2, 0)], 2 * rows, 192)
        out = torch.zeros((batch, rows), device=device)
        segment = qh.LinearSegment(qh.ptr(weights), qh.ptr(d_x), qh.ptr(out), 2 * rows, 192,
                                   192, rows, rows, qh.LINEAR_GATED, 1, 0)   # SiLU
    qh.call("qllm_linear_batch", ctypes.byref(segment), 1, batch, F32, None)
    got = out.cpu().numpy().astype(np.float64)
    finite = np.isfinite(want)
    assert np.array_equal(got[~finite], want[~finite], equal_nan=True)
    # six exact products of parts, a rounding for each that is added, and the gate's
    bound = 8 * 2.0 ** -24 * (np.abs(products[0]) + np.abs(products[1]))
    assert (np.abs(got[finite] - want[finite]) <= bound[finite]).all()


@pytest.mark.parametrize("element", [F32, BF16])
@pytest.mark.parametrize("splits", [1, 3, 7])
def test_linear_partials_and_side_by_side_columns(device, element, splits):
    rng = np.random.default_rng(splits)
    left, right = (mm.bf16(rng.standard_normal((50, n)) / 12) for n in (70, 100))
    weights = packed(device, [(left, 0, 1, 0), (right, 0, 1, 128)], 50, 256)
    x = np.zeros((5, 256), dtype=np.float32)
    x[:, :70] = mm.bf16(rng.standard_normal((5, 70)))
    x[:, 128:228] = mm.bf16(rng.standard_normal((5, 100)))
    d_x = padded_input(device, x, 256, element)
    out = torch.zeros((splits, 5, 52), device=device)
    segment = qh.LinearSegment(qh.ptr(weights), qh.ptr(d_x), qh.ptr(out), 64, 256, 256, 52, 50,
                               qh.LINEAR_PARTIALS, 0, splits)
    qh.call("qllm_linear_batch", ctypes.byref(segment), 1, 5, element, None)
    torch.cuda.synchronize()
    want = x[:, :70].astype(np.float64) @ left.T + x[:, 128:228].astype(np.float64) @ right.T
    close(out.sum(0)[:, :50], want, F32)


@pytest.mark.parametrize("element", [F32, BF16])
@pytest.mark.parametrize("rows,columns,batch", [
    (50, 192, 65), (300, 512, 129), (33, 64, 200), (1100, 1984, 67)])
def test_linear_partials_of_tall_batches(device, element, rows, columns, batch):
    """Parts of every count of a batch of more than 64 rows, among them more parts
    than steps of K, uneven shares and ragged tiles; the count the library advises."""
    rng = np.random.default_rng(rows)
    matrix = mm.bf16(rng.standard_normal((rows, columns)) / np.sqrt(columns))
    x = mm.bf16(rng.standard_normal((batch, columns)))
    weights = packed(device, [(matrix, 0, 1, 0)], rows, columns)
    d_x = padded_input(device, x, columns, element)
    stride = padded(rows, 4) + 4
    want = x.astype(np.float64) @ matrix.T.astype(np.float64)
    advised = qh.call("qllm_linear_parts", padded(rows, 16), columns, batch, element)
    assert 1 <= advised <= 16 and (advised == 1 or advised * batch <= 8192)
    for parts in sorted({1, 2, 3, 7, 16, advised}):
        out = torch.full((parts, batch, stride), 7.0, device=device)
        segment = qh.LinearSegment(qh.ptr(weights), qh.ptr(d_x), qh.ptr(out),
                                   padded(rows, 16), columns, columns, stride, rows,
                                   qh.LINEAR_PARTIALS, 0, parts)
        qh.call("qllm_linear_batch", ctypes.byref(segment), 1, batch, element, None)
        close(out[:, :, :rows].sum(0), want, F32)
        assert torch.all(out[:, :, rows:] == 7.0)


def test_linear_tall_tiles_of_all_sizes(device):
    """Ragged tiles of 64 batch rows (the larger ones:
    test_linear_tall_forms_of_every_epilogue)."""
    rng = np.random.default_rng(3)
    for rows, columns, batch in ((2100, 128, 700), (4096, 64, 1030), (300, 320, 129)):
        w = mm.bf16(rng.standard_normal((rows, columns)) / 12)
        x = mm.bf16(rng.standard_normal((batch, columns)))
        weights = packed(device, [(w, 0, 1, 0)], rows, columns)
        d_x = padded_input(device, x, columns, BF16)
        out = torch.zeros((batch, padded(rows, 4)), device=device)
        segment = qh.LinearSegment(qh.ptr(weights), qh.ptr(d_x), qh.ptr(out), padded(rows, 16),
                                   padded(columns, 64), padded(columns, 64), padded(rows, 4),
                                   rows, qh.LINEAR_STORE, 0, 0)
        qh.call("qllm_linear_batch", ctypes.byref(segment), 1, batch, BF16, None)
        torch.cuda.synchronize()
        close(out[:, :rows], x.astype(np.float64) @ w.T.astype(np.float64), F32)


# (batch rows, weight rows) of a workgroup of a whole launch and of one in parts
@pytest.mark.parametrize("element,rows,columns,batch,whole,parts,cut", [
    (BF16, 2090, 192, 2900, (128, 128), 2, (128, 256)),
    (BF16, 8170, 192, 1901, (128, 256), 5, (128, 256)),     # more parts than steps of K
    (BF16, 4070, 320, 1000, (64, 128), 3, (128, 128)),
    (BF16, 12270, 192, 333, (64, 128), 5, (128, 256)),
    (F32, 2090, 192, 2900, (64, 256), 3, (64, 256)),
    (F32, 12270, 192, 333, (64, 128), 2, (64, 256)),
    (F32, 4070, 192, 70, (64, 128), 5, (64, 256))])
def test_linear_tall_forms_of_every_epilogue(device, element, rows, columns, batch, whole,
                                             parts, cut):
    """Every form of the tall launch, with the epilogues of which a layer makes use:
    rows and batches that end inside a workgroup, strides of no whole vectors."""
    rng = np.random.default_rng(rows + batch)
    w = mm.bf16(rng.standard_normal((rows, columns)) / np.sqrt(columns))
    x = mm.bf16(rng.standard_normal((batch, columns)))
    want = x.astype(np.float64) @ w.T.astype(np.float64)
    weights, d_x = packed(device, [(w, 0, 1, 0)], rows, columns), padded_input(device, x,
                                                                              columns, element)

    def run(out, stride, epilogue, count, form, matrix=weights, height=rows, outputs=rows):
        segment = qh.LinearSegment(qh.ptr(matrix), qh.ptr(d_x), qh.ptr(out),
                                   padded(height, 16), columns, columns, stride, outputs,
                                   epilogue, 0, count)
        found = qh.LaunchLayout()
        qh.call("qllm_linear_layout", ctypes.byref(segment), 1, batch, element,
                ctypes.byref(found))
        assert (found.batch_rows, found.weight_rows) == form
        qh.call("qllm_linear_batch", ctypes.byref(segment), 1, batch, element, None)
        torch.cuda.synchronize()

    stride = padded(rows, 4)
    out = torch.full((batch, stride), 7.0, device=device)
    run(out, stride, qh.LINEAR_STORE, 0, whole)
    close(out[:, :rows], want, F32, "store")
    assert torch.all(out[:, rows:] == 7.0)
    for stride in (padded(rows, 4), rows + 1):
        base = rng.standard_normal((batch, stride)).astype(np.float32)
        out = on(device, base)
        run(out, stride, qh.LINEAR_ADD, 0, whole)
        close(out[:, :rows], base[:, :rows] + want, F32, "add")
        assert np.array_equal(out[:, rows:].cpu().numpy(), base[:, rows:])
        out = torch.full((parts, batch, stride), 7.0, device=device)
        run(out, stride, qh.LINEAR_PARTIALS, parts, cut)
        close(out[:, :, :rows].double().sum(0), want, F32, "partials")
        assert torch.all(out[:, :, rows:] == 7.0)
    half = rows // 2
    pair = packed(device, [(w[:half], 0, 2, 0), (w[half:2 * half], 1, 2, 0)],
                  2 * padded(half, 16), columns)
    out = torch.zeros((batch, padded(half, 4)), dtype=torch_type(element), device=device)
    run(out, padded(half, 4), qh.LINEAR_GATED, 0, whole, pair, 2 * padded(half, 16), half)
    gated = mo.gelu_tanh(want[:, :half]) * want[:, half:2 * half]
    close(out[:, :half], gated, element, "gated")
    assert torch.all(out[:, half:] == 0)


@pytest.mark.parametrize("rows,batch,form", [
    (70, 65, (64, 128)),          # a workgroup to a CU: loads first
    (3088, 777, (64, 128)),       # several to a CU
    (2090, 2900, (128, 128)), (8170, 1901, (128, 256))])
@pytest.mark.parametrize("columns,stride", [(64, 64), (128, 192), (256, 264), (448, 448),
                                            (576, 1024), (640, 640)])
def test_linear_tall_steps_ahead(device, rows, batch, form, columns, stride):
    """Launches of one to ten steps of K, fewer and more than the steps that a workgroup
    asks for ahead, over input rows with a gap between them."""
    rng = np.random.default_rng(rows + columns)
    w = mm.bf16(rng.standard_normal((rows, columns)) / np.sqrt(columns))
    x = mm.bf16(rng.standard_normal((batch, columns)))
    weights = packed(device, [(w, 0, 1, 0)], rows, columns)
    d_x = torch.full((batch, stride), float("nan"), dtype=torch.bfloat16, device=device)
    d_x[:, :columns] = on(device, x)
    out = torch.zeros((batch, padded(rows, 4)), device=device)
    segment = qh.LinearSegment(qh.ptr(weights), qh.ptr(d_x), qh.ptr(out), padded(rows, 16),
                               columns, stride, padded(rows, 4), rows, qh.LINEAR_STORE, 0, 0)
    found = qh.LaunchLayout()
    qh.call("qllm_linear_layout", ctypes.byref(segment), 1, batch, BF16, ctypes.byref(found))
    assert (found.batch_rows, found.weight_rows) == form
    qh.call("qllm_linear_batch", ctypes.byref(segment), 1, batch, BF16, None)
    got = out[:, :rows].double()
    x, w = on(device, x).double(), on(device, w).double()
    # exact products, every one of `columns` additions of a sum rounds by at most 2^-24
    bound = columns * 2.0 ** -24 * (x.abs() @ w.abs().T)
    assert ((got - x @ w.T).abs() <= bound).all()


def test_linear_of_rows_far_apart(device):
    """Rows 2^24 values apart, past a lane's 32-bit offset over 128 of them."""
    rng = np.random.default_rng(5)
    rows, batch, columns, stride = 40, 70, 128, 1 << 24
    w = mm.bf16(rng.standard_normal((rows, columns)) / 8)
    x = mm.bf16(rng.standard_normal((batch, columns)))
    weights = packed(device, [(w, 0, 1, 0)], rows, columns)
    d_x = torch.empty((batch, stride), dtype=torch.bfloat16, device=device)
    d_x[:, :columns] = on(device, x)
    out = torch.zeros((batch, rows), device=device)
    segment = qh.LinearSegment(qh.ptr(weights), qh.ptr(d_x), qh.ptr(out), 48, columns, stride,
                               rows, rows, qh.LINEAR_STORE, 0, 0)
    qh.call("qllm_linear_batch", ctypes.byref(segment), 1, batch, BF16, None)
    close(out, x.astype(np.float64) @ w.T.astype(np.float64), F32)


@pytest.mark.parametrize("rows,batch,form", [(70, 130, (64, 128)), (40000, 200, (128, 128))])
@pytest.mark.parametrize("columns", [64, 448])
def test_linear_tall_forms_of_rows_far_apart(device, rows, batch, form, columns):
    """The tall forms over rows 2^24 + 8 values apart, in the workgroups that rows side by
    side get and with their bits: a batch that ends within a tile, one and seven steps."""
    stride = (1 << 24) + 8
    torch.manual_seed(rows + columns)
    w = torch.randn(rows, columns, device=device).bfloat16()
    x = torch.randn(batch, columns, device=device).bfloat16()
    weights = torch.empty(qh.call("qllm_linear_packed_bytes", rows, columns), dtype=torch.uint8,
                          device=device)
    qh.call("qllm_linear_pack", qh.ptr(w), rows, columns, qh.ptr(weights), columns, 0, 1, 0, None)
    d_x = torch.empty((batch, stride), dtype=torch.bfloat16, device=device)
    d_x[:, :columns] = x
    outs = []
    for source, gap in ((x, columns), (d_x, stride)):
        out = torch.zeros((batch, padded(rows, 4)), device=device)
        segment = qh.LinearSegment(qh.ptr(weights), qh.ptr(source), qh.ptr(out),
                                   padded(rows, 16), columns, gap, padded(rows, 4), rows,
                                   qh.LINEAR_STORE, 0, 0)
        found = qh.LaunchLayout()
        qh.call("qllm_linear_layout", ctypes.byref(segment), 1, batch, BF16,
                ctypes.byref(found))
        assert (found.batch_rows, found.weight_rows) == form
        qh.call("qllm_linear_batch", ctypes.byref(segment), 1, batch, BF16, None)
        torch.cuda.synchronize()
        outs.append(out[:, :rows])
    assert torch.equal(*outs)
    bound = columns * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert ((outs[0].double() - x.double() @ w.double().T).abs() <= bound).all()


# ---- stream ---------------------------------------------------------------------


@pytest.mark.parametrize("element", [F32, BF16])
@pytest.mark.parametrize("width", [64, 90, 132])
def test_embedding_norms_partials_and_gather(device, element, width):
    rng = np.random.default_rng(width)
    table = mm.bf16(rng.standard_normal((30, width)))
    tokens = np.array([3, 29, 0, 3, 17], dtype=np.int32)
    x = torch.zeros((5, width), device=device)
    d_table, d_tokens = on(device, table, torch.bfloat16), on(device, tokens, torch.int32)
    qh.call("qllm_embedding_bf16_batch", qh.ptr(d_table), 30, qh.ptr(d_tokens), qh.ptr(x), 5,
            width, 0.75, None)
    torch.cuda.synchronize()
    assert np.array_equal(x.cpu().numpy(), table[tokens] * np.float32(0.75))

    stride = padded(width, 64)
    partials = rng.standard_normal((9, 5, padded(width, 4))).astype(np.float32)
    weights = rng.standard_normal((2, width)).astype(np.float32)
    d_weights = [on(device, w) for w in weights]
    outs = [torch.full((5, stride), 9.0, dtype=torch_type(element), device=device)
            for _ in range(2)]
    summed = torch.zeros((5, width), device=device)
    d_partials = on(device, partials)
    launch = qh.StreamNormLaunch(
        qh.ptr(x), qh.ptr(summed), qh.ptr(d_partials), 9, padded(width, 4),
        (ctypes.c_void_p * 2)(*map(qh.ptr, d_weights)),
        (ctypes.c_void_p * 2)(*map(qh.ptr, outs)), (ctypes.c_uint32 * 2)(stride, stride),
        5, width, 1e-5, element, None, None, None)
    qh.call("qllm_stream_norm", ctypes.byref(launch), None)
    torch.cuda.synchronize()
    stream = table[tokens].astype(np.float64) * 0.75 + partials[:, :, :width].sum(0)
    close(summed, stream, F32)
    for out, w in zip(outs, weights):
        close(out[:, :width], mo.rms(stream, 1e-5) * w, element)
        assert torch.all(out[:, width:] == 0)

    rows = torch.tensor([4, 0, 4], dtype=torch.int32, device=device)
    picked = torch.zeros((3, stride), dtype=torch_type(element), device=device)
    launch = qh.StreamNormLaunch(
        qh.ptr(summed), None, None, 0, 0, (ctypes.c_void_p * 2)(qh.ptr(d_weights[0]), None),
        (ctypes.c_void_p * 2)(qh.ptr(picked), None), (ctypes.c_uint32 * 2)(stride, 0),
        3, width, 1e-5, element, None, qh.ptr(rows), None)
    qh.call("qllm_stream_norm", ctypes.byref(launch), None)
    torch.cuda.synchronize()
    close(picked[:, :width], (mo.rms(stream, 1e-5) * weights[0])[[4, 0, 4]], element)


@pytest.mark.parametrize("element", [F32, BF16])
@pytest.mark.parametrize("width", [64, 90])
def test_token_shift_carries_the_last_norm(device, element, width):
    rng = np.random.default_rng(width)
    x = rng.standard_normal((7, width)).astype(np.float32)
    weight, *mus = rng.uniform(0.1, 1.0, (4, width)).astype(np.float32)
    stride = padded(width, 64)
    slot_stride = padded(width, 4) + 8
    carried = torch.zeros(2 * slot_stride, device=device)
    last = torch.zeros(padded(width, 4), device=device)
    d_weight, d_mus = on(device, weight), [on(device, mu) for mu in mus]
    normed = mo.rms(x.astype(np.float64), 1e-5) * weight
    before = np.zeros(width)
    for first, count in ((0, 1), (1, 2), (3, 4)):
        d_x = on(device, x[first:first + count])
        outs = [torch.zeros((count, stride), dtype=torch_type(element), device=device)
                for _ in mus]
        shift = qh.TokenShift(3, (ctypes.c_void_p * 6)(*map(qh.ptr, d_mus)),
                              (ctypes.c_void_p * 6)(*map(qh.ptr, outs)), qh.ptr(carried),
                              slot_stride, qh.ptr(last))
        step = steps(device, first, slot=1)
        launch = qh.StreamNormLaunch(
            qh.ptr(d_x), None, None, 0, 0, (ctypes.c_void_p * 2)(qh.ptr(d_weight), None),
            (ctypes.c_void_p * 2)(None, None), (ctypes.c_uint32 * 2)(stride, 0), count, width,
            1e-5, element, ctypes.pointer(shift), None, qh.ptr(step))
        qh.call("qllm_stream_norm", ctypes.byref(launch), None)
        torch.cuda.synchronize()
        part = normed[first:first + count]
        for out, mu in zip(outs, mus):
            close(out[:, :width], mo.shift_mix(part, before, mu), element)
        before = part[-1]
        close(last[:width], before, F32)
        carried[slot_stride:slot_stride + width] = last[:width]


@pytest.mark.parametrize("element", [F32, BF16])
@pytest.mark.parametrize("width,rows", [(64, 1), (90, 3), (2048, 1), (2048, 20), (4096, 17),
                                        (8192, 2), (5120, 4), (512, 512), (512, 513)])
@pytest.mark.parametrize("shifted", [False, True])
def test_first_norm_looks_its_rows_up(device, element, width, rows, shifted):
    """Rows of a thread per piece, of several and of no whole pieces: the same bits as the
    lookup and the norm by themselves, a token outside the table among them."""
    rng = np.random.default_rng(width + rows)
    vocabulary, stride = 50, padded(width, 64)
    table = on(device, mm.bf16(rng.standard_normal((vocabulary, width))), torch.bfloat16)
    ids = rng.integers(0, vocabulary, rows)
    ids[rows // 2] = vocabulary if rows > 1 else ids[0]
    ids = on(device, ids.astype(np.int32), torch.int32)
    weights = [on(device, w) for w in rng.standard_normal((2, width)).astype(np.float32)]
    mus = [on(device, m) for m in rng.uniform(0, 1, (6, width)).astype(np.float32)]
    carried = on(device, rng.standard_normal(padded(width, 4)).astype(np.float32))
    step = steps(device, 0, slot=0)

    def run(together):
        x = torch.full((rows, width), 7.0, device=device)
        outs = [torch.full((rows, stride), 9.0, dtype=torch_type(element), device=device)
                for _ in range(8)]
        last = torch.zeros(padded(width, 4), device=device)
        shift = qh.TokenShift(6, (ctypes.c_void_p * 6)(*map(qh.ptr, mus)),
                              (ctypes.c_void_p * 6)(*map(qh.ptr, outs[2:])), qh.ptr(carried),
                              padded(width, 4), qh.ptr(last))
        launch = qh.StreamNormLaunch(
            None if together else qh.ptr(x), qh.ptr(x) if together else None, None, 0, 0,
            (ctypes.c_void_p * 2)(*map(qh.ptr, weights)),
            (ctypes.c_void_p * 2)(*map(qh.ptr, outs[:2])),
            (ctypes.c_uint32 * 2)(stride, stride), rows, width, 1e-5, element,
            ctypes.pointer(shift) if shifted else None, None, qh.ptr(step))
        if together:
            qh.call("qllm_stream_norm_tokens", ctypes.byref(launch),
                    ctypes.byref(qh.TokenRows(qh.ptr(table), qh.ptr(ids), vocabulary, 0.75)),
                    None)
        else:
            qh.call("qllm_embedding_bf16_batch", qh.ptr(table), vocabulary, qh.ptr(ids),
                    qh.ptr(x), rows, width, 0.75, None)
            qh.call("qllm_stream_norm", ctypes.byref(launch), None)
        return [x, last, *outs]

    for one, two in zip(run(True), run(False)):
        assert torch.equal(one, two)


@pytest.mark.parametrize("columns", [64, 192, 320, 768, 1088, 1472, 1856, 2176, 3904])
@pytest.mark.parametrize("epilogue,splits", [(0, 1), (2, 1), (3, 3)])
def test_linear_parts_of_no_whole_rounds(device, columns, epilogue, splits):
    """Waves with zero to fifteen chunks: few rows have the bits that they have among 17,
    whose chunks are taken one by one, and are the products to bf16's rounding."""
    rng = np.random.default_rng(columns)
    matrix = mm.bf16(rng.standard_normal((96, columns)) / np.sqrt(columns))
    weights = packed(device, [(matrix, 0, 1, 0)], 96, columns)
    x = on(device, rng.standard_normal((17, columns)), torch.bfloat16)
    outputs = 48 if epilogue == 2 else 96

    def run(batch):
        out = torch.full((splits, batch, outputs), 7.0, device=device,
                         dtype=torch.bfloat16 if epilogue == 2 else torch.float32)
        segment = qh.LinearSegment(qh.ptr(weights), qh.ptr(x), qh.ptr(out), 96, columns, columns,
                                   outputs, outputs, epilogue, 0, splits)
        qh.call("qllm_linear_batch", ctypes.byref(segment), 1, batch, BF16, None)
        torch.cuda.synchronize()
        return out

    whole = run(17)
    for batch in (1, 16):
        assert torch.equal(run(batch), whole[:, :batch])
    if epilogue != 2:
        close(whole.sum(0), x.double().cpu().numpy() @ matrix.astype(np.float64).T, F32)


@pytest.mark.parametrize("element", [F32, BF16])
@pytest.mark.parametrize("width", [64, 90, 132, 2048, 2052, 4096, 4100])
@pytest.mark.parametrize("form,partials", [("plain", 0), ("plain", 1), ("plain", 8),
                                           ("plain", 9), ("branch", 3), ("shift", 5),
                                           ("tokens", 0), ("tokens shift", 0)])
def test_projection_takes_its_norm_in(device, element, width, form, partials):
    """One token's norm and its projections in one launch against the two launches, bit for
    bit: rows of one and two pieces a thread, of no whole pieces and of too many (which stay
    two launches), a stored and a gated matrix of more tiles than workgroups, one infinite
    weight.  One launch leaves the normalised rows as they were."""
    rng = np.random.default_rng(width + partials)
    columns, stride = padded(width, 64), padded(width, 64) + 8
    rows = [9040, 9056] if width <= 2052 else [4208, 64]
    torch.manual_seed(width)
    packs = []
    for r in rows:
        source = torch.randn(r, width, device=device).bfloat16()
        source[5, 3] = torch.inf
        packs.append(torch.empty(qh.call("qllm_linear_packed_bytes", r, columns),
                                 dtype=torch.uint8, device=device))
        qh.call("qllm_linear_pack", qh.ptr(source), r, width, qh.ptr(packs[-1]), columns, 0, 1,
                0, None)
        torch.cuda.synchronize()
    table = on(device, mm.bf16(rng.standard_normal((9, width))), torch.bfloat16)
    ids = on(device, np.array([4], dtype=np.int32), torch.int32)
    x = on(device, rng.standard_normal((1, width)).astype(np.float32))
    sums = on(device, rng.standard_normal((max(partials, 1), 1, padded(width, 4)))
              .astype(np.float32))
    norms = [on(device, w) for w in rng.standard_normal((3, width)).astype(np.float32)]
    mus = [on(device, m) for m in rng.uniform(0, 1, (2, width)).astype(np.float32)]
    carried = on(device, rng.standard_normal(padded(width, 4)).astype(np.float32))
    step = steps(device, 0, slot=0)
    shifted, tokens = "shift" in form, "tokens" in form
    one_launch = width % 4 == 0 and width <= 4096 and partials <= 8

    def run(together):
        stream = torch.full((1, width), 7.0, device=device)
        ins = [torch.full((1, stride), 9.0, dtype=torch_type(element), device=device)
               for _ in range(4)]
        last = torch.zeros(padded(width, 4), device=device)
        shift = qh.TokenShift(2, (ctypes.c_void_p * 6)(*map(qh.ptr, mus)),
                              (ctypes.c_void_p * 6)(*map(qh.ptr, ins[2:])), qh.ptr(carried),
                              1 << 40, qh.ptr(last))
        norm = qh.StreamNormLaunch(
            None if tokens else qh.ptr(x), qh.ptr(stream), qh.ptr(sums), partials,
            padded(width, 4), (ctypes.c_void_p * 2)(*map(qh.ptr, norms[:2])),
            (ctypes.c_void_p * 2)(*map(qh.ptr, ins[:2])),
            (ctypes.c_uint32 * 2)(stride, stride), 1, width, 1e-5, element,
            ctypes.pointer(shift) if shifted else None, None, qh.ptr(step),
            qh.ptr(norms[2]) if form == "branch" else None, 0.5, 1e-6)
        out = torch.zeros((1, padded(rows[0], 4)), device=device)
        gated = torch.zeros((1, rows[1] // 2), dtype=torch_type(element), device=device)
        segments = (qh.LinearSegment * 2)(
            qh.LinearSegment(qh.ptr(packs[0]), qh.ptr(ins[3 if shifted else 0]), qh.ptr(out),
                             padded(rows[0], 16), columns, stride, padded(rows[0], 4), rows[0],
                             0, 0, 1),
            qh.LinearSegment(qh.ptr(packs[1]), qh.ptr(ins[1]), qh.ptr(gated), rows[1], columns,
                             stride, rows[1] // 2, rows[1] // 2 - 3, 2, 0, 1))
        row = qh.TokenRows(qh.ptr(table), qh.ptr(ids), 9, 0.75)
        if together:
            arguments = ctypes.byref(norm), ctypes.byref(row) if tokens else None, segments, 2
            launches = ctypes.c_uint32()
            qh.call("qllm_linear_normed_launches", *arguments, ctypes.byref(launches))
            assert launches.value == (1 if one_launch else 2)
            qh.call("qllm_linear_normed", *arguments, None)
        else:
            if tokens:
                qh.call("qllm_stream_norm_tokens", ctypes.byref(norm), ctypes.byref(row), None)
            else:
                qh.call("qllm_stream_norm", ctypes.byref(norm), None)
            qh.call("qllm_linear_batch", segments, 2, 1, element, None)
        torch.cuda.synchronize()
        assert all(bool((rows == 9.0).all()) for rows in ins) == (together and one_launch)
        return stream, last, out, gated

    for one, two in zip(run(True), run(False)):
        assert torch.equal(one.isnan(), two.isnan())
        assert torch.equal(one.nan_to_num(), two.nan_to_num())


@pytest.mark.parametrize("element", [F32, BF16])
@pytest.mark.parametrize("over", ["partials", "input", "branch", "carried", "stream"])
def test_projections_that_write_over_what_the_norm_reads(device, element, over):
    """The results of the two launches also where one launch would still read what its
    workgroups write: sums, stream, branch weights, and a carried row that is the next."""
    rng = np.random.default_rng(3)
    width, rows = 512, 9040
    weights = on(device, rng.standard_normal((rows, width)) / 16, torch.bfloat16)
    pack = torch.empty(qh.call("qllm_linear_packed_bytes", rows, width), dtype=torch.uint8,
                       device=device)
    qh.call("qllm_linear_pack", qh.ptr(weights), rows, width, qh.ptr(pack), width, 0, 1, 0, None)
    norms = [on(device, w) for w in rng.standard_normal((2, width)).astype(np.float32)]
    mu = on(device, rng.uniform(0, 1, width).astype(np.float32))
    step = steps(device, 0, slot=0)
    torch.manual_seed(7)
    values = {name: torch.randn(size, device=device) for name, size in (
        ("input", rows), ("partials", rows), ("branch", rows), ("carried", width),
        ("stream", rows))}

    def run(together):
        held = {name: value.clone() for name, value in values.items()}
        held["out"] = torch.zeros(rows, device=device)
        ins = [torch.zeros(width, dtype=torch_type(element), device=device) for _ in range(2)]
        last = held["carried"] if over == "carried" else torch.zeros(width, device=device)
        shift = qh.TokenShift(1, (ctypes.c_void_p * 6)(qh.ptr(mu)),
                              (ctypes.c_void_p * 6)(qh.ptr(ins[1])), qh.ptr(held["carried"]),
                              width, qh.ptr(last))
        norm = qh.StreamNormLaunch(
            qh.ptr(held["input"]), qh.ptr(held["stream"]), qh.ptr(held["partials"]), 3, width,
            (ctypes.c_void_p * 2)(qh.ptr(norms[0])), (ctypes.c_void_p * 2)(qh.ptr(ins[0])),
            (ctypes.c_uint32 * 2)(width, width), 1, width, 1e-5, element,
            ctypes.pointer(shift) if over == "carried" else None, None, qh.ptr(step),
            qh.ptr(held["branch"]) if over == "branch" else None, 0.5, 1e-6)
        output = held["out" if over == "carried" else over]
        segment = qh.LinearSegment(qh.ptr(pack), qh.ptr(ins[over == "carried"]), qh.ptr(output),
                                   rows, width, width, rows, rows, 0, 0, 1)
        if together:
            launches = ctypes.c_uint32()
            qh.call("qllm_linear_normed_launches", ctypes.byref(norm), None,
                    ctypes.byref(segment), 1, ctypes.byref(launches))
            assert launches.value == 2   # (and nothing is run that would race)
            qh.call("qllm_linear_normed", ctypes.byref(norm), None, ctypes.byref(segment), 1,
                    None)
        else:
            qh.call("qllm_stream_norm", ctypes.byref(norm), None)
            qh.call("qllm_linear_batch", ctypes.byref(segment), 1, 1, element, None)
        torch.cuda.synchronize()
        return [*held.values(), last]

    for one, two in zip(run(True), run(False)):
        assert torch.equal(one, two)


# ---- attention -------------------------------------------------------------------


class Attention:
    """Pages, table and launches of one attention layer; rows are fed in any
    portions, outputs come back in order."""

    def __init__(self, device, element, heads, kv, dim, vdim, window, sinks, mix, scale,
                 rotary=0, base=1000.0, page_tokens=64, context=512, slots=1, strides=None):
        self.device, self.element = device, element
        self.heads, self.kv, self.dim, self.vdim = heads, kv, dim, vdim
        self.stride = (heads + kv) * dim + kv * vdim + heads
        self.stride += -self.stride % 4
        key, value = strides or (padded(dim, 64), padded(vdim, 64))
        key, value = (128 if 64 < s <= 128 else 256 if 128 < s <= 256 else s
                      for s in (key, value))
        self.key, self.mix = key, None if mix is None else on(device, mix)
        pages = context // page_tokens
        layer = qh.call("qllm_windowed_layer_bytes", page_tokens, kv, key, value, element)
        self.offset = 64
        self.pages = [torch.zeros(layer + 64, dtype=torch.uint8, device=device)
                      for _ in range(pages * slots)]
        # pages in no particular order
        order = np.random.default_rng(0).permutation(len(self.pages))
        self.table = torch.tensor([self.pages[i].data_ptr() for i in order],
                                  dtype=torch.int64, device=device)
        self.step = steps(device, 0)
        self.rotary, self.base = rotary, base
        self.frequencies = torch.tensor(
            [base ** (-2.0 * i / rotary) for i in range(rotary // 2)] or [0.0],
            dtype=torch.float64, device=device)
        self.layer = qh.WindowedAttention(
            heads, kv, dim, vdim, key, value, window, sinks, scale, qh.ptr(self.mix),
            page_tokens, pages, self.offset, qh.ptr(self.table), qh.ptr(self.step), element)

    def run(self, projections, position, slot=0, first=None, share=None, token=False):
        """`token`: a single row's launches as one call."""
        rows = projections.shape[0]
        d = on(self.device, projections)
        self.step.copy_(torch.tensor([position, slot, rows, 0], dtype=torch.int32))
        query = torch.zeros((rows, self.heads, self.key), dtype=torch_type(self.element),
                            device=self.device)
        kept = torch.zeros((rows, self.kv * self.vdim), device=self.device)
        at = self.heads * self.dim, (self.heads + self.kv) * self.dim
        gate = at[1] + self.kv * self.vdim
        d_first = None if first is None else on(self.device, first)
        d_share = None if share is None else torch.tensor([share], device=self.device)
        store = qh.RopeStoreLaunch(
            qh.ptr(d), self.stride, 0, at[0], at[1], self.rotary, qh.ptr(self.frequencies),
            qh.ptr(d_first), qh.ptr(d_share), qh.ptr(kept), qh.ptr(query), rows)
        if not token:
            qh.call("qllm_windowed_rope_store", ctypes.byref(self.layer), ctypes.byref(store),
                    None)
        size = qh.call("qllm_windowed_attention_workspace_bytes", ctypes.byref(self.layer),
                       rows, position + rows - 1)
        workspace = torch.zeros(max(size, 16), dtype=torch.uint8, device=self.device)
        out = torch.zeros((rows, self.heads * self.vdim), dtype=torch_type(self.element),
                          device=self.device)
        launch = qh.AttentionLaunch(
            qh.ptr(query), d.data_ptr() + 4 * gate, self.stride, qh.ptr(out),
            self.heads * self.vdim, rows, position + rows - 1, qh.ptr(workspace), size)
        if token:
            qh.call("qllm_windowed_attention_token", ctypes.byref(self.layer),
                    ctypes.byref(store), ctypes.byref(launch), None)
        else:
            qh.call("qllm_windowed_attention_rows", ctypes.byref(self.layer),
                    ctypes.byref(launch), None)
        torch.cuda.synchronize()
        assert np.array_equal(
            kept.cpu().numpy(),
            projections[:, at[1]:at[1] + self.kv * self.vdim])
        return out.float().cpu().numpy().astype(np.float64)

    def expected(self, projections, window, sinks, mix, scale, first=None, share=None):
        p = projections.astype(np.float64)
        rows = p.shape[0]
        at = self.heads * self.dim, (self.heads + self.kv) * self.dim
        where = np.arange(rows, dtype=np.float64)
        q = mo.rotate_interleaved(p[:, :at[0]].reshape(rows, self.heads, self.dim), where,
                                  self.rotary, self.base)
        k = mo.rotate_interleaved(p[:, at[0]:at[1]].reshape(rows, self.kv, self.dim), where,
                                  self.rotary, self.base)
        v = p[:, at[1]:at[1] + self.kv * self.vdim]
        if first is not None:
            v = (1.0 - share) * v + share * first
        v = v.reshape(rows, self.kv, self.vdim)
        gate = p[:, at[1] + self.kv * self.vdim:][:, :self.heads]
        out = mo.attention_core(q, k, v, where, where, scale, window or rows, sinks,
                                np.eye(self.heads) if mix is None else mix)
        return (out * mo.sigmoid(gate)[:, :, None]).reshape(rows, -1)


@pytest.mark.parametrize("element,heads,kv,dim,vdim,rotary,window,sinks", [
    (BF16, 16, 4, 128, 128, 128, 0, 0), (BF16, 8, 1, 64, 40, 16, 40, 3),
    (BF16, 6, 2, 200, 256, 64, 33, 40), (BF16, 4, 4, 24, 16, 0, 0, 0),
    (BF16, 4, 2, 36, 32, 36, 0, 0),      # dimensions not in eights: the two launches
    (F32, 4, 2, 40, 24, 40, 0, 3)])      # the general form likewise
def test_a_token_in_one_call(device, element, heads, kv, dim, vdim, rotary, window, sinks):
    """The token's rotation and store inside the launch of its scores: outputs and
    pages are the two launches', at the places of a token in a key fragment, a tile
    and a page, and at pages that held something else before."""
    rng = np.random.default_rng(dim)
    mix = mm.bf16(np.eye(heads) + 0.2 * rng.standard_normal((heads, heads)))
    total = 131
    one, two = (Attention(device, element, heads, kv, dim, vdim, window, sinks, mix,
                          dim ** -0.5, rotary) for _ in range(2))
    projections = mm.bf16(rng.standard_normal((total, one.stride)))
    first = mm.bf16(rng.standard_normal((total, kv * vdim)))
    for page in one.pages + two.pages:
        page.fill_(0x3f)                 # 0.75 in either type
    at = 0
    for position in (0, 1, 15, 16, 31, 32, 63, 64, 100, 127, 128, 130):
        for layer in (one, two):
            if position > at:
                layer.run(projections[at:position], at)
        share = 0.25 if position % 2 else None
        row = slice(position, position + 1)
        blend = dict(first=None if share is None else first[row], share=share)
        got = one.run(projections[row], position, token=True, **blend)
        want = two.run(projections[row], position, **blend)
        assert np.array_equal(got, want), position
        assert np.all(np.isfinite(want))
        at = position + 1
    for left, right in zip(one.pages, two.pages):
        assert torch.equal(left, right)


@pytest.mark.parametrize("element,heads,kv,dim,vdim,window", [
    (F32, 16, 4, 128, 128, 0), (F32, 5, 1, 40, 24, 700), (F32, 40, 2, 32, 32, 100),
    (BF16, 40, 2, 32, 32, 0)])
def test_general_splits_equal_a_workgroup_per_row(device, element, heads, kv, dim, vdim,
                                                  window):
    """One to four rows over a long context, dealt over workgroups, against the same
    rows as the end of a batch that takes a workgroup for each."""
    rng = np.random.default_rng(heads)
    total, scale = 1300, 1.0 / np.sqrt(dim)
    mix = mm.bf16(np.eye(heads) + 0.2 * rng.standard_normal((heads, heads)))
    layer = Attention(device, element, heads, kv, dim, vdim, window, 3, mix, scale,
                      context=1344)
    projections = mm.bf16(rng.standard_normal((total, layer.stride)))
    whole = layer.run(projections, 0)
    for rows in (1, 2, 3, 4):
        again = layer.run(projections[total - rows:], total - rows)
        close(again, whole[total - rows:], element)


@pytest.mark.parametrize("element,heads,kv,dim,vdim", [
    (F32, 5, 1, 16, 64), (F32, 16, 4, 128, 128), (F32, 4, 2, 128, 144), (BF16, 40, 2, 24, 32)])
@pytest.mark.parametrize("keys", [4, 31, 32, 33, 64, 65])
def test_general_rows_over_a_tile_or_two(device, element, heads, kv, dim, vdim, keys):
    """A few rows at the edges between one launch and three: one visible tile, and
    dimensions of 256 together."""
    rng = np.random.default_rng(keys + heads)
    scale = 1.0 / np.sqrt(dim)
    mix = mm.bf16(np.eye(heads) + 0.2 * rng.standard_normal((heads, heads)))
    layer = Attention(device, element, heads, kv, dim, vdim, 0, 0, mix, scale, context=128,
                      strides=(padded(dim, 32), padded(vdim, 16)))
    projections = mm.bf16(rng.standard_normal((keys, layer.stride)))
    want = layer.expected(projections, 0, 0, mix.astype(np.float64), scale)
    if keys > 4:
        layer.run(projections[:keys - 4], 0)
    close(layer.run(projections[keys - 4:], keys - 4), want[keys - 4:], element)
    close(layer.run(projections[keys - 1:], keys - 1), want[keys - 1:], element)


@pytest.mark.parametrize("element,heads,kv,dim,vdim,window", [
    (F32, 5, 1, 40, 24, 0), (F32, 33, 3, 16, 16, 2400), (BF16, 34, 2, 32, 32, 0)])
def test_general_splits_with_several_tiles_a_workgroup(device, element, heads, kv, dim, vdim,
                                                       window):
    """More tiles than score splits: a head's running maximum and sum pass from one
    tile's lanes to the next one's.  Odd head counts leave half waves without a head."""
    rng = np.random.default_rng(heads)
    total, scale = 4200, 2.0 / np.sqrt(dim)      # 132 tiles in 64 splits
    layer = Attention(device, element, heads, kv, dim, vdim, window, 3, None, scale,
                      context=4224)
    projections = mm.bf16(rng.standard_normal((total, layer.stride)))
    # maxima that grow from tile to tile, and one that comes first
    keys = slice(heads * dim, (heads + kv) * dim)
    projections[:, keys] *= np.linspace(0.25, 1.5, total)[:, None]
    projections[64, keys] *= 4.0
    projections = mm.bf16(projections)
    whole = layer.run(projections, 0)
    for rows in (1, 4):
        again = layer.run(projections[total - rows:], total - rows)
        close(again, whole[total - rows:], element)


@pytest.mark.parametrize("element", [F32, BF16])
@pytest.mark.parametrize("heads,kv,dim,vdim,window,sinks,mixed,rows", [
    (16, 4, 112, 144, 100, 5, True, 530),     # three rows a workgroup
    (6, 2, 72, 20, 0, 0, True, 259),          # a short last workgroup, a rest of dimensions
    (6, 2, 72, 20, 50, 33, False, 259),       # a workgroup per operand
    (20, 1, 320, 30, 64, 0, True, 40),        # two operands of one key/value head
    (40, 2, 24, 320, 0, 0, False, 40),
    (5, 5, 16, 16, 20, 1, True, 700),         # one head an operand
    (72, 72, 4, 496, 30, 0, True, 34),        # LDS holds one tile and no padding
], ids=str)
def test_general_prompts_match_the_oracle(device, element, heads, kv, dim, vdim, window, sinks,
                                          mixed, rows):
    """Rows of the general form: several to a workgroup, operands of more than 16
    heads, remainders of dimensions and workgroups."""
    rng = np.random.default_rng(rows)
    scale = 1.0 / np.sqrt(dim)
    mix = mm.bf16(np.eye(heads) + 0.2 * rng.standard_normal((heads, heads)))
    layer = Attention(device, element, heads, kv, dim, vdim, window, sinks,
                      mix if mixed else None, scale, context=704,
                      strides=(padded(dim, 32), padded(vdim, 16)))
    assert qh.call("qllm_windowed_attention_form", ctypes.byref(layer.layer),
                   rows) == qh.ATTENTION_GENERAL
    projections = mm.bf16(rng.standard_normal((rows, layer.stride)))
    want = layer.expected(projections, window, sinks,
                          (mix if mixed else np.eye(heads)).astype(np.float64), scale)
    close(layer.run(projections, 0), want, element)


@pytest.mark.parametrize("heads,kv,dim,vdim", [(16, 4, 128, 128), (6, 3, 64, 56),
                                               (4, 1, 250, 230), (12, 2, 64, 64)])
@pytest.mark.parametrize("keys", [256, 257, 511, 512, 513])   # tiles of eight waves, and past them
def test_split_rows_at_the_edges_of_their_forms(device, heads, kv, dim, vdim, keys):
    rng = np.random.default_rng(keys + heads)
    scale = 1.0 / np.sqrt(dim)
    mix = mm.bf16(np.eye(heads) + 0.2 * rng.standard_normal((heads, heads)))
    layer = Attention(device, BF16, heads, kv, dim, vdim, 0, 0, mix, scale, context=576)
    projections = mm.bf16(rng.standard_normal((keys, layer.stride)))
    want = layer.expected(projections, 0, 0, mix.astype(np.float64), scale)
    layer.run(projections[:keys - 5], 0)
    close(layer.run(projections[keys - 5:keys - 1], keys - 5), want[keys - 5:keys - 1], BF16)
    close(layer.run(projections[keys - 1:], keys - 1), want[keys - 1:], BF16)


def stand_out(rng, layer, projections, pairs, head, strength=None):
    """Makes the score of (query row, key row) of one head stand out: the key
    becomes the query direction (unrotated dimensions or rotary 0 assumed)."""
    dim, group = layer.dim, layer.heads // layer.kv
    key_at = layer.heads * dim + head // group * dim
    for query, key in pairs:
        direction = mm.bf16(rng.standard_normal(dim))
        direction *= np.float32((strength or 5.0) / np.linalg.norm(direction) * dim ** 0.25)
        projections[query, head * dim:(head + 1) * dim] = direction
        projections[key, key_at:key_at + dim] = direction


SHAPES = [
    # heads, kv, dim, vdim, window, sinks, rotary, page tokens
    (6, 2, 56, 44, 40, 5, 56, 64),
    (3, 1, 24, 40, 33, 0, 16, 32),
    (12, 4, 48, 64, 64, 1, 48, 64),
    (16, 4, 128, 128, 70, 37, 64, 64),
    (20, 4, 80, 24, 31, 33, 32, 96),
    (32, 8, 64, 64, 90, 4, 64, 64),
    (24, 8, 128, 96, 1, 2, 0, 32),
    (8, 8, 32, 32, 0, 0, 32, 64),
    (9, 3, 16, 128, 50, 64, 16, 64),
    (6, 6, 160, 72, 48, 3, 20, 64),
    (36, 12, 40, 40, 45, 8, 40, 64),
    (40, 2, 32, 32, 45, 7, 20, 64),
    (64, 8, 128, 120, 35, 3, 64, 64),
]


@pytest.mark.parametrize("element", [F32, BF16])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_windowed_attention_in_portions(device, element, shape):
    heads, kv, dim, vdim, window, sinks, rotary, page_tokens = shape
    rng = np.random.default_rng(heads * dim + window)
    total, scale = 230, 1.3 / np.sqrt(dim)
    mix = mm.bf16(np.eye(heads) + 0.4 * rng.standard_normal((heads, heads)))
    layer = Attention(device, element, heads, kv, dim, vdim, window, sinks, mix, scale, rotary,
                      page_tokens=page_tokens, context=page_tokens * (1 + 256 // page_tokens))
    projections = mm.bf16(rng.standard_normal((total, layer.stride)))
    first = rng.standard_normal((total, kv * vdim)).astype(np.float32)
    want = layer.expected(projections, window, sinks, mix.astype(np.float64), scale, first, 0.3)
    at = 0
    got = []
    for count in (1, 2, 31, 3, 64, 4, 5, 1, 80, 17, 1, 1, 20):
        got.append(layer.run(projections[at:at + count], at, first=first[at:at + count],
                             share=0.3))
        at += count
    assert at == total
    close(np.concatenate(got), want, element, str(shape))


@pytest.mark.parametrize("element", [F32, BF16])
@pytest.mark.parametrize("rows", [1, 3, 16])
@pytest.mark.parametrize("heads,kv,dim", [(4, 2, 64), (20, 4, 64)])
def test_edges_of_window_pages_and_kept_tokens(device, element, rows, heads, kv, dim):
    """One score stands out per case: a key just inside or outside the window,
    among or after the kept first tokens, at a page's border, at the query
    itself.  A mask off by one changes the output by its whole magnitude."""
    window, sinks, total = 48, 5, 192
    scale = dim ** -0.5
    rng = np.random.default_rng(rows)
    mix = mm.bf16(np.eye(heads) + 0.5 * rng.standard_normal((heads, heads)))
    query = total - 1
    keys = [query, query - 1, query - window + 1, query - window, query - window - 1,
            0, sinks - 1, sinks, sinks + 1, 127, 128, 63, 64, 159, 160]
    for head in (0, heads - 1):
        base = mm.bf16(0.5 * rng.standard_normal((total, 4 * heads * dim)))
        for key in keys:
            layer = Attention(device, element, heads, kv, dim, 32, window, sinks, mix, scale)
            projections = base[:, :layer.stride].copy()
            stand_out(rng, layer, projections, [(query, key)], head)
            want = layer.expected(projections, window, sinks, mix.astype(np.float64), scale)
            for wrong in ((window + 1, sinks), (window - 1, sinks), (window, sinks + 1),
                          (window, sinks - 1)):
                # the case would show such a mask: at the keys it is about the
                # planted score appears or goes
                if key in (query - window + 1, query - window, sinks - 1, sinks):
                    other = layer.expected(projections, *wrong, mix.astype(np.float64), scale)
                    shows = {(window + 1, sinks): query - window,
                             (window - 1, sinks): query - window + 1,
                             (window, sinks + 1): sinks,
                             (window, sinks - 1): sinks - 1}[wrong] == key
                    change = np.abs(other[-1] - want[-1]).max() / np.abs(want[-1]).max()
                    assert not shows or change > 0.2
            cut = total - rows
            layer.run(projections[:cut], 0)
            got = layer.run(projections[cut:], cut)
            close(got, want[cut:], element, f"head {head} key {key}")


def test_pages_and_slots_used_again(device):
    rng = np.random.default_rng(5)
    layer = Attention(device, BF16, 4, 2, 64, 64, 32, 2, None, 0.125, context=128, slots=2)
    long = mm.bf16(3.0 * rng.standard_normal((120, layer.stride)))
    short = mm.bf16(rng.standard_normal((40, layer.stride)))
    layer.run(long, 0, slot=1)
    for slot in (1, 0):
        want = layer.expected(short, 32, 2, None, 0.125)
        got = np.concatenate([layer.run(short[:33], 0, slot=slot),
                              layer.run(short[33:34], 33, slot=slot),
                              layer.run(short[34:], 34, slot=slot)])
        close(got, want, BF16, f"slot {slot}")


# ---- recurrences ------------------------------------------------------------------


class Recurrence:
    def __init__(self, device, element, kind, heads, dim, rank, rng, slots=2):
        self.device, self.element, self.kind = device, element, kind
        self.heads, self.dim, self.rank = heads, dim, rank
        n = heads * dim
        self.up = mm.bf16(rng.standard_normal((n, rank)) / np.sqrt(rank))
        self.base = mm.bf16(rng.standard_normal(n) - 1.0)
        self.bias, self.bonus, self.norm = mm.bf16(rng.standard_normal((3, n)))
        self.columns = [i * (n + 3) for i in range(5)]     # r k v gate rate, then low
        self.low = 5 * (n + 3)
        self.stride = self.low + rank + (-(self.low + rank)) % 4
        self.keep = [on(device, self.up, torch.bfloat16)] + [
            on(device, v) for v in (self.base, self.bias, self.bonus, self.norm)]
        self.slot_stride = n * dim + 12
        self.state = torch.zeros(slots * self.slot_stride, device=device)
        self.step = steps(device, 0)
        up, base, bias, bonus, norm = map(qh.ptr, self.keep)
        self.layer = qh.Recurrence(kind, heads, dim, rank, kind, 1e-5, 1e-6,
                                   -np.exp(-0.5), up, base, bias, bonus, norm,
                                   qh.ptr(self.state), self.slot_stride, qh.ptr(self.step),
                                   element)

    def run(self, projections, slot=1):
        rows = projections.shape[0]
        d = on(self.device, projections)
        self.step.copy_(torch.tensor([0, slot, rows, 0], dtype=torch.int32))
        size = qh.call("qllm_recurrence_workspace_bytes", ctypes.byref(self.layer), rows)
        workspace = torch.zeros(max(size, 16), dtype=torch.uint8, device=self.device)
        out = torch.zeros((rows, self.heads * self.dim), dtype=torch_type(self.element),
                          device=self.device)
        r, k, v, gate, rate = self.columns
        launch = qh.RecurrenceLaunch(qh.ptr(d), self.stride, r, k, v, gate, rate, self.low,
                                     qh.ptr(out), self.heads * self.dim, rows, None, None, 0,
                                     qh.ptr(workspace), size)
        qh.call("qllm_recurrence_rows", ctypes.byref(self.layer), ctypes.byref(launch), None)
        torch.cuda.synchronize()
        return out.float().cpu().numpy().astype(np.float64)

    def expected(self, projections):
        p = projections.astype(np.float64)
        rows, n = p.shape[0], self.heads * self.dim
        shape = (rows, self.heads, self.dim)
        r, k, v, gate, rate = (p[:, c:c + n] for c in self.columns)
        inner = np.tanh(p[:, self.low:self.low + self.rank]) @ self.up.T.astype(
            np.float64) + self.base
        zero = np.zeros((self.dim, self.dim))
        out = np.empty(shape)
        if self.kind == qh.RECURRENCE_DELTA:
            w = np.exp(-np.exp(-0.5) * mo.sigmoid(inner)).reshape(shape)
            a = mo.sigmoid(rate + self.bias).reshape(shape)
        else:
            w = np.exp(-np.exp(inner)).reshape(shape)
        r, k, v = (x.reshape(shape) for x in (r, k, v))
        states = []
        for h in range(self.heads):
            if self.kind == qh.RECURRENCE_DELTA:
                out[:, h], state = mo.delta_recurrence(r[:, h], k[:, h], v[:, h], w[:, h],
                                                       a[:, h], zero)
            else:
                out[:, h], state = mo.wkv_recurrence(
                    r[:, h], k[:, h], v[:, h], w[:, h],
                    self.bonus[h * self.dim:(h + 1) * self.dim].astype(np.float64), zero)
            states.append(state)
        gated = mo.sigmoid(gate) if self.kind == qh.RECURRENCE_DELTA else mo.silu(gate)
        return mo.rms(out, 1e-5).reshape(rows, n) * self.norm * gated, np.stack(states)


@pytest.mark.parametrize("kind", [qh.RECURRENCE_DELTA, qh.RECURRENCE_BONUS])
@pytest.mark.parametrize("dim,rank", [(64, 8), (64, 36), (24, 96), (64, 120), (256, 128),
                                      (64, 136), (1, 256), (16, 64), (32, 64), (48, 16),
                                      (96, 64), (128, 64), (192, 40)])
def test_recurrence_steps_of_any_rank(device, kind, dim, rank):
    """Single tokens at the edges of the low-rank rows that a thread holds (pieces of
    eight, at most sixteen of them) and of the parts that are added side by side."""
    rng = np.random.default_rng(dim + rank)
    layer = Recurrence(device, F32, kind, 2, dim, rank, rng)
    projections = mm.bf16(rng.standard_normal((5, layer.stride)))
    want, _ = layer.expected(projections)
    got = [layer.run(projections[at:at + 1]) for at in range(5)]
    close(np.concatenate(got), want, F32, "outputs", factor=2.0)


@pytest.mark.parametrize("element", [F32, BF16])
@pytest.mark.parametrize("kind", [qh.RECURRENCE_DELTA, qh.RECURRENCE_BONUS])
@pytest.mark.parametrize("heads,dim,rank", [(3, 64, 16), (2, 24, 8), (1, 128, 40), (5, 16, 1),
                                            (2, 80, 64), (1, 144, 33), (7, 5, 3)])
def test_recurrences_in_portions(device, element, kind, heads, dim, rank):
    rng = np.random.default_rng(heads * dim + kind)
    layer = Recurrence(device, element, kind, heads, dim, rank, rng)
    projections = mm.bf16(rng.standard_normal((150, layer.stride)))
    projections[:, layer.columns[1]:layer.columns[2]] *= np.float32(2 / np.sqrt(dim))
    want, states = layer.expected(projections)
    at, got = 0, []
    for count in (1, 1, 2, 37, 3, 16, 64, 1, 7, 17, 1):
        got.append(layer.run(projections[at:at + count]))
        at += count
    assert at == 150
    close(np.concatenate(got), want, element, "outputs", factor=2.0)
    n = heads * dim * dim
    state = layer.state[layer.slot_stride:layer.slot_stride + n].cpu().numpy()
    close(state.reshape(heads, dim, dim).astype(np.float64), states, F32, "state", factor=4.0)
    # the other slot was not touched
    assert torch.all(layer.state[:layer.slot_stride] == 0)
    # the same prompt in one piece, in a slot that holds another request's state
    layer.state[layer.slot_stride:] = 0
    close(layer.run(projections), want, element, "whole", factor=2.0)


@pytest.mark.parametrize("element", [F32, BF16])
@pytest.mark.parametrize("kind", [qh.RECURRENCE_DELTA, qh.RECURRENCE_BONUS])
@pytest.mark.parametrize("heads,dim", [(2, 64), (1, 24), (1, 130)])
def test_recurrences_over_long_prompts(device, element, kind, heads, dim):
    rng = np.random.default_rng(dim + kind)
    layer = Recurrence(device, element, kind, heads, dim, 6, rng)
    projections = mm.bf16(rng.standard_normal((1300, layer.stride)))
    projections[:, layer.columns[1]:layer.columns[2]] *= np.float32(2 / np.sqrt(dim))
    want, states = layer.expected(projections)
    n = heads * dim * dim
    for counts in ([1300], [600, 1, 699], [100, 530, 515, 155]):
        layer.state.zero_()
        got, at = [], 0
        for count in counts:
            got.append(layer.run(projections[at:at + count]))
            at += count
        close(np.concatenate(got), want, element, str(counts), factor=2.0)
        state = layer.state[layer.slot_stride:layer.slot_stride + n].cpu().numpy()
        close(state.reshape(heads, dim, dim).astype(np.float64), states, F32, "state",
              factor=4.0)
        assert torch.all(layer.state[:layer.slot_stride] == 0)


def test_launches_turn_down_what_does_not_fit(device):
    layer = Attention(device, BF16, 4, 2, 64, 64, 32, 2, None, 0.125, context=128)
    bad = qh.RopeStoreLaunch(layer.table.data_ptr(), 8, 0, 0, 0, 0, None, None, None, None,
                             layer.table.data_ptr(), 1)
    with pytest.raises(qh.QllmError):
        qh.call("qllm_windowed_rope_store", ctypes.byref(layer.layer), ctypes.byref(bad), None)
    launch = qh.AttentionLaunch(layer.table.data_ptr(), None, 0, layer.table.data_ptr(), 256, 1,
                                100, None, 0)
    with pytest.raises(qh.QllmError, match="workspace"):
        qh.call("qllm_windowed_attention_rows", ctypes.byref(layer.layer),
                ctypes.byref(launch), None)
    segment = qh.LinearSegment(layer.table.data_ptr(), layer.table.data_ptr(),
                               layer.table.data_ptr(), 15, 64, 64, 16, 15, 0, 0, 0)
    with pytest.raises(qh.QllmError, match="segment"):
        qh.call("qllm_linear_batch", ctypes.byref(segment), 1, 1, BF16, None)
