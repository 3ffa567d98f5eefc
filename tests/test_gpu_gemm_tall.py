"""The FP4 GEMM for tall batches (prompt prefill) against the CPU oracle, and
against the small-batch kernel on the same rows."""
import ctypes

import numpy as np
import pytest
import torch

import gpu_util as gu
import oracle_lib as ol
import qllm_hip as qh
import synth

pytestmark = pytest.mark.gpu


def tall(device, codes, scales, scheme, rows, padded, act, out_kind=qh.OUT_F32,
         residual=None):
    batch = act.shape[0]
    d_codes, d_scales = gu.device_tensor(codes, device), gu.device_tensor(scales, device)
    d_act = gu.device_tensor(ol.bf16_bits(act), device)
    matrix, keep = qh.prepack(qh.fp4_matrix(d_codes, d_scales, rows, padded, padded, scheme),
                              device)
    dtype = torch.bfloat16 if out_kind == qh.OUT_BF16 else torch.float32
    out = torch.zeros((batch, rows), dtype=dtype, device=device)
    d_residual = None if residual is None else gu.device_tensor(residual, device)
    qh.call("qllm_fp4_gemm_bf16_tall", matrix, qh.ptr(d_act), d_act.numel() * 2,
            qh.ptr(out), out_kind, qh.ptr(d_residual), batch, None)
    torch.cuda.synchronize()
    return out.float().cpu().numpy()


@pytest.mark.parametrize("rows,padded,batch", [
    (256, 64, 128), (300, 1024, 9), (1024, 5120, 200), (77, 128, 333),
    (2048, 1024, 1024), (512, 8192, 130)])
@pytest.mark.parametrize("scheme", [ol.SCALE_UE8M0_BLOCK32, ol.SCALE_F16_BLOCK16])
def test_tall_gemm_matches_oracle(device, scheme, rows, padded, batch):
    """Ragged shapes, in workgroups of 16, 48 and 64 batch rows: batches and weight
    rows that are no multiple of theirs or of 32, a single chunk of K.  (Larger
    batches: test_every_layout_matches_the_product.)"""
    rng = np.random.default_rng(rows + batch)
    codes, scales = synth.fp4_matrix(rng, rows, padded, scheme)
    act = ol.bf16_round(rng.standard_normal((batch, padded)).astype(np.float32))
    want = ol.fp4_linear_f64(codes, scales, scheme, rows, padded, act)
    got = tall(device, codes, scales, scheme, rows, padded, act)
    gu.assert_close(got, want, what="tall GEMM")
    if scheme == ol.SCALE_UE8M0_BLOCK32:
        # exact bf16 operands: only the F32 summation order separates the two
        error = np.abs(got - want).max() / np.abs(want).max()
        assert error < 2e-6 * np.sqrt(padded)


@pytest.mark.parametrize("batch", [16, 31, 45, 64, 125])
@pytest.mark.parametrize("scheme", [ol.SCALE_UE8M0_BLOCK32, ol.SCALE_F16_BLOCK16])
def test_tall_gemm_steps_ahead(device, scheme, batch):
    """One to eighteen chunks of K: fewer and more than a workgroup asks for ahead, ends
    at every place of a round of its tiles and of a step of several chunks."""
    rng = np.random.default_rng(batch)
    for chunks in (1, 2, 3, 4, 5, 6, 7, 9, 13, 15, 16, 17, 18):
        padded = 64 * chunks
        codes, scales = synth.fp4_matrix(rng, 77, padded, scheme)
        act = ol.bf16_round(rng.standard_normal((batch, padded)).astype(np.float32))
        got = tall(device, codes, scales, scheme, 77, padded, act)
        want = ol.fp4_linear_f64(codes, scales, scheme, 77, padded, act)
        magnitude = ol.fp4_linear_f64(codes & 0x77, scales, scheme, 77, padded, np.abs(act))
        # exact products (binary16 scales: two halves each); an addition rounds by 2^-24
        assert (np.abs(got - want) <= 2 * padded * 2.0 ** -24 * magnitude).all(), chunks


@pytest.mark.parametrize("scheme", [ol.SCALE_UE8M0_BLOCK32, ol.SCALE_F16_BLOCK16])
def test_tall_gemm_of_far_columns(device, scheme):
    """2^24 columns, past a lane's 32-bit offset over 128 rows of activations."""
    rows, padded, batch = 40, 1 << 24, 20
    block = 32 if scheme == ol.SCALE_UE8M0_BLOCK32 else 16
    codes = torch.randint(0, 256, (rows, padded // 2), dtype=torch.uint8, device=device)
    scales = (torch.full((rows, padded // 32), 127, dtype=torch.uint8, device=device)
              if block == 32 else
              torch.full((rows, padded // 16), 1.0, dtype=torch.float16, device=device))
    matrix, keep = qh.prepack(qh.fp4_matrix(codes, scales, rows, padded, padded, scheme),
                              device)
    columns = [0, 63, 64, padded // 2 + 5, padded - 1]
    act = torch.zeros((batch, padded), dtype=torch.bfloat16, device=device)
    x = torch.randn((batch, len(columns)), device=device).bfloat16()
    act[:, columns] = x
    out = torch.zeros((batch, rows), device=device)
    qh.call("qllm_fp4_gemm_bf16_tall", matrix, qh.ptr(act), act.numel() * 2, qh.ptr(out),
            qh.OUT_F32, None, batch, None)
    values = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6, -0., -.5, -1, -1.5, -2, -3, -4, -6],
                          dtype=torch.float64, device=device)
    picked = torch.stack([codes[:, c // 2] >> 4 * (c % 2) & 15 for c in columns], dim=1)
    want = x.double() @ values[picked.long()].T
    bound = len(columns) * 2.0 ** -24 * (x.double().abs() @ values[picked.long()].abs().T)
    assert ((out.double() - want).abs() <= bound).all()


@pytest.mark.parametrize("padded,batch", [((1 << 24) + 192, 1), ((1 << 24) + 192, 50),
                                          ((1 << 24) + 192, 130), (1 << 27, 20)])
@pytest.mark.parametrize("scheme", [ol.SCALE_UE8M0_BLOCK32, ol.SCALE_F16_BLOCK16])
def test_tall_gemm_and_swiglu_past_32_bit_offsets(device, scheme, padded, batch):
    """Workgroups of 16, 64 and 32 rows over matrices whose activation rows, and of
    2^27 columns weight tiles too, lie further apart than a 32-bit offset; one that ends
    within a step of several chunks."""
    rows, columns = 40, [0, 63, 64, padded // 2 + 5, padded - 130, padded - 1]
    block = 32 if scheme == ol.SCALE_UE8M0_BLOCK32 else 16
    values = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6, -0., -.5, -1, -1.5, -2, -3, -4, -6],
                          dtype=torch.float64, device=device)
    act = torch.zeros((batch, padded), dtype=torch.bfloat16, device=device)
    x = torch.randn((batch, len(columns)), device=device).bfloat16()
    act[:, columns] = x
    matrices, sums, bounds = [], [], []
    for _ in range(1 if padded == 1 << 27 else 2):
        codes = torch.randint(0, 256, (rows, padded // 2), dtype=torch.uint8, device=device)
        scales = (torch.full((rows, padded // 32), 127, dtype=torch.uint8, device=device)
                  if block == 32 else
                  torch.full((rows, padded // 16), 1.0, dtype=torch.float16, device=device))
        matrices.append(qh.prepack(qh.fp4_matrix(codes, scales, rows, padded, padded, scheme),
                                   device))
        picked = torch.stack([codes[:, c // 2] >> 4 * (c % 2) & 15 for c in columns], dim=1)
        sums.append(x.double() @ values[picked.long()].T)
        bounds.append(len(columns) * 2.0 ** -24 *
                      (x.double().abs() @ values[picked.long()].abs().T))
        del codes, scales
    out = torch.zeros((batch, rows), device=device)
    qh.call("qllm_fp4_gemm_bf16_tall", matrices[0][0], qh.ptr(act), act.numel() * 2, qh.ptr(out),
            qh.OUT_F32, None, batch, None)
    torch.cuda.synchronize()
    assert ((out.double() - sums[0]).abs() <= bounds[0]).all()
    if len(matrices) == 1:
        return
    gated = torch.zeros((batch, rows), dtype=torch.bfloat16, device=device)
    qh.call("qllm_fp4_swiglu_bf16_tall", matrices[0][0], matrices[1][0], qh.ptr(act),
            act.numel() * 2, qh.ptr(gated), batch, None)
    torch.cuda.synchronize()
    # two roundings to bf16, each by at most 2^-9, and twice that for the exponential
    want = torch.nn.functional.silu(sums[0]) * sums[1]
    assert ((gated.double() - want).abs() <= 2.0 ** -7 * want.abs() + 1e-5).all()


@pytest.mark.parametrize("scheme", [ol.SCALE_UE8M0_BLOCK32, ol.SCALE_F16_BLOCK16])
def test_tall_gemm_residual_and_bf16_output(device, scheme):
    rng = np.random.default_rng(5)
    rows, padded, batch = 640, 1024, 150
    codes, scales = synth.fp4_matrix(rng, rows, padded, scheme)
    act = ol.bf16_round(rng.standard_normal((batch, padded)).astype(np.float32))
    residual = rng.standard_normal((batch, rows)).astype(np.float32)
    want = ol.fp4_linear_f64(codes, scales, scheme, rows, padded, act)
    got = tall(device, codes, scales, scheme, rows, padded, act, residual=residual)
    gu.assert_close(got, want + residual, what="tall GEMM + residual")
    got = tall(device, codes, scales, scheme, rows, padded, act, out_kind=qh.OUT_BF16)
    gu.assert_close(got, want, rtol=1e-2, atol=1e-3, what="tall GEMM bf16")


@pytest.mark.parametrize("scheme", [ol.SCALE_UE8M0_BLOCK32, ol.SCALE_F16_BLOCK16])
def test_tall_gemm_rows_equal_the_small_batch_kernel(device, scheme):
    """The same five rows through the verify-step kernel and through the tall
    one (as rows 123..127 of a batch of 128)."""
    rng = np.random.default_rng(8)
    rows, padded = 1024, 5120
    codes, scales = synth.fp4_matrix(rng, rows, padded, scheme)
    act = ol.bf16_round(rng.standard_normal((128, padded)).astype(np.float32))
    small = gu.gemm(device, codes, scales, scheme, rows, padded, act[123:128])
    big = tall(device, codes, scales, scheme, rows, padded, act)[123:128]
    gu.assert_close(big, small, rtol=2e-3, atol=2e-4, what="tall vs small-batch rows")


def test_tall_gemm_binary16_scales_at_the_ends_of_their_exact_range(device):
    """Block scales of 2^-13 and of 10912 (6 x 10912 = 65472 is the largest
    product binary16 holds): inside that range weight x scale is carried
    exactly by the two binary16 halves, so the tall kernel agrees with the
    oracle as tightly as for ordinary scales.  Scales below the range (6e-5)
    lose the low half's last bits: within 2^-11 of each product."""
    rng = np.random.default_rng(21)
    rows, padded, batch = 256, 1024, 130
    codes, _ = synth.fp4_matrix(rng, rows, padded, ol.SCALE_F16_BLOCK16)
    act = ol.bf16_round(rng.standard_normal((batch, padded)).astype(np.float32))
    for low, high, tolerance in ((2.0 ** -13, 10912.0, 2e-6), (6e-5, 8192.0, 2.0 ** -11)):
        values = np.where(rng.random((rows, padded // 16)) < 0.5, low, high)
        scales = values.astype(np.float16).view(np.uint16)
        want = ol.fp4_linear_f64(codes, scales, ol.SCALE_F16_BLOCK16, rows, padded, act)
        got = tall(device, codes, scales, ol.SCALE_F16_BLOCK16, rows, padded, act)
        assert np.isfinite(got).all()
        # the error bound is relative to the sum of |products|, not to the result
        magnitude = ol.fp4_linear_f64(codes & 0x77, scales, ol.SCALE_F16_BLOCK16, rows, padded,
                                      np.abs(act))
        assert (np.abs(got - want) <= tolerance * np.sqrt(padded) * magnitude + 1e-30).all()
        small = gu.gemm(device, codes, scales, ol.SCALE_F16_BLOCK16, rows, padded, act[:5])
        assert (np.abs(small - want[:5]) <= 2e-6 * np.sqrt(padded) * magnitude[:5] + 1e-30).all()


def test_tall_split_outputs(device):
    rng = np.random.default_rng(9)
    scheme, padded, batch = ol.SCALE_F16_BLOCK16, 1024, 140
    parts = [512, 64, 64]
    rows = sum(parts)
    codes, scales = synth.fp4_matrix(rng, rows, padded, scheme)
    act = ol.bf16_round(rng.standard_normal((batch, padded)).astype(np.float32))
    whole = tall(device, codes, scales, scheme, rows, padded, act)
    d_codes, d_scales = gu.device_tensor(codes, device), gu.device_tensor(scales, device)
    d_act = gu.device_tensor(ol.bf16_bits(act), device)
    matrix, keep = qh.prepack(qh.fp4_matrix(d_codes, d_scales, rows, padded, padded, scheme),
                              device)
    outs = [torch.zeros((batch, part), device=device) for part in parts]
    segments = (qh.GemmSegment * 3)(*[qh.GemmSegment(qh.ptr(o), part, qh.OUT_F32)
                                      for o, part in zip(outs, parts)])
    qh.call("qllm_fp4_gemm_bf16_tall_split", matrix, qh.ptr(d_act), d_act.numel() * 2,
            segments, 3, batch, None)
    torch.cuda.synchronize()
    first = 0
    for out, part in zip(outs, parts):
        assert np.array_equal(out.cpu().numpy(), whole[:, first:first + part])
        first += part
    bad = (qh.GemmSegment * 2)(qh.GemmSegment(qh.ptr(outs[0]), 520, qh.OUT_F32),
                               qh.GemmSegment(qh.ptr(outs[1]), 120, qh.OUT_F32))
    with pytest.raises(qh.QllmError, match="multiples of 32"):
        qh.call("qllm_fp4_gemm_bf16_tall_split", matrix, qh.ptr(d_act), d_act.numel() * 2,
                bad, 2, batch, None)


@pytest.mark.parametrize("rows,padded,batch", [(1024, 1024, 200), (300, 128, 77), (96, 64, 129)])
@pytest.mark.parametrize("scheme", [ol.SCALE_UE8M0_BLOCK32, ol.SCALE_F16_BLOCK16])
def test_tall_swiglu_equals_two_gemms_and_the_product(device, scheme, rows, padded, batch):
    """One launch over the gate and the up matrix against two tall GEMMs and
    the SiLU-product launch with bf16 rounding points: bit-equal, and against
    the oracle's F64 projections within bf16 rounding."""
    rng = np.random.default_rng(rows + padded + batch)
    act = ol.bf16_round(rng.standard_normal((batch, padded)).astype(np.float32))
    d_act = gu.device_tensor(ol.bf16_bits(act), device)
    matrices, keep, f32, f64 = [], [], [], []
    for _ in range(2):
        codes, scales = synth.fp4_matrix(rng, rows, padded, scheme)
        tensors = gu.device_tensor(codes, device), gu.device_tensor(scales, device)
        matrix, packed = qh.prepack(qh.fp4_matrix(*tensors, rows, padded, padded, scheme), device)
        out = torch.zeros((batch, rows), device=device)
        qh.call("qllm_fp4_gemm_bf16_tall", matrix, qh.ptr(d_act), d_act.numel() * 2,
                qh.ptr(out), qh.OUT_F32, None, batch, None)
        matrices.append(matrix); keep.append((tensors, packed)); f32.append(out)
        f64.append(ol.fp4_linear_f64(codes, scales, scheme, rows, padded, act))
    qh.call("qllm_silu_product", qh.ptr(f32[0]), qh.ptr(f32[1]), qh.ptr(f32[0]),
            batch * rows, 1, None)
    fused = torch.zeros((batch, rows), dtype=torch.bfloat16, device=device)
    qh.call("qllm_fp4_swiglu_bf16_tall", matrices[0], matrices[1], qh.ptr(d_act),
            d_act.numel() * 2, qh.ptr(fused), batch, None)
    torch.cuda.synchronize()
    got = fused.float().cpu().numpy()
    assert np.array_equal(got, f32[0].cpu().numpy())
    want = f64[0] / (1.0 + np.exp(np.minimum(-f64[0], 80.0))) * f64[1]
    gu.assert_close(got, want, rtol=2e-2, atol=2e-2 * np.abs(want).max(), what="tall SwiGLU")
    with pytest.raises(qh.QllmError, match="invalid tall FP4 SwiGLU"):
        qh.call("qllm_fp4_swiglu_bf16_tall", matrices[0], None, qh.ptr(d_act),
                d_act.numel() * 2, qh.ptr(fused), batch, None)


def test_tall_gemm_rejects_row_major(device):
    rng = np.random.default_rng(1)
    codes, scales = synth.fp4_matrix(rng, 64, 64, 0)
    d = [gu.device_tensor(x, device) for x in (codes, scales)]
    act = torch.zeros((16, 64), dtype=torch.bfloat16, device=device)
    out = torch.zeros((16, 64), device=device)
    matrix = qh.fp4_matrix(d[0], d[1], 64, 64, 64, 0)
    with pytest.raises(qh.QllmError, match="invalid tall"):
        qh.call("qllm_fp4_gemm_bf16_tall", matrix, qh.ptr(act), act.numel() * 2,
                qh.ptr(out), qh.OUT_F32, None, 16, None)


@pytest.mark.parametrize("rows,padded,batch", [
    (96, 64, 1), (132, 576, 15), (4, 1024, 16), (260, 832, 17), (1056, 192, 33),
    (640, 1088, 64), (388, 1024, 65), (2048, 5120, 48), (1024, 1216, 300),
    (160, 1024, 49), (2048, 2112, 97)])
@pytest.mark.parametrize("scheme", [ol.SCALE_UE8M0_BLOCK32, ol.SCALE_F16_BLOCK16])
def test_launches_cut_along_k_match_the_oracle(device, scheme, rows, padded, batch):
    """Workgroup heights at their edges (1, 16 / 17, 32 / 33, 64 / 65 rows) and
    ragged weight rows through the forms with a workspace; parts that share the
    chunks unevenly or hold one chunk each, every number of them; gate and up.
    Matrices under 2^20 elements take one launch with a workspace too."""
    rng = np.random.default_rng(rows + batch)
    act = ol.bf16_round(rng.standard_normal((batch, padded)).astype(np.float32))
    d_act = gu.device_tensor(ol.bf16_bits(act), device)
    residual = rng.standard_normal((batch, rows)).astype(np.float32)
    d_residual = gu.device_tensor(residual, device)
    matrices, wants, keep = [], [], []
    for _ in range(2):
        codes, scales = synth.fp4_matrix(rng, rows, padded, scheme)
        wants.append(ol.fp4_linear_f64(codes, scales, scheme, rows, padded, act))
        d_codes, d_scales = gu.device_tensor(codes, device), gu.device_tensor(scales, device)
        matrix, kept = qh.prepack(
            qh.fp4_matrix(d_codes, d_scales, rows, padded, padded, scheme), device)
        matrices.append(matrix)
        keep.append((d_codes, d_scales, kept))
    size = qh.call("qllm_fp4_tall_workspace_bytes")
    workspace = torch.empty(size, dtype=torch.uint8, device=device)
    # F32 sums of at most `padded` exact products, in any order
    bound = 2e-6 * np.sqrt(padded) * np.abs(wants[0]).max()

    for space, count in ((workspace, size), (None, 0)):
        out = torch.full((batch, rows), np.nan, device=device)
        qh.call("qllm_fp4_gemm_bf16_tall_cut", matrices[0], qh.ptr(d_act),
                d_act.numel() * 2, qh.ptr(out), qh.OUT_F32, qh.ptr(d_residual), batch,
                qh.ptr(space), count, None)
        assert np.abs(out.cpu().numpy() - residual - wants[0]).max() < bound + 1e-6
    out = torch.full((batch, rows), np.nan, dtype=torch.bfloat16, device=device)
    qh.call("qllm_fp4_swiglu_bf16_tall_cut", matrices[0], matrices[1], qh.ptr(d_act),
            d_act.numel() * 2, qh.ptr(out), batch, qh.ptr(workspace), size, None)
    want = ol.silu_product(wants[0], wants[1], True)
    # two roundings to bf16 (the gate's SiLU, the product), each of which may fall
    # to the neighbouring value, at most 2^-7 of it away
    error = np.abs(out.float().cpu().numpy() - want)
    assert (error <= 2.0 ** -6 * np.abs(want) + 4 * bound * (1 + np.abs(wants[1]))).all()
    if rows % 32 == 0:
        segments = (qh.GemmSegment * 2)()
        parts = [torch.full((batch, n), np.nan, device=device) for n in (32, rows - 32)]
        for segment, part in zip(segments, parts):
            segment.output, segment.rows = qh.ptr(part), part.shape[1]
            segment.output_kind = qh.OUT_F32
        qh.call("qllm_fp4_gemm_bf16_tall_split_cut", matrices[0], qh.ptr(d_act),
                d_act.numel() * 2, ctypes.addressof(segments), 2, batch,
                qh.ptr(workspace), size, None)
        got = torch.cat(parts, dim=1).cpu().numpy()
        assert np.abs(got - wants[0]).max() < bound
    advised = qh.call("qllm_fp4_tall_parts", matrices[0], batch)
    assert (advised > 1) == (rows * padded >= 1 << 20) and advised <= 16
    for count in range(1, min(16, padded // 64) + 1):
        sums = torch.full((count, batch, rows), np.nan, device=device)
        qh.call("qllm_fp4_gemm_bf16_tall_partial", matrices[0], qh.ptr(d_act),
                d_act.numel() * 2, qh.ptr(sums), count, batch, None)
        assert np.abs(sums.sum(0).cpu().numpy() - wants[0]).max() < bound
    for count in (0, 17, padded // 64 + 1):
        with pytest.raises(qh.QllmError, match="invalid partial"):
            qh.call("qllm_fp4_gemm_bf16_tall_partial", matrices[0], qh.ptr(d_act),
                    d_act.numel() * 2, qh.ptr(workspace), count, batch, None)


UE8M0, F16 = ol.SCALE_UE8M0_BLOCK32, ol.SCALE_F16_BLOCK16


# (batch rows of a workgroup, whether K is cut) of a plain and of a gate-and-up launch
@pytest.mark.parametrize("scheme,rows,padded,batch,plain,swiglu", [
    (UE8M0, 2100, 8896, 1000, (128, True), (48, True)),
    (UE8M0, 2112, 8896, 1000, (128, True), (48, True)),
    (F16, 2100, 8896, 1000, (128, True), (128, True)),
    (F16, 1088, 11200, 1500, (128, True), (128, True)),
    (UE8M0, 1088, 11200, 900, (64, True), (128, True)),
    (UE8M0, 5092, 128, 3001, (128, False), (128, False)),
    (F16, 5092, 128, 3001, (128, False), (128, False)),
    (UE8M0, 5120, 64, 3001, (128, False), (128, False)),
    (UE8M0, 3072, 64, 500, (64, False), (64, False)),
    (F16, 3072, 64, 500, (64, False), (64, False)),
    (UE8M0, 3072, 2048, 100, (64, True), (64, True)),
    (F16, 1536, 4096, 100, (64, True), (64, True)),
    (UE8M0, 1100, 2112, 100, (48, True), (48, True)),
    (F16, 1100, 2112, 48, (48, True), (48, True)),
    (F16, 1088, 2112, 33, (48, True), (48, True)),
    (UE8M0, 1100, 2112, 20, (32, True), (32, True)),
    (F16, 1100, 2112, 20, (32, True), (32, True)),
    (F16, 1088, 2112, 16, (16, True), (16, True))])
def test_every_layout_matches_the_product(device, scheme, rows, padded, batch, plain, swiglu):
    """Every height of a workgroup, whole and cut along K, against the product in 64
    bits: weight rows and batches that end inside a workgroup, every output kind,
    a residual that is the output, segments of different kinds, gate and up."""
    rng = np.random.default_rng(rows + batch)
    act = ol.bf16_round(rng.standard_normal((batch, padded)).astype(np.float32))
    d_act = gu.device_tensor(ol.bf16_bits(act), device)
    act64 = torch.from_numpy(act).to(device, torch.float64)
    matrices, wants, keep = [], [], []
    for _ in range(2):
        codes, scales = synth.fp4_matrix(rng, rows, padded, scheme)
        values = torch.from_numpy(synth.dequantize(codes, scales, scheme)).to(device)
        wants.append((act64 @ values.T).cpu().numpy())
        tensors = gu.device_tensor(codes, device), gu.device_tensor(scales, device)
        matrix, kept = qh.prepack(qh.fp4_matrix(*tensors, rows, padded, padded, scheme),
                                  device)
        matrices.append(matrix)
        keep.append((tensors, kept))
    del values
    want = wants[0]
    size = qh.call("qllm_fp4_tall_workspace_bytes")
    workspace = torch.full((size // 4,), float("nan"), device=device)   # parts are written first

    def layout(gate_and_up, parts=0):
        found = qh.LaunchLayout()
        qh.call("qllm_fp4_tall_layout", matrices[0], gate_and_up, batch, size, parts,
                ctypes.byref(found))
        return found.batch_rows, found.parts

    own = layout(0)[1]
    assert [(height, parts > 1) for height, parts in (layout(0), layout(1))] == [plain, swiglu]
    # F32 sums of `padded` exact products, in any order
    bound = 2e-6 * np.sqrt(padded) * np.abs(want).max()

    def run(kind, residual=None, in_place=False):
        out = torch.full((batch, rows), float("nan"), device=device,
                         dtype=torch.bfloat16 if kind == qh.OUT_BF16 else torch.float32)
        if in_place:
            out.copy_(residual)
            residual = out
        qh.call("qllm_fp4_gemm_bf16_tall_cut", matrices[0], qh.ptr(d_act),
                d_act.numel() * 2, qh.ptr(out), kind, qh.ptr(residual), batch,
                qh.ptr(workspace), size, None)
        return out.double().cpu().numpy()

    rest = torch.from_numpy(rng.standard_normal((batch, rows)).astype(np.float32)).to(device)
    rest64 = rest.double().cpu().numpy()
    assert np.abs(run(qh.OUT_F32) - want).max() < bound
    sums = run(qh.OUT_F32, rest)
    assert np.abs(sums - rest64 - want).max() < bound + 1e-6
    assert np.array_equal(run(qh.OUT_F32, rest, in_place=True), sums)
    rounded = run(qh.OUT_F32_BF16_ROUNDED)
    assert np.array_equal(run(qh.OUT_BF16), rounded)
    assert (np.abs(rounded - want) <= 2.0 ** -8 * np.abs(want) + 1.01 * bound).all()
    if rows % 32 == 0:
        widths, kinds = (64, 32, rows - 96), (qh.OUT_F32, qh.OUT_BF16,
                                              qh.OUT_F32_BF16_ROUNDED)
        outs = [torch.full((batch, n), float("nan"), device=device,
                           dtype=torch.bfloat16 if k == qh.OUT_BF16 else torch.float32)
                for n, k in zip(widths, kinds)]
        segments = (qh.GemmSegment * 3)(*[qh.GemmSegment(qh.ptr(o), n, k)
                                          for o, n, k in zip(outs, widths, kinds)])
        qh.call("qllm_fp4_gemm_bf16_tall_split_cut", matrices[0], qh.ptr(d_act),
                d_act.numel() * 2, ctypes.addressof(segments), 3, batch,
                qh.ptr(workspace), size, None)
        got = np.concatenate([o.double().cpu().numpy() for o in outs], axis=1)
        assert np.array_equal(got[:, 64:], rounded[:, 64:])
        assert np.array_equal(got[:, :64], run(qh.OUT_F32)[:, :64])
    out = torch.full((batch, rows), float("nan"), dtype=torch.bfloat16, device=device)
    qh.call("qllm_fp4_swiglu_bf16_tall_cut", matrices[0], matrices[1], qh.ptr(d_act),
            d_act.numel() * 2, qh.ptr(out), batch, qh.ptr(workspace), size, None)
    product = ol.silu_product(want, wants[1], True)
    # two roundings to bf16 (the gate's SiLU, the product), each of which may fall
    # to the neighbouring value, at most 2^-7 of it away
    error = np.abs(out.double().cpu().numpy() - product)
    assert (error <= 2.0 ** -6 * np.abs(product) + 4 * bound * (1 + np.abs(wants[1]))).all()
    assert layout(0, own) == (plain[0], own)
    for parts in {own, min(2, padded // 64)}:
        sums = torch.full((parts, batch, rows), float("nan"), device=device)
        qh.call("qllm_fp4_gemm_bf16_tall_partial", matrices[0], qh.ptr(d_act),
                d_act.numel() * 2, qh.ptr(sums), parts, batch, None)
        assert np.abs(sums.double().sum(0).cpu().numpy() - want).max() < bound


# (as above; parts of the tiles past the last full round of the compute units, 0: whole)
@pytest.mark.parametrize("scheme,rows,padded,batch,plain,swiglu,tails", [
    (F16, 8228, 2112, 1254, (128, False), (128, False), (3, 0)),
    (F16, 5100, 2112, 1360, (80, False), (128, False), (3, 0)),
    (F16, 6176, 4160, 1201, (112, False), (128, False), (4, 0)),
    (UE8M0, 8228, 2112, 1254, (80, False), (128, False), (4, 0)),
    (F16, 4100, 2112, 1254, (64, False), (80, False), (0, 4)),
    (F16, 5100, 2112, 777, (48, False), (112, False), (0, 4)),
    (UE8M0, 4100, 4160, 1201, (64, False), (112, False), (0, 2)),
    (UE8M0, 6176, 2112, 1307, (80, False), (128, False), (0, 4)),
    (F16, 6180, 2112, 66, (48, True), (80, True), (0, 0)),
    (UE8M0, 6180, 1024, 1003, (112, False), (112, False), (0, 0))])
def test_cut_last_tiles_match_the_product(device, scheme, rows, padded, batch, plain, swiglu,
                                          tails):
    """Workgroups of 80 and 112 batch rows, and launches that cut the tiles of their last
    round alone: batches and weight rows that end inside a workgroup, a residual that is
    the output, segments, gate and up; no more workspace than asked for."""
    rng = np.random.default_rng(rows + batch)
    act = ol.bf16_round(rng.standard_normal((batch, padded)).astype(np.float32))
    d_act = gu.device_tensor(ol.bf16_bits(act), device)
    act64 = torch.from_numpy(act).to(device, torch.float64)
    matrices, wants, keep = [], [], []
    for _ in range(2):
        codes, scales = synth.fp4_matrix(rng, rows, padded, scheme)
        values = torch.from_numpy(synth.dequantize(codes, scales, scheme)).to(device)
        wants.append(act64 @ values.T)
        tensors = gu.device_tensor(codes, device), gu.device_tensor(scales, device)
        matrix, kept = qh.prepack(qh.fp4_matrix(*tensors, rows, padded, padded, scheme),
                                  device)
        matrices.append(matrix)
        keep.append((tensors, kept))
    del values
    size = max(qh.call("qllm_fp4_tall_parts_bytes", matrices[0], kind, batch)
               for kind in (0, 1))
    workspace = torch.full((size // 4 + 4,), float("nan"), device=device)

    for gate_and_up, expected in ((0, plain), (1, swiglu)):
        found = qh.LaunchLayout()
        qh.call("qllm_fp4_tall_layout", matrices[0], gate_and_up, batch, size, 0,
                ctypes.byref(found))
        assert (found.batch_rows, found.parts > 1) == expected
        assert qh.call("qllm_fp4_tall_tail_parts", matrices[0], gate_and_up, batch,
                       size) == tails[gate_and_up]
        assert qh.call("qllm_fp4_tall_tail_parts", matrices[0], gate_and_up, batch, 0) == 0
    # F32 sums of `padded` exact products, in any order
    want = wants[0]
    bound = 2e-6 * np.sqrt(padded) * want.abs().max().item()
    rest = torch.randn((batch, rows), device=device)

    def run(kind, residual=None):
        out = torch.full((batch, rows), float("nan"), device=device,
                         dtype=torch.bfloat16 if kind == qh.OUT_BF16 else torch.float32)
        if residual is not None:
            residual = out.copy_(residual)
        qh.call("qllm_fp4_gemm_bf16_tall_cut", matrices[0], qh.ptr(d_act),
                d_act.numel() * 2, qh.ptr(out), kind, qh.ptr(residual), batch,
                qh.ptr(workspace), size, None)
        return out

    product = run(qh.OUT_F32)
    assert (product.double() - want).abs().max() < bound
    assert torch.equal(run(qh.OUT_BF16), product.bfloat16())
    # (the product and the residual are added once more in F32)
    assert (run(qh.OUT_F32, rest).double() - rest.double() - want).abs().max() < bound + 1e-6
    if rows % 32 == 0:
        widths = 64, rows - 64
        outs = [torch.full((batch, n), float("nan"), device=device) for n in widths]
        segments = (qh.GemmSegment * 2)(*[qh.GemmSegment(qh.ptr(o), n, qh.OUT_F32)
                                          for o, n in zip(outs, widths)])
        qh.call("qllm_fp4_gemm_bf16_tall_split_cut", matrices[0], qh.ptr(d_act),
                d_act.numel() * 2, ctypes.addressof(segments), 2, batch,
                qh.ptr(workspace), size, None)
        assert torch.equal(torch.cat(outs, dim=1), product)
    out = torch.full((batch, rows), float("nan"), dtype=torch.bfloat16, device=device)
    qh.call("qllm_fp4_swiglu_bf16_tall_cut", matrices[0], matrices[1], qh.ptr(d_act),
            d_act.numel() * 2, qh.ptr(out), batch, qh.ptr(workspace), size, None)
    product = torch.nn.functional.silu(want).float().bfloat16().double() * wants[1]
    # two roundings to bf16 (the gate's SiLU, the product), each of which may fall
    # to the neighbouring value, at most 2^-7 of it away
    error = (out.double() - product).abs()
    assert (error <= 2.0 ** -6 * product.abs() + 4 * bound * (1 + wants[1].abs())).all()
