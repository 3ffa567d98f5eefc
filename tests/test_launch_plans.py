"""How launches are laid out and what they need, asked of the library without a GPU."""
import pytest

import qllm_hip as qh

UE8M0, F16 = qh.SCALE_UE8M0_BLOCK32, qh.SCALE_F16_BLOCK16


def matrix(rows, padded, scheme):
    """A matrix that is planned for and never read."""
    return qh.Fp4Matrix(16, 16, rows, padded, padded, scheme, 1, 0)   # tiled


@pytest.mark.parametrize("scheme", [UE8M0, F16])
@pytest.mark.parametrize("rows,padded,most", [
    (5120, 17408, 128 << 20), (10240, 5120, 128 << 20), (2048, 2048, 64 << 20),
    (1024, 1024, 32 << 20), (256, 512, 0), (5121, 17408, 0)])
def test_parts_of_prompts_fit_what_is_set_aside(rows, padded, most, scheme):
    """The bytes asked for cover every batch's advised parts, are no more than the
    most any launch has a use for, and nothing where no batch is cut."""
    m = matrix(rows, padded, scheme)
    needed = 0
    for batch in range(1, 4200):
        parts = qh.call("qllm_fp4_tall_parts", m, batch)
        if parts > 1:
            needed = max(needed, parts * batch * rows * 4)
        if batch in (1, 48, 300, 1000, 4199):
            room = qh.call("qllm_fp4_tall_parts_bytes", m, 0, batch)
            assert needed <= room <= qh.call("qllm_fp4_tall_workspace_bytes")
            # (asked for 16 rows at a time)
            assert room <= max(needed * 1.35, 16 * 16 * 16 * rows)
    assert room <= most and (room > 0) == (most > 0)
    assert qh.call("qllm_fp4_tall_parts_bytes", m, 1, 40) <= 16 * 2 * 48 * rows * 4


@pytest.mark.parametrize("element", [qh.ELEMENT_BF16, qh.ELEMENT_F32])
@pytest.mark.parametrize("rows,columns", [(2048, 640), (2048, 7680), (4096, 16384), (512, 1024),
                                          (16, 64), (5120, 5120)])
def test_part_rows_of_linears_cover_what_is_advised(rows, columns, element):
    needed = 0
    for batch in range(65, 4200):
        parts = qh.call("qllm_linear_parts", rows, columns, batch, element)
        assert parts == 1 or parts * batch <= 8192
        if parts > 1:
            needed = max(needed, parts * batch)
        if batch in (65, 100, 128, 512, 1000, 4199):
            room = qh.call("qllm_linear_part_rows", rows, columns, batch, element)
            # (asked for 64 rows at a time)
            assert needed <= room <= max(needed * 1.35, 16 * 128)
    assert qh.call("qllm_linear_part_rows", rows, columns, 64, element) == 0
