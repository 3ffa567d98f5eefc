"""How launches are laid out and what they need, asked of the library without a GPU."""
import ctypes

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


@pytest.mark.parametrize("scheme", [UE8M0, F16])
@pytest.mark.parametrize("rows,timed", [(3068, False), (3072, True), (17408, True),
                                        (17412, False), (32000, False)])
def test_untimed_matrices_keep_the_old_heights(rows, timed, scheme):
    """Workgroups of 80 and 112 batch rows and tiles that are cut alone."""
    m = matrix(rows, 2048, scheme)
    room = qh.call("qllm_fp4_tall_workspace_bytes")
    new = set()
    for batch in range(33, 2400, 7):
        for swiglu in (0, 1):
            layout = qh.LaunchLayout()
            qh.call("qllm_fp4_tall_layout", m, swiglu, batch, room, 0, ctypes.byref(layout))
            cut = qh.call("qllm_fp4_tall_tail_parts", m, swiglu, batch, room)
            new.add(layout.batch_rows in (80, 112) or cut > 0)
    assert new == ({True, False} if timed else {False})


@pytest.mark.parametrize("scheme", [UE8M0, F16])
@pytest.mark.parametrize("padded", [1 << 24, 1 << 27, (1 << 31) + 64])
def test_matrices_past_32_bit_offsets_are_taken(padded, scheme):
    for swiglu in (0, 1):
        for batch, height in ((1, 16), (20, 32), (40, 64), (700, 64)):
            layout = qh.LaunchLayout()
            qh.call("qllm_fp4_tall_layout", matrix(40, padded, scheme), swiglu, batch, 0, 0,
                    ctypes.byref(layout))
            assert (layout.batch_rows, layout.parts) == (height, 1)


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


@pytest.mark.parametrize("rows,columns,batch,parts,form", [
    (12288, 4096, 300, 0, (64, 128)), (12288, 4096, 340, 0, (128, 128)),   # 480, 576 workgroups
    (10912, 1536, 400, 0, (64, 128)), (10944, 1536, 400, 0, (128, 128)),   # 2^24 weights
    (16384, 1472, 300, 0, (64, 128)), (16384, 1536, 300, 0, (128, 128)),   # 24 steps
    (4096, 12288, 160, 8, (128, 128)), (4096, 12224, 160, 8, (64, 128)),   # of a part
    (2816, 1024, 1500, 0, (64, 128)), (3072, 3072, 1500, 0, (64, 128))])
def test_small_workgroups_of_large_matrices_are_two_a_cu(rows, columns, batch, parts, form):
    segment = qh.LinearSegment(1 << 12, 1 << 13, 1 << 14, rows, columns, columns, rows, rows,
                               qh.LINEAR_PARTIALS if parts else 0, 0, parts)
    layout = qh.LaunchLayout()
    qh.call("qllm_linear_layout", ctypes.byref(segment), 1, batch, qh.ELEMENT_BF16,
            ctypes.byref(layout))
    assert (layout.batch_rows, layout.weight_rows) == form


def test_rows_far_apart_have_tall_layouts():
    """Those of rows side by side, but for the largest."""
    for rows, batch in ((64, 65), (8192, 300), (40000, 200), (40000, 300), (40000, 3000)):
        found = []
        for stride in (128, 1 << 24, 1 << 30):
            segment = qh.LinearSegment(1 << 12, 1 << 13, 1 << 14, rows, 128, stride, rows, rows,
                                       0, 0, 0)
            layout = qh.LaunchLayout()
            qh.call("qllm_linear_layout", ctypes.byref(segment), 1, batch, qh.ELEMENT_BF16,
                    ctypes.byref(layout))
            found.append((layout.batch_rows, layout.weight_rows))
        near = {(128, 256): (128, 128)}.get(found[0], found[0])
        assert near in ((64, 128), (128, 128)) and found[1:] == [near] * 2


def attention(rows, first, query_heads, kv_heads, splits=1, head_dim=256, split_tokens=0):
    """A prompt's attention that is planned for and never run."""
    return qh.Q4hAttentionLaunch(
        rows=rows, first_context_tokens=first + 1, query_heads=query_heads, kv_heads=kv_heads,
        head_dim=head_dim, split_tokens=split_tokens, maximum_splits=splits, page_tokens=64)


@pytest.mark.parametrize("query_heads,kv_heads,rows,first,shared", [
    (24, 4, 20, 9000, False), (24, 4, 2, 2000, False),       # few rows over a long context
    (16, 16, 8, 4000, False), (32, 32, 2, 9000, False),      # ... also with workgroups enough
    (24, 4, 48, 1000, True), (24, 4, 100, 9000, True),
    (24, 4, 683, 2000, True), (24, 4, 800, 3000, True), (24, 4, 938, 500, True),
    (24, 2, 800, 500, True), (8, 1, 3000, 1000, True), (24, 4, 3001, 0, True)])
def test_prompts_share_cache_tiles_where_that_takes_less(query_heads, kv_heads, rows, first,
                                                         shared):
    """The form of a prompt's attention at head_dim 256 and its splits, on either side of
    a full round of workgroups."""
    batch = 32 // (query_heads // kv_heads)
    alone = min(8, max(1, -(-256 // (-(-rows // batch) * kv_heads))))
    splits = qh.call("qllm_attention_paged_q4h_shared_splits",
                     attention(rows, first, query_heads, kv_heads), batch, alone, 8)
    assert (splits > 0) == shared and splits <= 8
    if shared and rows >= 100:   # (of few rows the batches may take those splits as well)
        launch = attention(rows, first, query_heads, kv_heads, splits)
        assert qh.call("qllm_attention_paged_q4h_shares_tiles", launch, batch) == 1
    # the few heads' shorter round is cut so that compute units do not idle
    if (query_heads, rows) == (8, 3000):
        assert splits > 1


@pytest.mark.parametrize("change", [dict(head_dim=128), dict(split_tokens=64), dict(rows=0),
                                    dict(kv_heads=0), dict(query_heads=2)])
def test_launches_that_cannot_share_tiles(change):
    sizes = dict(rows=1000, first=0, query_heads=24, kv_heads=4)
    assert qh.call("qllm_attention_paged_q4h_shared_splits", attention(**sizes), 5, 1, 8) > 0
    launch = attention(**{**sizes, **change})
    assert qh.call("qllm_attention_paged_q4h_shared_splits", launch, 5, 1, 8) == 0
    assert qh.call("qllm_attention_paged_q4h_shares_tiles", launch, 5) == 0


@pytest.mark.parametrize("query_heads,kv_heads,rows,first,form", [
    (64, 8, 1, 0, (0, 1)), (64, 8, 300, 0, (0, 1)), (64, 8, 16384, 0, (1, 1)),
    (64, 8, 120, 2048, (0, 1)),        # two splits: 320 workgroups, a second round
    (64, 8, 48, 8000, (0, 4)),         # 256 workgroups
    (64, 8, 1000, 2048, (1, 3)),       # 504 workgroups, two rounds
    (16, 4, 1500, 2048, (0, 1)), (32, 32, 48, 8000, (0, 8)), (3, 1, 65535, 0, (1, 1)),
    (512, 512, 100, 100, None), (7, 7, 100000, 60000, None)])
@pytest.mark.parametrize("most", [1, 3, 8])
def test_prompt_forms_of_128_dimensions(query_heads, kv_heads, rows, first, form, most):
    batch = 48 // (query_heads // kv_heads)
    splits = ctypes.c_uint32()
    shared = qh.call("qllm_attention_paged_q4h_prompt_form",
                     attention(rows, first, query_heads, kv_heads, head_dim=128), batch, most,
                     ctypes.byref(splits))
    assert shared in (0, 1) and 1 <= splits.value <= most
    workgroups = kv_heads * -(-rows // (batch * (8 if shared else 1)))
    assert splits.value == 1 or workgroups * splits.value <= (512 if shared else 256)
    if most == 8 and form:
        assert (shared, splits.value) == form


@pytest.mark.parametrize("change", [dict(head_dim=256), dict(split_tokens=64), dict(rows=0),
                                    dict(kv_heads=0), dict(query_heads=2)])
def test_launches_without_a_prompt_form(change):
    sizes = {**dict(rows=1000, first=0, query_heads=16, kv_heads=4, head_dim=128), **change}
    splits = ctypes.c_uint32(9)
    assert qh.call("qllm_attention_paged_q4h_prompt_form", attention(**sizes), 12, 8,
                   ctypes.byref(splits)) == 0 and splits.value == 0


@pytest.mark.parametrize("query_heads,kv_heads,rows,first,form", [
    (48, 8, 1168, 0, (1, 2)), (32, 32, 2196, 193, (1, 2)), (32, 8, 1156, 0, (1, 3)),
    (16, 8, 4302, 0, (1, 2)), (28, 4, 1199, 0, (1, 3)), (64, 2, 572, 168, (1, 2)),
    (40, 40, 589, 0, (0, 1))])
def test_prompt_forms_of_close_estimates(query_heads, kv_heads, rows, first, form):
    """Where the estimates are close, batches of their own up to 31 of them and splits for
    one workgroup a compute unit: 6 to 14 % less than the least of the estimates took."""
    splits = ctypes.c_uint32()
    shared = qh.call("qllm_attention_paged_q4h_prompt_form",
                     attention(rows, first, query_heads, kv_heads, head_dim=128),
                     48 // (query_heads // kv_heads), 8, ctypes.byref(splits))
    assert (shared, splits.value) == form


@pytest.mark.parametrize("query_heads,kv_heads,rows,first,shared", [
    (1, 1, 65535, 0, 0), (1, 1, 65536, 0, 1), (8, 1, 65536, 0, 1), (64, 2, 70000, 0, 1), (7, 7, 65536, 0, 1),
    (7, 7, 100000, 60000, 1), (1, 1, 300000, 0, 1), (1, 1, 65535 * 8, 0, 1),
    (1, 1, 65535 * 8 + 1, 0, None), (64, 8, 1 << 20, 0, None)])
def test_prompt_forms_take_their_rows(query_heads, kv_heads, rows, first, shared):
    """Batches of their own only for rows that launch takes, 65535, whatever the estimates
    say; shared tiles up to eight times as many; beyond them no form."""
    splits = ctypes.c_uint32(9)
    form = qh.call("qllm_attention_paged_q4h_prompt_form",
                   attention(rows, first, query_heads, kv_heads, head_dim=128),
                   48 // (query_heads // kv_heads), 8, ctypes.byref(splits))
    assert (form, splits.value > 0) == ((shared, True) if shared is not None else (0, False))


@pytest.mark.parametrize("change", [dict(query_heads=15), dict(batch=13), dict(first=-1),
                                    dict(first=0xffffffff - 100)])
def test_sizes_that_no_prompt_form_takes(change):
    sizes = {**dict(rows=1000, first=0, query_heads=16, kv_heads=4, head_dim=128, batch=12),
             **change}
    batch = sizes.pop("batch")
    splits = ctypes.c_uint32(9)
    assert qh.call("qllm_attention_paged_q4h_prompt_form", attention(**sizes), batch, 8,
                   ctypes.byref(splits)) == 0 and splits.value == 0


@pytest.mark.parametrize("head_dim,most", [(128, 64), (128, 32), (128, 8), (256, 64), (256, 16),
                                           (256, 1)])
def test_exact_splits_follow_the_context(head_dim, most):
    """A tile of 32 tokens a wave at most, as long as there is room; never fewer splits for a
    longer context."""
    room = min(most, 32) if head_dim == 128 else most

    def splits(context):
        return qh.call("qllm_attention_paged_f16_splits", context, head_dim, most)

    assert splits(0) == 0 and splits(1) == splits(64) == 1
    before = 1
    for context in list(range(1, 20000, 31)) + [256 * room, 256 * room + 1, 0xffffffff]:
        found = splits(context)
        if context > 256 * room:
            assert found == 0
            continue
        assert before <= found <= room and found * 256 >= context
        assert found <= max(-(-context // 32), 16) and (found == 1 or context > 64)
        before = found if context < 19900 else 1
    assert qh.call("qllm_attention_paged_f16_splits", 100, 64, most) == 0


# ---- a norm with its projections ------------------------------------------------

MIB = 1 << 20


def normed(form, element, changes=(), width=2048, rows=(4096, 4096), partials=0):
    """How many launches qllm_linear_normed makes of one row whose buffers lie a MiB apart
    (nothing is read), a stored and a gated matrix."""
    place = {name: MIB * (16 + i) for i, name in enumerate((
        "input", "stream", "partials", "weight0", "weight1", "ins0", "ins1", "ins2", "ins3",
        "mu0", "mu1", "previous", "last", "step", "branch", "table", "ids", "out", "gated",
        "matrix0"))}
    place["matrix1"] = 256 * MIB
    other = dict(changes)
    for name in list(other):
        if name in place:
            value = other.pop(name)
            place[name] = (place[value[0]] + value[1]) if isinstance(value, tuple) else value
    columns = -(-width // 64) * 64
    shifted, tokens = "shift" in form, "tokens" in form
    pointers = ctypes.c_void_p * 6
    shift = qh.TokenShift(2, pointers(place["mu0"], place["mu1"]),
                          pointers(place["ins2"], place["ins3"]), place["previous"],
                          other.pop("slot_stride", (1 << 14) + 16), place["last"])
    norm = qh.StreamNormLaunch(
        None if tokens else place["input"], place["stream"], place["partials"], partials, width,
        (ctypes.c_void_p * 2)(place["weight0"], place["weight1"]),
        (ctypes.c_void_p * 2)(place["ins0"], place["ins1"]),
        (ctypes.c_uint32 * 2)(columns, columns), 1, width, 1e-5, element,
        ctypes.pointer(shift) if shifted else None, None, place["step"],
        place["branch"] if form == "branch" else None, 0.5, 1e-6)
    segments = (qh.LinearSegment * 2)(
        qh.LinearSegment(place["matrix0"], place["ins3" if shifted else "ins0"], place["out"],
                         rows[0], columns, columns, rows[0], rows[0], 0, 0, 1),
        qh.LinearSegment(place["matrix1"], place["ins1"], place["gated"], rows[1], columns,
                         columns, rows[1] // 2, rows[1] // 2, 2, 0, 1))
    norm.rows = other.pop("batch", 1)
    for name, value in other.items():
        setattr(segments[0], name, value)
    row = qh.TokenRows(place["table"], place["ids"], 9, 0.75)
    launches = ctypes.c_uint32()
    qh.call("qllm_linear_normed_launches", ctypes.byref(norm),
            ctypes.byref(row) if tokens else None, segments, 2, ctypes.byref(launches))
    return launches.value


FORMS = [("plain", 0), ("plain", 8), ("branch", 3), ("shift", 5), ("tokens", 0),
         ("tokens shift", 0)]


@pytest.mark.parametrize("element", [qh.ELEMENT_BF16, qh.ELEMENT_F32])
@pytest.mark.parametrize("form,partials", FORMS)
def test_a_row_and_its_projections_are_one_launch(form, partials, element):
    for width in (64, 132, 2048, 2052, 4096):
        rows = (4096, 4096) if width > 448 else (1024, 1024)
        assert normed(form, element, width=width, rows=rows, partials=partials) == 1
    assert normed(form, element, width=90, partials=partials) == 2     # no whole pieces
    assert normed(form, element, width=4100, partials=partials) == 2
    assert normed(form, element, dict(batch=2), partials=partials) == 2
    assert normed(form, element, dict(epilogue=1), partials=partials) == 2
    assert normed(form, element, dict(epilogue=3), partials=partials) == 2
    assert normed(form, element, dict(weight0=MIB + 4), partials=partials) == 2   # not aligned
    assert normed("plain", element, partials=9) == 2
    # many short tiles, and a long stored head of bf16
    assert normed("plain", element, width=256, rows=(32784, 32)) == 2
    assert normed("plain", element, width=448, rows=(32784, 32)) == 2
    assert normed("plain", element, width=512, rows=(32784, 32)) == 1


@pytest.mark.parametrize("element", [qh.ELEMENT_BF16, qh.ELEMENT_F32])
@pytest.mark.parametrize("form,partials", FORMS)
def test_a_norm_whose_inputs_are_written_over_is_two_launches(form, partials, element):
    """Projections that write over what the norm or another projection reads, the stream
    and the shift's last row likewise: the first and the last bytes of every range, and
    just past both."""
    width, size = 2048, 2 if element == qh.ELEMENT_BF16 else 4
    row = 4 * width
    reads = {"weight0": row, "weight1": row, "ins1": width * size, "matrix1": 4096 * width * 2}
    if "tokens" in form:
        reads |= {"table": 9 * width * 2}
    else:
        reads |= {"input": row}
    if partials:
        reads |= {"partials": partials * row}
    if form == "branch":
        reads |= {"branch": row}
    if "shift" in form:
        reads |= {"mu0": row, "mu1": row, "previous": row, "last": row}
    writes = {"out": 4096 * 4, "gated": 2048 * size}
    if partials or "tokens" in form:
        writes["stream"] = row
        reads["stream"] = row
    if "shift" in form:
        writes["last"] = row

    def launches(changes):
        return normed(form, element, dict(changes, slot_stride=1 << 26), partials=partials)

    for writer, written in writes.items():
        for reader, read in reads.items():
            if writer == reader or (writer, reader) == ("stream", "input"):
                continue
            # (the carried rows: every slot's)
            for place, apart in ((0, False), (read - 16, False), (16 - written, False),
                                 (read, True), (-written, True)):
                assert launches({writer: (reader, place)}) == (1 if apart else 2), (
                    writer, reader, place)


def test_a_last_row_that_is_a_carried_one_is_two_launches():
    for slot, launches in ((0, 2), (3, 2), (3.5, 1)):
        assert normed("shift", qh.ELEMENT_F32, {"last": ("previous", int(slot * ((1 << 16) + 64)))},
                      partials=2) == launches
