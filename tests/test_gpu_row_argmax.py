"""GPU parity of speculator_argmax (torch.argmax(logits, -1).clamp_(0, vocab_size - 1),
arctic_speculator.py:846-848, 862) against torch itself: exact indices."""
import pytest
import torch

from arcticinference_amd import _native

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def reference(logits, vocab_size):
    # the reference's expression, on the CPU in fp32 (every 16-bit value is exact in fp32, so the order and
    # the ties are the same)
    return torch.argmax(logits.float().cpu(), dim=-1).clamp_(0, vocab_size - 1)


def segments(rows, cols, dtype):
    """How many segments a row is cut into (1: not split) and a segment's elements, as the library has them."""
    code = {torch.float32: _native.DTYPE_F32, torch.float16: _native.DTYPE_F16, torch.bfloat16: _native.DTYPE_BF16}[dtype]
    parts = max(1, _native.load().arctic_argmax_workspace_bytes(rows, cols, code) // (16 * rows))
    return parts, cols if parts == 1 else -(-cols // parts) + 63 & ~63   # parts of whole 64 elements


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("shape", [(512, 128256), (64, 32000), (7, 513), (3, 5, 1000), (9, 1), (2, 7), (33, 4100)])
def test_random_logits(ops, dtype, shape):
    g = torch.Generator().manual_seed(5)
    logits = torch.randn(*shape, generator=g).to(dtype)          # bf16 makes many exact ties
    got = ops.speculator_argmax(logits.to(DEV), shape[-1])
    assert got.dtype == torch.int64 and got.shape == logits.shape[:-1]
    assert torch.equal(got.cpu(), reference(logits, shape[-1]))
    # the GPU's own torch.argmax agrees as well
    assert torch.equal(got, torch.argmax(logits.to(DEV), dim=-1))


def test_ties_take_the_lowest_index(ops):
    x = torch.zeros(6, 5000, dtype=torch.bfloat16)
    x[1, 4097], x[1, 77], x[1, 4999] = 3.0, 3.0, 3.0
    x[2] = -float("inf")                                            # a row of -inf answers 0
    x[3, 100] = -0.0                                                 # -0 == +0: still index 0
    x[4, 17], x[4, 2050] = float("inf"), float("inf")
    x[5, 4999] = 1.0
    got = ops.speculator_argmax(x.to(DEV), 5000).cpu()
    assert got.tolist() == [0, 77, 0, 0, 17, 4999]
    assert torch.equal(got, reference(x, 5000))


def test_nan_beats_every_number_and_the_first_nan_wins(ops):
    g = torch.Generator().manual_seed(6)
    x = torch.randn(5, 9000, generator=g)
    x[0, 8000] = float("nan")
    x[1, 5], x[1, 8999] = float("nan"), float("nan")
    x[2, 3000], x[2, 10] = float("nan"), float("inf")
    x[3, 100], x[3, 101] = float("inf"), -float("inf")              # a chunk sum that is NaN without any NaN in it
    for dtype in (torch.float32, torch.bfloat16, torch.float16):
        xs = x.to(dtype)
        got = ops.speculator_argmax(xs.to(DEV), 9000).cpu()
        assert got[:4].tolist() == [8000, 5, 3000, 100]
        assert torch.equal(got, reference(xs, 9000))


def test_clamp_and_row_pitch(ops):
    g = torch.Generator().manual_seed(7)
    full = torch.randn(40, 1100, generator=g).to(torch.bfloat16).to(DEV)
    for view in (full[:, :1000], full[:, 4:1003], full[::2, :999]):   # aligned pitch, odd start, skipped rows
        got = ops.speculator_argmax(view, 1000)
        assert torch.equal(got, torch.argmax(view.float(), dim=-1).clamp_(0, 999))
    # logits wider than the vocabulary (padded head): indices beyond it are clamped
    padded = torch.zeros(4, 1024, dtype=torch.float16, device=DEV)
    padded[:, 1010] = 5.0
    assert ops.speculator_argmax(padded, 1000).tolist() == [999] * 4


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_rows_that_start_between_16_byte_boundaries(ops, dtype):
    """A contiguous [rows, vocab] with an odd vocabulary (GPT-2's 50257) puts every row at another offset from a
    16-byte boundary: the elements in front of the first boundary, the 16-byte chunks and the elements behind the
    last chunk are three stretches of one row, and the lowest index among equal values may lie in any of them."""
    rows, cols = 24, 50257
    g = torch.Generator().manual_seed(8)
    x = (torch.randint(0, 9, (rows, cols), generator=g).float() - 4).to(dtype)      # ties everywhere
    x[1, :] = -float("inf")                        # answers 0, which lies in front of row 1's first boundary
    x[2, 0] = 50.0                                 # the very first element wins
    x[3, 1], x[3, 9000] = 50.0, 50.0               # equal values in front of the boundary and in a chunk
    x[4, cols - 1], x[4, 30000] = 50.0, 50.0       # ... in a chunk and behind the last chunk
    x[5, cols - 1] = 50.0                          # the very last element wins
    x[6, 2], x[6, 40000] = float("nan"), float("nan")   # the first NaN lies in front of the boundary
    x[7, 3], x[7, 4] = float("inf"), float("nan")
    d = x.to(DEV)
    assert d.data_ptr() % 16 == 0 and (cols * x.element_size()) % 16 != 0
    got = ops.speculator_argmax(d, cols)
    assert torch.equal(got.cpu(), reference(x, cols))
    assert got[[1, 2, 3, 4, 5, 6, 7]].tolist() == [0, 0, 1, 30000, cols - 1, 2, 4]
    # a view that starts one element into such a buffer, and one row alone
    view = d[:, 1:]
    assert torch.equal(ops.speculator_argmax(view, cols - 1).cpu(), reference(x[:, 1:], cols - 1))
    assert torch.equal(ops.speculator_argmax(d[5:6, 3:], cols).cpu(), reference(x[5:6, 3:], cols))


def test_empty_and_errors(ops):
    assert ops.speculator_argmax(torch.empty(0, 64, device=DEV), 64).shape == (0,)
    with pytest.raises(RuntimeError, match="non-empty last dimension"):
        ops.speculator_argmax(torch.empty(4, 0, device=DEV), 1)
    with pytest.raises(RuntimeError, match="fp32, fp16 or bf16"):
        ops.speculator_argmax(torch.zeros(4, 8, dtype=torch.float64, device=DEV), 8)
    with pytest.raises(RuntimeError, match="last dimension must be contiguous"):
        ops.speculator_argmax(torch.zeros(8, 4, device=DEV).t(), 8)


def test_random_configurations(ops):
    """Seeded sweep over types, row counts, row lengths around the chunk and workgroup sizes, row pitches, start
    offsets (rows that start between two 16-byte boundaries read their first elements one by one), value ranges with many ties, and sprinkled NaN / inf."""
    import random
    rnd = random.Random(13)
    for it in range(60):
        g = torch.Generator().manual_seed(700 + it)
        dtype = rnd.choice([torch.bfloat16, torch.float16, torch.float32])
        rows = rnd.choice([1, 2, 17, 130])
        cols = rnd.choice([1, 2, 7, 8, 9, 63, 64, 65, 255, 256, 257, 1023, 1025, 4096, 8200, 33000])
        pad, off = rnd.choice([0, 0, 1, 8, 24]), rnd.choice([0, 0, 1, 3, 8])
        levels = rnd.choice([2, 5, 1000])                 # few distinct values: ties everywhere
        base = torch.randint(0, levels, (rows, off + cols + pad), generator=g).float() - levels / 2
        for special in (float("nan"), float("inf"), -float("inf")):
            if rnd.random() < 0.3:
                r, c = rnd.randrange(rows), rnd.randrange(off + cols + pad)
                base[r, c] = special
        base = base.to(dtype)
        logits = base[:, off:off + cols]
        vocab = rnd.choice([cols, max(1, cols - 3), cols + 5])
        got = ops.speculator_argmax(base.to(DEV)[:, off:off + cols], vocab)
        want = torch.argmax(logits.float(), dim=-1).clamp_(0, vocab - 1)
        assert torch.equal(got.cpu(), want), f"configuration {it}: {dtype}, {rows} x {cols}, pad {pad}, offset {off}"


@pytest.mark.parametrize("rows", [257, 300, 512, 513, 768, 769])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_row_counts_around_the_in_step_kernel(ops, rows, dtype):
    """Launches of 257 to 512 rows of more than 4096 16-byte chunks (here the longest) keep the waves of a row in step, a
    chunk at a time, behind a barrier whose trip count has to be the same for every wave whatever the row length; shorter rows
    and more of them do not.  Rows shorter than one chunk per lane, rows with a ragged last batch and an element-wise tail, ties
    everywhere, NaN and infinities, pitched rows."""
    g = torch.Generator().manual_seed(900 + rows)
    for cols, pad in ((8, 0), (1000, 8), (4100, 0), (8200, 24), (33001, 7)):
        base = (torch.randint(0, 7, (rows, cols + pad), generator=g).float() - 3)
        base[rows // 2, cols // 2] = float("nan")
        base[rows - 1, 0] = float("inf")
        base[0, cols - 1] = float("inf")
        base[1] = -float("inf")
        base = base.to(dtype)
        got = ops.speculator_argmax(base.to(DEV)[:, :cols], cols)
        want = torch.argmax(base[:, :cols].float(), dim=-1)
        assert torch.equal(got.cpu(), want), f"{rows} x {cols} (+{pad}), {dtype}"


@pytest.mark.parametrize("rows,cols,dtype,pad,cut", [
    (1, 81920, torch.bfloat16, 0, 10), (1, 81919, torch.float16, 0, 9),
    (85, 128257, torch.float16, 0, 8), (86, 128256, torch.bfloat16, 0, 8), (85, 144000, torch.bfloat16, 1, 6),
    (5, 131103, torch.bfloat16, 3, 16), (3, 40960, torch.float32, 0, 10), (2, 300001, torch.float32, 1, 16),
    (257, 98304, torch.bfloat16, 0, 8), (260, 49160, torch.float32, 0, 8), (513, 80008, torch.float16, 0, 8)])
def test_rows_split_over_workgroups(ops, rows, cols, dtype, pad, cut):
    """Rows are cut into segments (some few, some a few more than one or two for every CU): single maxima, tied pairs, infinities and NaNs on both sides of
    the cuts, in the middle and at the ends, another answer every time, in eager calls whose outputs take the blocks of
    the ones before and in a captured graph whose inputs change between replays (the workspace keeps what the last replay
    left)."""
    g = torch.Generator().manual_seed(cols)
    parts, segment = segments(rows, cols, dtype)
    assert parts == cut
    places = [segment, 0, cols - 1, segment - 1, parts // 2 * segment + 17, cols - 2, (parts - 1) * segment]
    at = lambda r, k: places[(r + k) % len(places)]
    levels = torch.tensor([-float("inf"), -2.0, -0.0, 0.0, 1.5])
    batches = []
    for k in range(9):
        x = levels[torch.randint(0, 5, (rows, cols + pad), generator=g)]
        for r in range(rows):
            if k < 4:      # one maximum
                x[r, at(r, k)] = 3.0
            elif k == 4:   # a tied pair
                x[r, at(r, 0)] = x[r, at(r, 3)] = 3.0
            elif k == 5:   # infinity, with the other one in its chunk
                p = at(r, 2)
                x[r, p ^ 1 if p ^ 1 < cols else p - 1] = -float("inf")
                x[r, p] = float("inf")
            elif k == 6:   # NaNs beat infinity, the first one wins
                x[r, at(r, 1)] = float("inf")
                x[r, at(r, 2)] = x[r, at(r, 5)] = float("nan")
            elif k == 7:   # nothing but the lowest value
                x[r] = -float("inf")
        batches.append(x.to(dtype))   # the last batch: many equal maxima
    on_gpu = [x.to(DEV)[:, :cols] for x in batches]
    for _ in range(2):
        for x, y in zip(batches, on_gpu):
            assert torch.equal(ops.speculator_argmax(y, cols).cpu(), reference(x[:, :cols], cols))
    static = torch.empty(rows, cols + pad, dtype=dtype, device=DEV)[:, :cols]
    static.copy_(on_gpu[0])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = ops.speculator_argmax(static, cols - 1)
    assert got.shape == (rows,) and got.is_contiguous()
    for x, y in zip(batches + batches[:2], on_gpu + on_gpu[:2]):
        static.copy_(y)
        graph.replay()
        assert torch.equal(got.cpu(), reference(x[:, :cols], cols - 1))


@pytest.mark.parametrize("rows,cols,dtype,pad,split", [
    (48, 65536, torch.bfloat16, 0, True), (48, 65535, torch.bfloat16, 0, False), (49, 65536, torch.float16, 0, False),   # 8192 chunks
    (71, 80000, torch.bfloat16, 0, True), (72, 80000, torch.bfloat16, 0, True), (72, 79999, torch.bfloat16, 0, False),   # 10000
    (9, 40959, torch.float32, 0, False),
    (85, 81920, torch.bfloat16, 0, True), (85, 144000, torch.float16, 0, True),           # eight segments, six
    (86, 83039, torch.bfloat16, 1, False), (86, 83040, torch.bfloat16, 1, True),          # 180 chunks for each row but 5100
    (128, 71759, torch.float32, 0, False), (128, 72000, torch.float32, 1, True), (129, 144512, torch.bfloat16, 0, False),
    (256, 98304, torch.bfloat16, 0, False), (257, 98304, torch.bfloat16, 0, True), (304, 98304, torch.float16, 0, True),
    (305, 98304, torch.float16, 0, False), (288, 49152, torch.float32, 0, True), (289, 49152, torch.float32, 0, False),
    (289, 98304, torch.float32, 0, True),
    (257, 98304, torch.bfloat16, 3, True),   # not split where rows start anywhere (the segments are those of aligned ones)
    (512, 80000, torch.bfloat16, 0, False), (513, 80000, torch.bfloat16, 0, True), (600, 80000, torch.bfloat16, 0, True),
    (601, 80000, torch.float16, 0, False), (704, 80000, torch.bfloat16, 0, False), (705, 80000, torch.float16, 0, False),
    (601, 229368, torch.bfloat16, 0, False), (601, 229376, torch.bfloat16, 0, True), (704, 229376, torch.bfloat16, 0, True),
    (705, 229376, torch.float16, 0, False)])
def test_row_counts_where_the_split_begins_and_ends(ops, rows, cols, dtype, pad, split):
    """The winner in every segment of a row (where it is not split, in every eighth), on both sides of the cuts and at both ends,
    ties of the first and the last place."""
    x = torch.randint(-3, 2, (rows, cols + pad), generator=torch.Generator().manual_seed(rows), dtype=torch.int8).to(dtype)
    parts, segment = segments(rows, cols, dtype)
    assert (parts > 1) == split
    if parts == 1:
        parts, segment = 8, -(-cols // 8)
    places = [0, cols - 1, *(min(cols - 1, segment * k + d) for k in range(1, parts) for d in (-1, 0, 63, 64))]
    for r in range(0, rows, 2):
        x[r, places[r // 2 % len(places)]] = 4.0
        if r % 3 == 0:
            x[r, cols - 1] = 4.0
    for _ in range(2):
        assert torch.equal(ops.speculator_argmax(x.to(DEV)[:, :cols], cols).cpu(), reference(x[:, :cols], cols))


@pytest.mark.parametrize("rows,cols,dtype,pad", [
    (256, 40000, torch.bfloat16, 0), (257, 32775, torch.float16, 0), (257, 32776, torch.float16, 0), (300, 32783, torch.bfloat16, 2),
    (420, 65536, torch.bfloat16, 0), (421, 65543, torch.bfloat16, 0), (421, 65544, torch.bfloat16, 3), (512, 48000, torch.float16, 0),
    (512, 47999, torch.float16, 0), (513, 48000, torch.bfloat16, 1), (512, 16387, torch.float32, 0), (512, 16388, torch.float32, 0),
    (300, 20483, torch.float32, 2), (384, 14400, torch.float32, 0), (384, 14399, torch.float32, 1), (385, 14400, torch.float32, 1),
    (421, 49593, torch.bfloat16, 0), (421, 49601, torch.float16, 0), (421, 56000, torch.bfloat16, 0), (421, 55992, torch.bfloat16, 0)])
def test_where_waves_keep_in_step_and_where_not(ops, rows, cols, dtype, pad):
    """The winner at a row's ends and about the ends of its batches of one and of four chunks for each of 1024 lanes."""
    x = torch.randint(-3, 2, (rows, cols + pad), generator=torch.Generator().manual_seed(cols), dtype=torch.int8).to(dtype)
    batch = 1024 * (4 if dtype is torch.float32 else 8)
    places = [0, cols - 1, *(min(cols - 1, batch * k + d) for k in range(1, 9) for d in (-1, 0, 7))]
    for r in range(0, rows, 2):
        x[r, places[r // 2 % len(places)]] = 4.0
        if r % 3 == 0:
            x[r, cols - 1] = 4.0
    assert torch.equal(ops.speculator_argmax(x.to(DEV)[:, :cols], cols).cpu(), reference(x[:, :cols], cols))


def test_split_rows_on_two_streams_at_once(ops):
    """Each call exchanges winners in memory of its own: calls of two streams that run at the same time do not meet."""
    cols = 128256
    logits = [torch.randn(rows, cols, generator=torch.Generator().manual_seed(rows)).to(torch.bfloat16) for rows in (5, 32)]
    want = [reference(x, cols) for x in logits]
    on_gpu = [x.to(DEV) for x in logits]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    got = [[], []]
    for _ in range(60):
        for k in (0, 1):
            with torch.cuda.stream(streams[k]):
                got[k].append(ops.speculator_argmax(on_gpu[k], cols))
    torch.cuda.synchronize()
    for k in (0, 1):
        assert all(torch.equal(t.cpu(), want[k]) for t in got[k])


@pytest.mark.parametrize("shape", [(3, 128256), (2, 2, 100000), (4, 1000)])
def test_the_result_is_the_answers_alone(ops, shape, tmp_path):
    """What the workgroups of a split row exchange is no part of the tensor's storage: it is not saved with it, and the
    tensor can be resized."""
    logits = torch.randn(*shape, generator=torch.Generator().manual_seed(8)).to(torch.bfloat16)
    got = ops.speculator_argmax(logits.to(DEV), shape[-1])
    want = reference(logits, shape[-1])
    assert got.untyped_storage().nbytes() == want.numel() * 8
    torch.save(got, tmp_path / "tokens.pt")
    saved = torch.load(tmp_path / "tokens.pt", weights_only=True)
    assert saved.untyped_storage().nbytes() == want.numel() * 8 and torch.equal(saved.cpu(), want)
    grown = got.clone().resize_(want.numel() + 1000)
    got.resize_(want.numel() + 1000)[want.numel():] = 0
    assert torch.equal(got[:want.numel()].cpu(), want.flatten()) and torch.equal(grown[:want.numel()].cpu(), want.flatten())


def test_rows_that_are_not_split_hold_no_memory_for_it(ops):
    """300 rows that start between 16-byte boundaries get a workgroup each, and their answers a block of their own size."""
    for pad, least, most in ((1, 0, 4096), (0, 300 * 8 * 16, 1 << 20)):
        logits = torch.zeros(300, 98304 + pad, dtype=torch.bfloat16, device=DEV)
        ops.speculator_argmax(logits[:, :98304], 98304)
        before = torch.cuda.memory_allocated()
        got = ops.speculator_argmax(logits[:, :98304], 98304)
        assert least <= torch.cuda.memory_allocated() - before <= most and int(got.max()) == 0


def test_no_rows_of_any_width(ops):
    got = ops.speculator_argmax(torch.empty(0, 2 ** 31 + 8, device=DEV, dtype=torch.bfloat16), 7)
    assert got.shape == (0,) and got.dtype == torch.int64
