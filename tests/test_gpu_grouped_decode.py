"""The grouped form of the decode kernel (a few rows per slot in use): against the naive kernel and the persistent launch, exactly, on small
integers and powers of two, where a slot's rows pass a group of 16 or a pass of 32, slots are empty or without an expert, columns do not
fill a tile and slabs do not fill the waves; and stale offsets stay inside the operands."""
import pytest
import torch

import modular_amd as mx
from modular_amd import _lib

pytestmark = pytest.mark.gpu
BLK = mx.blockwise_fp8_config()

# rows of the slots, their experts, N, K: one slab of one row; every edge of a slot; one tile per slot; more tiles than blocks on the chip (32 weight rows each),
# fewer (16); a tile of two columns
CASES = [([1], [0], 16, 128), ([1, 0, 16, 17, 31, 0, 32, 33, 64, 65], [3, 0, 1, 9, -1, 2, 5, 4, 6, 7], 200, 640), ([2, 0, 3], [2, 1, 0], 32, 2176),
         ([1] * 24, list(range(24)), 1536, 256), ([40, 1], [1, 0], 66, 7168), ([3, 5, 2], [0, -1, 2], 8, 384)]


def exact(counts, ids, N, K, kind, dev, spare=3):
    g = torch.Generator().manual_seed(N + K + len(counts))
    T, E = sum(counts) + spare, max(len(counts), max(ids) + 1)
    ints = lambda *s: torch.randint(-2, 3, s, generator=g).float().to(torch.float8_e4m3fn).to(dev)
    power = lambda *s: (2.0 ** torch.randint(-1, 2, s, generator=g).float()).to(dev)
    off = torch.zeros(len(counts) + 1, dtype=torch.int64)
    off[1:] = torch.cumsum(torch.tensor(counts), 0)
    scales = (power(K // 128, -(-T // 4) * 4), power(E, -(-N // 128), K // 128)) if kind == "block" else (power(T, 1), power(E, N, 1))
    return ints(T, K), ints(E, N, K), *scales, off.to(torch.uint32).to(dev), torch.tensor(list(ids) + [-1] * (E - len(ids)), dtype=torch.int32).to(dev)


def run(case, kind, out, active, row_index=None, most=None):
    a, b, sa, sb, off, ids = case
    stats = torch.tensor([most or a.shape[0], active], dtype=torch.int64).to(torch.uint32)
    if kind == "row":
        return mx.grouped_matmul_rowwise_dynamic_scaled_fp8(a, b, sa, sb, off, ids, stats, out_type=out)
    return mx.grouped_dynamic_scaled_fp8_matmul(a, b, sa, sb, off, ids, stats, BLK.input_scale, BLK.weight_scale, out_type=out,
                                                **({} if row_index is None else {"out_row_index": row_index}))


@pytest.mark.parametrize("kind", ["block", "row"])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_bits_of_the_persistent_launch(dev, tune, case, kind):
    counts, ids, N, K = CASES[case]
    operands, used = exact(counts, ids, N, K, kind, dev), sum(counts)
    for out in (torch.bfloat16, torch.float32):
        tune(MAXFP8_GROUPED_DECODE=100000)
        got = run(operands, kind, out, len(counts))
        tune(MAXFP8_GROUPED_DECODE=0)
        want = run(operands, kind, out, len(counts))
        assert torch.equal(got[:used], want[:used])
        # ... which is the sum itself
        a, b, sa, sb = (t.double().cpu() for t in operands[:4])
        at = 0
        for rows, e in zip(counts, ids):
            x = a[at:at + rows]
            if e < 0 or rows == 0:
                ref = torch.zeros(rows, N, dtype=torch.float64)
            elif kind == "row":
                ref = (x @ b[e].T) * sa[at:at + rows] * sb[e].T
            else:
                xs = x * sa[:, at:at + rows].repeat_interleave(128, 0).T
                ref = xs @ (b[e] * sb[e].repeat_interleave(128, 0)[:N].repeat_interleave(128, 1)).T
            assert torch.equal(got[at:at + rows].cpu(), ref.to(out))
            at += rows


def test_row_index_many_slots_and_stale_offsets(dev, tune):
    tune(MAXFP8_GROUPED_DECODE=100000)
    counts = [1 if z % 7 == 3 else 0 for z in range(512)]         # 73 of 512 slots, in both halves of the list
    operands = exact(counts, list(range(512)), 48, 256, "block", dev, spare=0)
    T = sum(counts)
    order = torch.randperm(T, generator=torch.Generator().manual_seed(1))
    plain, moved = run(operands, "block", torch.bfloat16, 512), run(operands, "block", torch.bfloat16, 512, order.to(torch.int64).to(torch.uint32).to(dev))
    assert torch.equal(moved[order.to(dev)], plain)
    # offsets past the rows there are: held to them
    a, b, sa, sb, off, ids = exact([5, 6], [1, 0], 40, 384, "block", dev, spare=0)
    want = run((a, b, sa, sb, off, ids), "block", torch.bfloat16, 2)
    stale = torch.tensor([0, 5, 1 << 30], dtype=torch.int64).to(torch.uint32).to(dev)
    assert torch.equal(run((a, b, sa, sb, stale, ids), "block", torch.bfloat16, 2), want)


# rows in all, slots, the caller's bound on a slot's rows (None: the rows in all)
@pytest.mark.parametrize("rows, slots, most, decode", [(448, 20, None, True), (449, 20, None, False), (84, 1, None, True), (85, 1, None, False), (104, 2, None, True),
                                                       (105, 2, None, False), (440, 20, 128, True), (440, 20, 129, False), (512, 300, 2, False)])
def test_up_to_how_many_rows(dev, rows, slots, most, decode):
    from torch.profiler import ProfilerActivity, profile

    even = rows // slots
    operands = exact([rows - even * (slots - 1)] + [even] * (slots - 1), list(range(slots)), 32, 128, "block", dev, spare=0)
    with profile(activities=[ProfilerActivity.CUDA]) as seen:
        run(operands, "block", torch.bfloat16, slots, most=most)
        torch.cuda.synchronize()
    names = [e.name for e in seen.events()]
    assert any("gemm_grouped_skinny_kernel" in n for n in names) == decode and any("gemm_grouped_persist_kernel" in n for n in names) != decode


# one slot of most of the rows: its 32-row parts are tiles of their own (up to 14 of them, in front of, between and behind other slots; without an expert)
@pytest.mark.parametrize("counts, ids", [([448], [0]), ([1, 0, 300, 31, 33], [2, 0, 1, 3, 4]), ([0] * 300 + [161, 2] + [0] * 200 + [97], [0] * 300 + [1, 0] + [1] * 200 + [2]),
                                         ([5, 230, 200], [1, -1, 0])])
def test_one_slot_of_most_of_the_rows(dev, tune, counts, ids):
    operands, used = exact(counts, ids, 72, 640, "block", dev), sum(counts)
    T = operands[0].shape[0]
    order = torch.cat([torch.randperm(used, generator=torch.Generator().manual_seed(2)), torch.arange(used, T)])
    index = order.to(torch.int64).to(torch.uint32).to(dev)
    got = {}
    for rows in (100000, 0):
        tune(MAXFP8_GROUPED_DECODE=rows)
        got[rows] = [run(operands, "block", torch.bfloat16, len(counts), i) for i in (None, index)]
    assert torch.equal(got[100000][0][:used], got[0][0][:used])
    assert torch.equal(got[100000][1][order[:used].to(dev)], got[0][0][:used])


def test_one_slot_of_most_of_the_rows_is_no_slower(dev, tune):
    """448 rows of one slot of 64, 3072 x 4096: 40 us, on the persistent launch 70; with a slot's 32-row parts one after the other it was 94."""
    counts = [0] * 20 + [448] + [0] * 43
    a, b, sa, sb, off, _ = exact(counts, [0] * 64, 3072, 4096, "block", dev, spare=0)
    case = a, b, sa, sb, off, torch.arange(64, dtype=torch.int32, device=dev)

    def microseconds():
        graph = torch.cuda.CUDAGraph()
        run(case, "block", torch.bfloat16, 64)
        with torch.cuda.graph(graph):
            for _ in range(8):
                run(case, "block", torch.bfloat16, 64)
        times = []
        for _ in range(5):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            graph.replay()
            end.record()
            torch.cuda.synchronize()
            times.append(start.elapsed_time(end) * 1000 / 8)
        return min(times)

    tune(MAXFP8_GROUPED_DECODE=448)
    decode = microseconds()
    tune(MAXFP8_GROUPED_DECODE=0)
    assert decode < microseconds()
