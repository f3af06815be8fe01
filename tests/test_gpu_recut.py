"""How calls cut their pages: a fixed plan (a chunk size) as given, whatever surrounds
a sequence, and a balanced plan over short sequences at their starts. Against the
float64 oracle at lengths where the two differ in splits, items and pieces."""

import sys

import pytest
import torch

from oracle import attention_c64
from small_q_attention_amd import _lib, cuda as sqa, inputs
from tests._helpers import assert_parity

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _announce(request):
    sys.__stderr__.write(f"\n[gpu-test] {request.node.nodeid}\n")
    sys.__stderr__.flush()


def _call(tensors, ns, pps, nbytes):
    q, k, v, bt, sl = tensors
    out = torch.full_like(q, float("nan"))
    ws = torch.full((max(nbytes, 16) // 4 + 4,), float("nan"), device="cuda").view(torch.uint8)
    _lib.launch(q, k, v, bt, sl, out, ws[:nbytes] if nbytes else None, ns, pps,
                torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("q_len", [2, 8, 16])
@pytest.mark.parametrize("chunk", [16, 48, 512, 1 << 20])
@pytest.mark.parametrize("lens", [
    [1], [63], [193], [4099],                      # one sequence: 1 page .. 257 pages
    [0, 5, 511, 513, 2050], [640] * 3, [300] * 130,  # ragged, uniform, many
])
def test_chunked_plans_run_as_given(q_len, chunk, lens):
    """Against the oracle, and the same bits whatever the size of the workspace: the
    splits are the plan's, where one as large as the automatic plan's is given too."""
    case = inputs.Case(batch=len(lens), q_len=q_len, seq_lens=lens, seed=2100 + q_len)
    host = inputs.make_inputs(case)
    tensors = tuple(t.cuda() for t in host)
    bt = tensors[3]
    ref = attention_c64(*host, 16, 8)
    label = f"q{q_len} ck{chunk} B{len(lens)}"
    out = sqa.paged_mtp_attention(*tensors, 16, max(lens), chunk_keys=chunk)
    assert_parity(out, ref, label=label)
    b = len(lens)
    ns, pps = _lib.plan_splits(0, b, q_len, 32, 8, 128, max(lens), bt.shape[1], chunk)
    own = _lib.workspace_bytes(b, q_len, 32, 8, 128, ns, pps)
    for nbytes in (own, own + (64 << 20)):
        assert torch.equal(_call(tensors, ns, pps, nbytes), out), f"{label} {nbytes} bytes"


@pytest.mark.parametrize("q_len", [2, 4, 8])
@pytest.mark.parametrize("chunk", [48, 512, 1 << 20])
def test_chunked_sequences_do_not_depend_on_their_surroundings(q_len, chunk):
    """A chunk size cuts a sequence at the same keys alone and in a batch, under a table
    of its own width and a wider one, promised its length and the batch's longest: the
    same bits (the batch's rows stay within one form of the merge kernel)."""
    lens = [700, 65, 4099] if q_len == 2 else [700, 1300]
    q, k, v, bt, sl = (t.cuda() for t in inputs.make_inputs(
        inputs.Case(batch=len(lens), q_len=q_len, seq_lens=lens, seed=2200 + q_len)))
    wide = torch.zeros(len(lens), 600, dtype=torch.int32, device="cuda")
    wide[:, :bt.shape[1]] = bt
    together = sqa.forward_v3(q, k, v, wide, sl, 16, chunk, max(lens))
    for i, n in enumerate(lens):
        one = slice(i, i + 1)
        for table in (bt[one, :-(-n // 16)].contiguous(), wide[one].contiguous()):
            alone = sqa.forward_v3(q[one].contiguous(), k, v, table, sl[one].contiguous(), 16,
                                   chunk, n)
            assert torch.equal(alone, together[one]), f"{n} keys, table of {table.shape[1]}"


@pytest.mark.parametrize("lens", [[1000], [1000] * 3, [1000, 100, 700, 330, 1], [650] * 2])
@pytest.mark.parametrize("splits,pps", [(1, 20), (5, 4), (40, 1), (2, 20)])
def test_a_plan_reads_its_pages_of_longer_sequences(lens, splits, pps):
    """A plan covers the first num_splits * pages_per_split pages of every sequence and
    no more: longer sequences see only those keys, shorter ones all of theirs."""
    batch = len(lens)
    q, k, v, bt, sl = (t.cuda() for t in inputs.make_inputs(
        inputs.Case(batch=batch, q_len=4, seq_lens=lens, seed=2200)))
    own = _lib.workspace_bytes(batch, 4, 32, 8, 128, splits, pps)
    out = _call((q, k, v, bt, sl), splits, pps, own)
    # Behind them lies the draft of the longer ones: every row sees all of the keys, as a
    # lone query at the end of a sequence of that length would.
    cover = splits * pps * 16
    seen = torch.tensor([min(n, cover) for n in lens], dtype=torch.int32)
    want = attention_c64(q.cpu()[:, 3:].contiguous(), k.cpu(), v.cpu(), bt.cpu(), seen, 16, 8)
    assert_parity(out[:, 3:].contiguous(), want, label=f"B{batch} {splits}x{pps}")
    assert torch.equal(out, _call((q, k, v, bt, sl), splits, pps, own + (64 << 20)))


@pytest.mark.parametrize("q_len", [2, 8, 16])
@pytest.mark.parametrize("lens,promise,width", [
    ([100] * 2, 100, 7), ([0, 1, 17, 190, 33], 190, 12), ([400] * 40, 400, 25),
    ([31 * (i % 16) for i in range(130)], 465, 32), ([90, 5, 0, 64] * 64, 90, 6),
    # Longer than promised: the last split runs on to the sequence's end.
    ([700, 90, 3000, 16, 0, 1], 128, 200),
    # A table whose rows hold more than a split may: not cut, the promise broken too.
    ([700, 90, 3000, 16, 0, 1], 128, 2300),
    ([700, 90, 300, 16, 0, 1], 0, 44),  # no promise: the table's width
])
def test_short_sequences_are_cut_at_their_starts(q_len, lens, promise, width):
    case = inputs.Case(batch=len(lens), q_len=q_len, seq_lens=lens, seed=2400 + q_len)
    q, k, v, bt, sl = inputs.make_inputs(case)
    wide = torch.zeros(len(lens), width, dtype=torch.int32)
    wide[:, :bt.shape[1]] = bt
    ref = attention_c64(q, k, v, bt, sl, 16, 8)
    dev = tuple(t.cuda() for t in (q, k, v, wide, sl))
    for given in {promise, 0}:
        out = sqa.paged_mtp_attention(*dev, 16, given)
        assert_parity(out, ref, label=f"q{q_len} B{len(lens)} promise {given}")
        assert torch.equal(out, sqa.paged_mtp_attention(*dev, 16, given))


@pytest.mark.parametrize("q_len", [2, 8])
@pytest.mark.parametrize("lens,width", [
    ([1500] * 8, 200),                                 # too wide a table for the cut
    ([1500, 90, 700, 1499, 0, 33, 1200, 1500], 200),
    ([700] * 5, 300), ([1100] * 5, 300),               # splits of 12 pages
    ([100] * 64, 7), ([100] * 64, 9), ([400] * 40, 60),
    ([500] * 8, 2000), ([1000] * 4, 1500), ([16, 90, 250] * 10, 2000),  # short items
])
def test_a_promised_length_does_not_change_the_bits(q_len, lens, width):
    """The cut of short sequences looks at the table's width, the same whatever length is
    promised, and at no more of the workspace than the plan asks for."""
    case = inputs.Case(batch=len(lens), q_len=q_len, seq_lens=lens, seed=2600 + q_len)
    q, k, v, bt, sl = inputs.make_inputs(case)
    wide = torch.zeros(len(lens), width, dtype=torch.int32)
    wide[:, :bt.shape[1]] = bt
    dev = tuple(t.cuda() for t in (q, k, v, wide, sl))
    plain = sqa.paged_mtp_attention(*dev, 16, 0)
    assert_parity(plain, attention_c64(q, k, v, bt, sl, 16, 8), label=f"q{q_len} width {width}")
    for promise in (max(lens), max(lens) + 16, (max(lens) + width * 16) // 2, width * 16):
        assert torch.equal(sqa.paged_mtp_attention(*dev, 16, promise), plain), promise
        ns, pps = _lib.plan_splits(0, len(lens), q_len, 32, 8, 128, promise, width, 0)
        own = _lib.workspace_bytes(len(lens), q_len, 32, 8, 128, ns, pps)
        assert torch.equal(_call(dev, ns, pps, own + (64 << 20)), plain), promise


@pytest.mark.parametrize("lens,width,cut", [
    ([1500] * 8, 94, True), ([1500] * 8, 200, False),  # splits of 6 pages; 14 would be needed
    ([1100] * 5, 300, True), ([1100] * 5, 301, False),  # of 12; 14
    ([300] * 40, 24, True), ([300] * 40, 60, False),   # of 8; 20
])
def test_which_batches_are_cut_at_their_starts(lens, width, cut):
    """A balanced plan leaves its (first slot, count) table in the workspace; one that is
    cut runs as a fixed plan and leaves that part alone. 256 compute units (two head
    groups of the 8 kv heads share them)."""
    if _lib.load().sqa_device_cu_count(0) != 256:
        pytest.skip("the widths are those of 256 compute units")
    q, k, v, bt, sl = inputs.make_inputs(
        inputs.Case(batch=len(lens), q_len=2, seq_lens=lens, seed=2700))
    wide = torch.zeros(len(lens), width, dtype=torch.int32)
    wide[:, :bt.shape[1]] = bt
    dev = tuple(t.cuda() for t in (q, k, v, wide, sl))
    ns, pps = _lib.plan_splits(0, len(lens), 2, 32, 8, 128, max(lens), width, 0)
    assert pps < 0
    nbytes = _lib.workspace_bytes(len(lens), 2, 32, 8, 128, ns, pps)
    ws = torch.full((nbytes // 4,), float("nan"), device="cuda")
    out = torch.empty_like(dev[0])
    _lib.launch(*dev, out, ws, ns, pps, torch.cuda.current_stream().cuda_stream)
    table = ws[ns * 8 * 8 * (128 + 2):][:2 * len(lens)]
    assert torch.isnan(table).all().item() == cut
    assert torch.isnan(table).any().item() == cut
    assert_parity(out, attention_c64(q, k, v, bt, sl, 16, 8), label=f"width {width}")


def test_a_chunked_plan_over_a_table_past_two_to_the_31_entries():
    """Three rows of 2**30 pages each (12 GiB, of which a few pages are written): the third
    row starts at entry 2**31."""
    width = 1 << 30
    free, _ = torch.cuda.mem_get_info()
    if free < 20 << 30:
        pytest.skip("needs 20 GiB of device memory")
    lens = [700, 90, 660]
    q, k, v, bt, sl = inputs.make_inputs(
        inputs.Case(batch=3, q_len=4, seq_lens=lens, seed=2800))
    table = torch.empty(3, width, dtype=torch.int32, device="cuda")
    table[:, :64].zero_()
    table[:, :bt.shape[1]] = bt.cuda()
    dev = (q.cuda(), k.cuda(), v.cuda(), table, sl.cuda())
    own = _lib.workspace_bytes(3, 4, 32, 8, 128, 6, 8)
    out = _call(dev, 6, 8, own + (64 << 20))
    del dev, table
    torch.cuda.empty_cache()
    assert_parity(out, attention_c64(q, k, v, bt, sl, 16, 8), label="wide table")
