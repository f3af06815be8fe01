"""Calls with a chunk size run the automatic cut of the same pages where their
workspace holds it: against the float64 oracle, and against the plan run as given
(a workspace of that plan's own size, or none), at lengths where the two differ in
splits, items and pieces."""

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
    [0, 5, 511, 513, 2050], [640] * 3, [300] * 130,  # balanced cuts, ragged, uniform, many
])
def test_chunked_plans_are_cut_like_the_automatic_one(q_len, chunk, lens):
    case = inputs.Case(batch=len(lens), q_len=q_len, seq_lens=lens, seed=2100 + q_len)
    host = inputs.make_inputs(case)
    tensors = tuple(t.cuda() for t in host)
    q, k, v, bt, sl = tensors
    ref = attention_c64(*host, 16, 8)
    label = f"q{q_len} ck{chunk} B{len(lens)}"
    assert_parity(sqa.paged_mtp_attention(*tensors, 16, max(lens), chunk_keys=chunk), ref,
                  label=label)
    b = len(lens)
    ns, pps = _lib.plan_splits(0, b, q_len, 32, 8, 128, max(lens), bt.shape[1], chunk)
    own = _lib.workspace_bytes(b, q_len, 32, 8, 128, ns, pps)
    more = _lib.call_workspace_bytes(0, b, q_len, 32, 8, 128, ns, pps, bt.shape[1])
    assert more >= own
    for nbytes in {own, more}:
        assert_parity(_call(tensors, ns, pps, nbytes), ref, label=f"{label} {nbytes} bytes")


@pytest.mark.parametrize("batch", [1, 3])
@pytest.mark.parametrize("splits,pps", [(1, 20), (5, 4), (40, 1)])
def test_a_recut_plan_reads_the_pages_of_the_plan_as_given(batch, splits, pps):
    """A plan covers the first num_splits * pages_per_split pages of every sequence
    and no more, however it is cut: longer sequences see only those keys."""
    lens = [1000] * batch
    q, k, v, bt, sl = (t.cuda() for t in inputs.make_inputs(
        inputs.Case(batch=batch, q_len=4, seq_lens=lens, seed=2200)))
    pages = splits * pps
    own = _lib.workspace_bytes(batch, 4, 32, 8, 128, splits, pps)
    as_given = _call((q, k, v, bt, sl), splits, pps, own)
    recut = _call((q, k, v, bt, sl), splits, pps, 64 << 20)
    # The draft lies behind them: every row sees all of their keys, as a lone
    # query at the end of a sequence of that length would.
    short = torch.full((batch,), pages * 16, dtype=torch.int32)
    want = attention_c64(q.cpu()[:, :1].contiguous(), k.cpu(), v.cpu(), bt.cpu(), short, 16, 8)
    for out, label in ((as_given, "as given"), (recut, "re-cut")):
        assert_parity(out[:, :1].contiguous(), want, label=label)
    assert (as_given.float() - recut.float()).abs().max().item() <= 2e-3


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
