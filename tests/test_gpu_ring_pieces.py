"""Work items whose page ring runs through the ends of sequences: pieces shorter
than, as long as and longer than the ring (8, 4 and 2 pages at head dim 64, 128 and
256), more page ids than one pass of a workgroup loads, Q fragments in two LDS
buffers or in registers, each piece with its own draft tree, against the float64
oracle."""

import sys

import pytest
import torch

from oracle import attention_c64
from small_q_attention_amd import _lib, inputs
from small_q_attention_amd.masks import as_words, pack_draft_mask
from tests._helpers import assert_parity

pytestmark = pytest.mark.gpu

F8 = torch.float8_e4m3fn
SHORT = [1, 15, 16, 17, 33, 64, 65, 0, 127, 128, 129, 144, 2, 200, 48, 31]
LONG = [4500, 16, 1, 3000, 70, 2049, 33]  # about 600 pages: ids in three passes


@pytest.fixture(autouse=True)
def _announce(request):
    sys.__stderr__.write(f"\n[gpu-test] {request.node.nodeid}\n")
    sys.__stderr__.flush()


@pytest.mark.parametrize("lens", [SHORT, LONG], ids=["short", "long"])
@pytest.mark.parametrize("d,hq,hkv,q_len,qdt,fp8", [
    (64, 32, 8, 2, torch.float16, False),    # two heads in one block
    (64, 32, 8, 8, torch.bfloat16, True),    # two heads, two blocks each
    (64, 8, 2, 16, torch.float16, False),    # one head, four blocks
    (128, 8, 2, 4, torch.float16, False),    # one head group, idle waves
    (128, 32, 8, 8, torch.bfloat16, False),  # two blocks
    (128, 32, 8, 16, torch.float16, True),   # page pairs, Q in registers
    (128, 32, 8, 16, torch.bfloat16, True),  # Q in registers
    (256, 16, 4, 8, torch.float16, False),   # a ring of two pages
    (256, 16, 4, 4, torch.float16, True),
])
def test_the_ring_runs_through_sequence_ends(lens, d, hq, hkv, q_len, qdt, fp8):
    case = inputs.Case(batch=len(lens), q_len=q_len, seq_lens=lens, seed=2300 + d + q_len,
                       num_query_heads=hq, num_kv_heads=hkv, head_dim=d)
    q, k, v, bt, sl = inputs.make_inputs(case)
    q = q.to(qdt)
    k, v = (t.to(F8 if fp8 else qdt) for t in (k, v))
    g = torch.Generator().manual_seed(2300)
    vis = torch.rand(len(lens), q_len, q_len, generator=g) < 0.5
    vis[:, torch.arange(q_len), torch.arange(q_len)] = True
    mask = pack_draft_mask(vis)
    words = as_words(mask, len(lens), q_len).cuda()
    dev = [t.cuda() for t in (q, k, v, bt, sl)]
    for draft, packed in ((None, None), (words, mask)):
        ref = attention_c64(q, k, v, bt, sl, 16, hkv, draft_mask=packed)
        for n_items in (1, 2, 5):
            ns = len(lens) + n_items
            nbytes = _lib.workspace_bytes(len(lens), q_len, hq, hkv, d, ns, 0)
            ws = torch.full((nbytes // 4,), float("nan"), dtype=torch.float32, device="cuda")
            out = torch.full_like(dev[0], float("nan"))
            _lib.launch_general(dev[0], out, dev[1], dev[2], dev[3], dev[4], draft, d ** -0.5,
                                1.0, ns, 0, ws, torch.cuda.current_stream().cuda_stream)
            torch.cuda.synchronize()
            assert_parity(out, ref, label=f"d{d} q{q_len} fp8={fp8} items {n_items} "
                                          f"tree={draft is not None}")
