"""Merge kernel with several output rows per wave (many rows of few splits): rows of
no split, one, two and many more than the launch expects, row counts that are no
multiple of a workgroup's, fp16 and fp32 partials at every head dim, against the
float64 oracle."""

import sys

import pytest
import torch

from oracle import attention_c64
from small_q_attention_amd import cuda as sqa, inputs
from tests._helpers import assert_parity

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _announce(request):
    sys.__stderr__.write(f"\n[gpu-test] {request.node.nodeid}\n")
    sys.__stderr__.flush()


@pytest.mark.parametrize("d,hq,hkv,q_len,qdt,batch", [
    (128, 32, 8, 16, torch.float16, 67),   # 34304 rows, 16 threads each
    (128, 12, 3, 8, torch.float16, 131),   # 12576 rows
    (128, 32, 8, 4, torch.bfloat16, 65),   # fp32 partials: 32 threads per row
    (64, 32, 8, 8, torch.float16, 67),     # 8 threads per row
    (64, 32, 8, 8, torch.bfloat16, 67),
    (256, 16, 4, 8, torch.float16, 67),    # 32 threads per row
    (256, 16, 4, 4, torch.bfloat16, 67),   # 64: a wave per row again
])
@pytest.mark.parametrize("longest", [700, 9000])
def test_rows_of_few_splits_share_a_wave(d, hq, hkv, q_len, qdt, batch, longest):
    lens = [(37 * i) % 90 for i in range(batch)]
    lens[batch // 2], lens[-1] = longest, 650
    case = inputs.Case(batch=batch, q_len=q_len, seq_lens=lens, seed=2500 + d + q_len,
                       num_query_heads=hq, num_kv_heads=hkv, head_dim=d)
    q, k, v, bt, sl = inputs.make_inputs(case)
    q, k, v = (t.to(qdt) for t in (q, k, v))
    out = sqa.paged_mtp_attention(*(t.cuda() for t in (q, k, v, bt, sl)), 16, longest)
    assert_parity(out, attention_c64(q, k, v, bt, sl, 16, hkv),
                  label=f"d{d} hq{hq} q{q_len} {qdt} B{batch} longest {longest}")
