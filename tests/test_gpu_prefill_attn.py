"""The prefill attention's launch variants against the oracle (the cases,
checks and tolerance of test_gpu_parity's _prefill_case)."""
import pytest

from _refs import BASELINE, Cfg
from test_gpu_parity import _prefill_case

pytestmark = pytest.mark.gpu


# Calls of few queries, whose (query, KV head) pairs are each shared by several
# waves: one query (a workgroup's other pairs past the call), an odd count,
# counts on both sides of a change of the waves a pair, and selections of fewer
# tiles than waves (5 and 3 blocks: waves without a tile).
@pytest.mark.parametrize("cfg, pre, n_q", [
    (BASELINE, 5000, 1), (BASELINE, 5000, 3), (BASELINE, 5000, 129), (BASELINE, 5000, 257),
    (Cfg(top_k_blocks=2, local_tokens=64), 3000, 5), (Cfg(top_k_blocks=1, local_tokens=1), 900, 9),
    (Cfg(head_dim=64), 5000, 11),
])
def test_prefill_few_queries(cfg, pre, n_q):
    _prefill_case(cfg, pre, n_q, seed=700 + n_q)
