"""The prefill attention's launch variants against the oracle (the cases,
checks and tolerance of test_gpu_parity's _prefill_case)."""
import numpy as np
import pytest
import torch

from _ckpt import CKPT
from _gpu import assert_close_attn, cfg_of, graph_nodes, kv_rows, np_of
from _refs import BASELINE, Cfg
from qwfnfer_amd import qsa
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


# Queries that attend every block (a prompt's first thousands, a dense layer),
# taken a block of queries at a time: counts that leave a partial query block and
# tile, chunks from the first token and from inside a tile, one that ends past the
# last such query (the rest selects), both group counts a workgroup, each layout.
@pytest.mark.parametrize("cfg, pre, n_q", [
    (BASELINE, 0, 515), (BASELINE, 37, 1030), (BASELINE, 4000, 850), (BASELINE, 0, 1),
    (Cfg(top_k_blocks=0), 5001, 520),
    (Cfg(head_dim=64), 3, 600), (Cfg(head_dim=256), 64, 530), (Cfg(n_head=8), 10, 540), (Cfg(n_head=4), 10, 540),
    (Cfg(n_head=24, head_dim=256), 100, 520),
    (Cfg(kv_type=1), 5, 420), (Cfg(kv_type=2), 63, 400), (Cfg(kv_type=2, block_tokens=16, top_k_blocks=300), 1, 401),
    (CKPT, 129, 390),
])
def test_prefill_every_block(cfg, pre, n_q):
    _prefill_case(cfg, pre, n_q, seed=800 + n_q, dtype=np.float16 if n_q % 2 else np.float32)


# The same layouts at counts that take the shared pass when the selection is asked for
# too, and 16 queries more than one round of the per-query kernel.
@pytest.mark.parametrize("cfg, pre, n_q", [
    (Cfg(kv_type=1), 5, 1130), (Cfg(kv_type=2), 63, 1051), (Cfg(kv_type=2, block_tokens=16, top_k_blocks=300), 1, 1040),
    (CKPT, 129, 700), (BASELINE, 0, 528),
])
def test_prefill_every_block_longer(cfg, pre, n_q):
    _prefill_case(cfg, pre, n_q, seed=840 + n_q)


@pytest.mark.parametrize("cfg, pre, n_q, shared", [
    (Cfg(top_k_blocks=0), 900, 512, False), (Cfg(top_k_blocks=0), 900, 513, True),
    (Cfg(top_k_blocks=0, n_head=8), 900, 512, False), (Cfg(top_k_blocks=0, head_dim=256), 900, 512, True),
    (Cfg(top_k_blocks=0, kv_type=2), 8000, 500, False), (Cfg(top_k_blocks=0, kv_type=2), 8000, 600, True),
    (Cfg(top_k_blocks=0, kv_type=2), 0, 520, False), (Cfg(top_k_blocks=0, kv_type=2), 0, 1100, True),
    (Cfg(kv_type=2), 0, 400, True), (Cfg(kv_type=2), 3500, 400, False), (Cfg(kv_type=2), 3500, 700, True),
    (Cfg(top_k_blocks=0, kv_type=1), 0, 512, False), (Cfg(top_k_blocks=0, kv_type=1), 0, 1300, True),
    (Cfg(top_k_blocks=0, kv_type=1), 1500, 500, False), (Cfg(top_k_blocks=0, kv_type=1), 1500, 700, True),
])
def test_prefill_every_block_line(cfg, pre, n_q, shared):
    """Which calls share tiles: those measured faster so (they launch no indexer)."""
    print(f"line: {n_q} queries after {pre}", flush=True)
    c = cfg_of(cfg)
    dev = qsa.KvCache.allocate(c, 1, (pre + n_q) // cfg.page_tokens + 1)
    rows = torch.zeros((n_q, cfg.n_head_kv, cfg.head_dim), dtype=torch.float16, device="cuda")
    q, ws = torch.zeros((n_q, cfg.n_head, cfg.head_dim), device="cuda"), qsa.Workspace.for_prefill(c, pre + n_q, n_q)
    out = torch.empty_like(q)
    n = graph_nodes(lambda: qsa.sparse_attn_prefill(dev, q, 0, pre, ws, rows, rows, out=out))
    before = 2 if cfg.kv_type == 2 else 3            # the rows, the pooled keys, the V scales
    assert (n == before + 1) == shared and n >= before + 1


def _uneven_rows(rng, n, cfg):
    """kv_rows with keys that grow along the rows (a tile's largest logit passes the
    earlier ones for some queries and not for others) and another V scale every tile."""
    k, v = kv_rows(rng, n, cfg)
    k *= np.linspace(0.2, 2.0, n, dtype=np.float32)[:, None, None]
    v *= np.exp(rng.uniform(np.log(0.1), np.log(10.0), (n // 64 + 1, 1, 1))).astype(np.float32).repeat(64, 0)[:n]
    return k, v


# 64-dim heads, where two waves of a tile's conversion read the scales of one 32-dim
# block: from 512 queries (two KV heads), whole and partial query blocks and tiles.
@pytest.mark.parametrize("pre, n_q", [(0, 512), (3, 577), (61, 1030), (640, 513)])
def test_prefill_every_block_narrow_heads(pre, n_q):
    print(f"narrow heads: {n_q} queries after {pre}", flush=True)
    first = _prefill_case(Cfg(head_dim=64), pre, n_q, seed=820 + pre, kv=_uneven_rows)[0]
    again = _prefill_case(Cfg(head_dim=64), pre, n_q, seed=820 + pre, kv=_uneven_rows)[0]
    np.testing.assert_array_equal(first, again)


def _chunk(cfg, pre, n_q, seed, edit=None, sel=False, q_batch=None):
    """Output of a chunk over seeded rows (a row of the chunk's V changed by `edit`)."""
    c = cfg_of(cfg)
    rng = np.random.default_rng(seed)
    k, v = kv_rows(rng, pre + n_q, cfg)
    q = torch.from_numpy(rng.standard_normal((n_q, cfg.n_head, cfg.head_dim), dtype=np.float32)).cuda()
    if edit:
        edit(v)
    dev = qsa.KvCache.allocate(c, 1, (pre + n_q) // cfg.page_tokens + 1)
    kd, vd = torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda()
    if pre:
        qsa.append_q8_0(dev, kd[:pre], vd[:pre], torch.arange(pre, dtype=torch.int32, device="cuda"))
        qsa.pool_rebuild(dev, 0, pre // cfg.block_tokens)
    ws = qsa.Workspace.for_prefill(c, pre + n_q, q_batch or n_q)
    s = n = None
    if sel:
        s = torch.empty((n_q, cfg.n_head_kv, c.max_selected(pre + n_q)), dtype=torch.int32, device="cuda")
        n = torch.empty((n_q, cfg.n_head_kv), dtype=torch.int32, device="cuda")
    out = qsa.sparse_attn_prefill(dev, q, 0, pre, ws, kd[pre:].contiguous(), vd[pre:].contiguous(), sel=s, n_sel=n)
    torch.cuda.synchronize()
    return np_of(out)


def test_prefill_every_block_selection_and_batches_are_invisible():
    """The same bytes whether the selection is asked for or not, and whatever
    batch the workspace holds, over a chunk that ends past the last query that
    attends every block."""
    a = _chunk(BASELINE, 4000, 850, 90)
    np.testing.assert_array_equal(a, _chunk(BASELINE, 4000, 850, 90, sel=True))
    np.testing.assert_array_equal(a, _chunk(BASELINE, 4000, 850, 90, sel=True, q_batch=100))
    np.testing.assert_array_equal(a, _chunk(BASELINE, 4000, 850, 90, q_batch=100))


@pytest.mark.parametrize("kv_type", [0, 1, 2])
@pytest.mark.parametrize("bad", [300, 575, 511])
def test_prefill_every_block_non_finite_rows(kv_type, bad):
    """A non-finite V row reaches the queries at and after its position (the dims
    of its 32-value block, NaN or infinite) and no earlier one, wherever it lies in its
    tile and query block."""
    cfg = Cfg(kv_type=kv_type)
    n_q = 576

    def edit(v):
        v[bad, 1, 40] = np.inf                       # block 1 of KV head 1

    dims = slice(32, 64) if kv_type != 2 else slice(40, 41)   # a quantized block shares its scale

    def zero(v):                                     # the reference run: the key stays, those values are 0
        v[bad, 1, dims] = 0.0

    got, ref = _chunk(cfg, 0, n_q, 91, edit), _chunk(cfg, 0, n_q, 91, zero)
    G = cfg.n_head // cfg.n_head_kv
    assert not np.isfinite(got[bad:, G:, dims]).any()
    got[bad:, G:, dims], ref[bad:, G:, dims] = 0.0, 0.0
    assert_close_attn(got, ref.astype(np.float64))


@pytest.mark.parametrize("kv_type, unit", [(0, 1.0), (0, 1e-3), (0, 5e3), (1, 1.0), (1, 1e-3), (1, 5e3), (2, 1.0), (2, 1e-3)])
@pytest.mark.parametrize("n_q, bad", [(576, 300), (576, 575), (576, 511), (90, 511), (90, 575)])
def test_prefill_before_a_non_finite_row(kv_type, unit, n_q, bad):
    """The queries before a non-finite V row give the bytes of a cache where it holds
    zeros, in the kernel of a block of queries (576) and of one query (90): the largest V
    scale of a call, which sets the unit that the values (or weights) are split in, is
    the largest finite one.  Rows far below 1, and rows past fp16's largest value (at 5e3
    a quantized block's scale still fits)."""
    cfg = Cfg(kv_type=kv_type)
    pre = 576 - n_q
    dims = slice(32, 64) if kv_type != 2 else slice(40, 41)

    def edit(v):
        v *= unit
        v[bad, 1, 40] = np.inf

    def zero(v):
        v *= unit
        v[bad, 1, dims] = 0.0

    got, ref = _chunk(cfg, pre, n_q, 92, edit), _chunk(cfg, pre, n_q, 92, zero)
    np.testing.assert_array_equal(got[:bad - pre], ref[:bad - pre])
    G, at = cfg.n_head // cfg.n_head_kv, slice(bad - pre, None)
    assert not np.isfinite(got[at, G:, dims]).any()
    got[at, G:, dims], ref[at, G:, dims] = 0.0, 0.0
    assert_close_attn(got[at] / unit, ref[at].astype(np.float64) / unit)


def test_prefill_every_block_f16_precision():
    """F16: the shared pass is no further from 64 bits than the per-query kernel over the
    same rows (1,100 queries in one call and in calls of 100).  Both round a logit's sums
    over the high parts four times at its size; summing high and low parts in turn rounded
    it eight times, sqrt(2) the error; 1.2 lies between."""
    cfg = Cfg(kv_type=2)
    pre, n_q, G = 300, 1100, cfg.n_head // cfg.n_head_kv
    n = pre + n_q
    rng = np.random.default_rng(21)
    k, v = (torch.from_numpy(x).cuda().half() for x in kv_rows(rng, n, cfg))
    q = torch.from_numpy(rng.standard_normal((n_q, cfg.n_head, cfg.head_dim), dtype=np.float32)).cuda()
    c = cfg_of(cfg)
    dev = qsa.KvCache.allocate(c, 1, n // cfg.page_tokens + 1)
    qsa.append_q8_0(dev, k, v, torch.arange(n, dtype=torch.int32, device="cuda"))
    qsa.pool_rebuild(dev, 0, n // cfg.block_tokens)
    ws = qsa.Workspace.for_prefill(c, n, n_q)
    shared = qsa.sparse_attn_prefill(dev, q, 0, pre, ws)
    single = torch.cat([qsa.sparse_attn_prefill(dev, q[i:i + 100], 0, pre + i, ws) for i in range(0, n_q, 100)])
    seen = torch.arange(n, device="cuda") <= pre + torch.arange(n_q, device="cuda")[:, None]
    err = {"shared": 0.0, "single": 0.0}
    for h in range(cfg.n_head):
        s = q[:, h].double() @ k[:, h // G].double().T.contiguous() / cfg.head_dim ** 0.5
        ref = torch.softmax(s.masked_fill(~seen, -float("inf")), 1) @ v[:, h // G].double()
        for name, out in (("shared", shared), ("single", single)):
            err[name] += float(((out[:, h].double() - ref) ** 2).sum())
    print(f"squared errors {err}", flush=True)
    assert 0.0 < err["shared"] <= 1.2 ** 2 * err["single"]
