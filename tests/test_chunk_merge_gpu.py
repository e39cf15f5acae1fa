"""The merge of a chunk's splits has a kernel path for each number of them up to four and one for more; heads of whole
16-byte units and others: contexts against the oracle."""
import os

import numpy as np
import pytest
import torch

import oracle
import saragossa_amd as skv

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[2, 3, 4, 5, 9])
def splits(request):
    env = {"SKV_PREFILL_TILES": "2", "SKV_PREFILL_WGS": "1000000", "SKV_DECODE_WGS": "1000000", "SKV_PREFILL_MAX_SPLITS": str(request.param)}
    saved = {k: os.environ.get(k) for k in env}
    os.environ.update(env)
    skv.flags.reload()
    yield request.param
    for k, v in saved.items():
        if v is None:
            os.environ.pop(k, None)
        else:
            os.environ[k] = v
    skv.flags.reload()


@pytest.mark.parametrize("element,tol", [("bf16", 1e-4), ("f32", 2e-5)])
@pytest.mark.parametrize("head_dim", [64, 42])
def test_splits_of_a_chunk_are_merged(state, splits, head_dim, element, tol):
    q_heads, kv_heads, base, rows = 4, 2, 2400, 37
    rng = np.random.default_rng(splits * head_dim)
    make = state.full_attention_f32 if element == "f32" else state.full_attention_bf16
    kv = make(base + rows, q_heads, kv_heads, head_dim)
    kv.set_block_table(rng.permutation(kv.pages()).astype(np.int32))
    k, v = (rng.standard_normal((base + rows, kv_heads * head_dim), dtype=np.float32) for _ in range(2))
    q = rng.standard_normal((rows, q_heads * head_dim), dtype=np.float32)
    kv.seed(k[:base], v[:base], base)
    qd, kd, vd = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (q, k[base:], v[base:]))
    out = torch.full((rows, q_heads * head_dim), float("nan"), device="cuda")
    kv.encode_prefill_rows(torch.cuda.current_stream().cuda_stream, qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), rows, out.data_ptr())
    cache = oracle.LayerKvCache("f32" if element == "f32" else "bf16r")
    lay = oracle.layout(q_heads, kv_heads, head_dim)
    cache.append_batch(k[:base], v[:base], lay)
    want = np.stack([oracle.decode_step(cache, k[base + i], v[base + i], q[i], lay) for i in range(rows)])
    assert np.abs(out.cpu().numpy() - want).max() <= tol
