"""The grouped GEMMs at the edges of their work items: experts of 0, 1, 2, 3,
15..17, 32, 33 and 128..145 tokens (16-token chunks, twins, wide units of up to
8 chunks, an expert split over several), rows that end inside a group of tiles,
and prompts past the sort's register batches."""
import numpy as np
import pytest

import helpers as H
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def layer(gpu, n_embd, n_ff, n_expert, n_used, seed):
    from llamd_rs_amd import synth
    router = synth.normal(seed, 0.02, n_expert * n_embd).reshape(n_expert, n_embd)
    w = [synth.q6k_matrix(seed + i, 0.05, n_expert * r, k)
         for i, (r, k) in enumerate([(n_ff, n_embd), (n_ff, n_embd), (n_embd, n_ff)], 1)]
    return gpu.MoeLayer(router, *w, n_embd, n_ff, n_expert, n_used), w


def prefill(L, gpu, m, x, ids, w, flags):
    X, I, W = (gpu.DeviceBuffer.from_array(a) for a in (x, ids, w))
    out = gpu.DeviceBuffer(x.nbytes)
    assert L.llamd_hip_moe_prefill_ex(m.handle, X.ptr, I.ptr, W.ptr, out.ptr, len(x), flags) == 0
    assert L.llamd_fwd_sync() == 0
    return out.download(np.empty_like(x))


def by_chunks(L, gpu, m, x, ids, w, flags):
    """The same call with a 16-token chunk per wave."""
    prev = L.llamd_hip_tune(b"batched_twin", 0)
    try:
        return prefill(L, gpu, m, x, ids, w, flags)
    finally:
        L.llamd_hip_tune(b"batched_twin", prev)


EDGES = [0, 1, 2, 3, 15, 16, 17, 32, 33, 128, 129, 145]


@pytest.mark.parametrize("n_embd,n_ff,counts", [
    (768, 256, EDGES),                                         # twins
    (512, 256, EDGES + [255, 256, 257] + [0] * 113),           # REDUCTION: wide units of 2 chunks
    (512, 256, EDGES + [255, 256, 257] + [18] * 60 + [0] * 53)])  # of 8
def test_grouped_edges_of_chunks_twins_and_units(gpu, n_embd, n_ff, counts):
    """Exact rows equal the CPU's; REDUCTION rows differ from them by the f32
    rounding of nb terms and by quants of the SwiGLU output that it moves: one
    step of 1/127 of a block's largest value, on one of its 256 values."""
    n_expert = len(counts)
    m, (gate, up, down) = layer(gpu, n_embd, n_ff, n_expert, 1, 900)
    ids = np.repeat(np.arange(n_expert, dtype=np.int32), counts)[:, None]
    ids = ids[np.argsort(H.sample(len(ids), 5))]     # tokens of an expert scattered
    ids = np.concatenate([ids, [[-1], [n_expert]]]).astype(np.int32)  # two that add no term
    n = len(ids)
    x = (H.sample(n * n_embd, 6) * 2).astype(np.float32).reshape(n, n_embd)
    w = (H.sample(n, 7).reshape(n, 1) + np.float32(2)).astype(np.float32)
    L = gpu.lib()
    got = prefill(L, gpu, m, x, ids, w, 0)
    want = O.moe_ffn_tokens(x[:-2], n_embd, n_ff, n_expert, gate, up, down, ids[:-2].astype(np.uint32), w[:-2])
    assert np.array_equal(got[:-2].view(np.uint32), np.asarray(want, np.float32).reshape(-1, n_embd).view(np.uint32))
    assert not got[-2:].any()
    red = prefill(L, gpu, m, x, ids, w, 1)
    assert not red[-2:].any()
    rms = np.sqrt((got[:-2].astype(np.float64) ** 2).mean(1, keepdims=True))
    assert (np.abs(red[:-2] - got[:-2]) / rms).max() < 3e-2
    assert np.linalg.norm(red - got) / np.linalg.norm(got) < 1e-3
    assert np.array_equal(by_chunks(L, gpu, m, x, ids, w, 0).view(np.uint32), got.view(np.uint32))
    assert np.array_equal(by_chunks(L, gpu, m, x, ids, w, 1).view(np.uint32), red.view(np.uint32))


@pytest.mark.parametrize("counts", [(17, 1, 64, 2, 33, 3), (32, 31, 16, 49)])
def test_grouped_edges_of_mostly_empty_experts(gpu, counts):
    """Fewer than 8 pairs per expert, so exact rows take the kernel for groups of
    one and two tokens and REDUCTION rows the twins, with some experts of more
    than a chunk: exact rows equal the CPU's, REDUCTION rows are the same bits by
    twins and by chunks."""
    n_embd, n_ff, n_expert = 512, 256, 64
    m, (gate, up, down) = layer(gpu, n_embd, n_ff, n_expert, 1, 930)
    ids = np.repeat(3 * np.arange(len(counts), dtype=np.int32) + 1, counts)[:, None]
    ids = ids[np.argsort(H.sample(len(ids), 18))].copy()
    n = len(ids)
    x = (H.sample(n * n_embd, 19) * 2).astype(np.float32).reshape(n, n_embd)
    w = (H.sample(n, 20).reshape(n, 1) + np.float32(2)).astype(np.float32)
    L = gpu.lib()
    got = prefill(L, gpu, m, x, ids, w, 0)
    want = O.moe_ffn_tokens(x, n_embd, n_ff, n_expert, gate, up, down, ids.astype(np.uint32), w)
    assert np.array_equal(got.view(np.uint32), np.asarray(want, np.float32).reshape(-1, n_embd).view(np.uint32))
    red = prefill(L, gpu, m, x, ids, w, 1)
    assert np.linalg.norm(red - got) / np.linalg.norm(got) < 1e-3
    assert np.array_equal(by_chunks(L, gpu, m, x, ids, w, 1).view(np.uint32), red.view(np.uint32))


@pytest.mark.parametrize("n_tok,n_used,taken", [(256, 4, 4), (129, 8, 8), (330, 8, 8), (700, 8, 12), (150, 8, 100)])
def test_reduction_wide_units_of_few_experts(gpu, n_tok, n_used, taken):
    """`taken` of 128 experts take the prompt, so that wide units have up to 1,
    2, 4, 8 and 8 chunks: rows within the REDUCTION tolerance of the bit-exact
    ones, and the same bits with the tokens in another order."""
    n_embd, n_ff, n_expert = 512, 256, 128
    m, _ = layer(gpu, n_embd, n_ff, n_expert, n_used, 970)
    rng = np.random.default_rng(n_tok)
    names = rng.permutation(n_expert)[:taken]
    ids = np.stack([rng.permutation(names)[:n_used] for _ in range(n_tok)]).astype(np.int32)
    x = (H.sample(n_tok * n_embd, 16) * 2).astype(np.float32).reshape(n_tok, n_embd)
    w = (H.sample(n_tok * n_used, 17).reshape(n_tok, n_used) + np.float32(2)).astype(np.float32)
    L = gpu.lib()
    got = prefill(L, gpu, m, x, ids, w, 0)
    red = prefill(L, gpu, m, x, ids, w, 1)
    assert np.linalg.norm(red - got) / np.linalg.norm(got) < 1e-3
    assert np.array_equal(by_chunks(L, gpu, m, x, ids, w, 1).view(np.uint32), red.view(np.uint32))
    turn = rng.permutation(n_tok)
    again = prefill(L, gpu, m, x[turn].copy(), ids[turn].copy(), w[turn].copy(), 1)
    assert np.array_equal(again.view(np.uint32), red[turn].view(np.uint32))


@pytest.mark.parametrize("n_tok,n_used", [(1024, 8), (1025, 8), (3073, 8), (64, 2)])
def test_grouped_prompt_lengths(gpu, n_tok, n_used):
    """Past 8192 and 24576 pairs the sort takes its other routes: every token's
    row equals the row it gets in a call of 64 tokens, and those of the last 64
    are the CPU's."""
    n_embd, n_ff, n_expert = 256, 256, 16
    m, (gate, up, down) = layer(gpu, n_embd, n_ff, n_expert, n_used, 950)
    x = (H.sample(n_tok * n_embd, 8) * 2).astype(np.float32).reshape(n_tok, n_embd)
    score = H.sample(n_tok * n_expert, 9).reshape(n_tok, n_expert)
    ids = np.argsort(-score, axis=1)[:, :n_used].astype(np.int32)
    w = (H.sample(n_tok * n_used, 10).reshape(n_tok, n_used) + np.float32(2)).astype(np.float32)
    L = gpu.lib()
    whole = prefill(L, gpu, m, x, ids, w, 0)
    for a in list(range(0, n_tok - 64, max(64, n_tok // 6))) + [n_tok - 64]:
        s = slice(a, a + 64)
        part = prefill(L, gpu, m, x[s].copy(), ids[s].copy(), w[s].copy(), 0)
        assert np.array_equal(part.view(np.uint32), whole[s].view(np.uint32)), a
    want = O.moe_ffn_tokens(x[s], n_embd, n_ff, n_expert, gate, up, down, ids[s].astype(np.uint32), w[s])
    assert np.array_equal(part.view(np.uint32), np.asarray(want, np.float32).reshape(-1, n_embd).view(np.uint32))
    red = prefill(L, gpu, m, x, ids, w, 1)
    assert np.linalg.norm(red - whole) / np.linalg.norm(whole) < 1e-3


@pytest.mark.parametrize("rows,k,nseq", [(40, 256, 2), (8192, 768, 16), (8197, 512, 1 + 16), (8197, 1280, 16),
                                         (8256, 512, 16), (8256, 768, 33), (2112, 256, 64),
                                         (2072, 512, 81), (8216, 256, 40), (8232, 512, 33)])
def test_one_group_kernels(gpu, rows, k, nseq):
    """One group of tokens on few tiles (classes split over waves), on many
    (planes staged), with a last workgroup that is part empty, and on tiles and
    chunks that no workgroup can share: the CPU's bits."""
    from llamd_rs_amd import synth
    w = synth.q6k_matrix(77, 0.02, rows, k)
    dw = gpu.DeviceWeights.upload(w, rows, k // 256)
    xs = [synth.normal(30 + i, 1.0, k) for i in range(nseq)]
    acts = [O.quantize_q8_k(x) for x in xs]
    got = dw.matvec_batched([gpu.BlockQ8K(a.d, a.qs, a.bsums) for a in acts])
    for i in {0, nseq // 2, nseq - 1}:
        assert np.array_equal(np.asarray(got[i]).view(np.uint32),
                              np.asarray(O.matvec_q6k_act(w, rows, k, acts[i])).view(np.uint32)), i
