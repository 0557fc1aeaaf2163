"""The attention entry points against the oracle's in-order composition, bit
for bit, where the split over positions, heads and dimensions can go wrong:
blocks of 64 positions, chunks of 64 and 128 positions and the 32 that the last
one ends with, the pieces of the exact sum (2560, 3072 and 6144 terms on
workgroups of 320, 384 and 768 threads), both sides of the fused logits, ragged
batches, a position beyond a sequence's slice and the values that softmax
ignores."""
import numpy as np
import pytest

import helpers as H
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def bits_equal(a, b):
    a, b = (np.ascontiguousarray(x, np.float32).reshape(-1) for x in (a, b))
    return a.shape == b.shape and np.array_equal(a.view(np.uint32), b.view(np.uint32))


def run_one(gpu, q, kc, vc, n_head, n_head_kv, hd, n_kv, max_kv=None):
    """llamd_fwd_attention (max_kv None) or _meta, of one sequence."""
    L = gpu.lib()
    Q, K, V = (gpu.DeviceBuffer.from_array(a) for a in (q, kc, vc))
    out = gpu.DeviceBuffer(q.nbytes)
    if max_kv is None:
        L.llamd_fwd_attention(Q.ptr, K.ptr, V.ptr, out.ptr, None, n_head, n_head_kv, hd, n_kv)
    else:
        meta = gpu.DeviceBuffer.from_array(np.array([0, n_kv - 1], np.int32))
        L.llamd_fwd_attention_meta(Q.ptr, K.ptr, V.ptr, out.ptr, None, n_head, n_head_kv, hd, meta.ptr, max_kv)
    assert L.llamd_fwd_sync() == 0 and L.llamd_fwd_last_error() == 0
    return out.download(np.empty(q.size, np.float32))


@pytest.mark.parametrize("n_head,n_head_kv,hd,lengths", [
    (32, 4, 128, (1, 8, 9, 20, 31, 33, 55, 56, 57, 64, 65, 96, 97, 129, 160, 161, 256, 257, 352, 1000, 4100)),
    (8, 1, 128, (6144, 6145, 6657, 8193, 16384)),
    (12, 12, 64, (1, 63, 64, 97, 129, 300, 2051)),
    (16, 1, 64, (65, 700)),
    (4, 2, 32, (40, 300)), (34, 2, 128, (130,))])   # these two on the general kernel
def test_attention_bit_exact(gpu, n_head, n_head_kv, hd, lengths):
    kv_dim, top = n_head_kv * hd, max(lengths)
    q = (H.sample(n_head * hd, 81) * 3).astype(np.float32)
    kc = H.sample(top * kv_dim, 82).reshape(top, kv_dim)
    vc = H.sample(top * kv_dim, 83).reshape(top, kv_dim)
    for n_kv in lengths:
        want = O.attend(q, kc[:n_kv], vc[:n_kv], n_kv, n_head, n_head_kv, hd)
        assert bits_equal(run_one(gpu, q, kc, vc, n_head, n_head_kv, hd, n_kv), want), n_kv
        # the position on the device, whatever max_kv says of this one cache
        for max_kv in (top, 0 if n_kv < 300 else 64):
            got = run_one(gpu, q, kc, vc, n_head, n_head_kv, hd, n_kv, max_kv)
            assert bits_equal(got, want), (n_kv, max_kv)


@pytest.mark.parametrize("nseq,n_head,n_head_kv,hd,max_kv", [
    (3, 32, 4, 128, 300), (13, 32, 4, 128, 200), (16, 12, 12, 64, 160), (2, 8, 8, 128, 700),
    (13, 32, 4, 128, 500), (16, 12, 12, 64, 420), (7, 32, 4, 128, 700)])
def test_batched_attention_ragged_bit_exact(gpu, nseq, n_head, n_head_kv, hd, max_kv):
    kv_dim = n_head_kv * hd
    q = (H.sample(nseq * n_head * hd, 84) * 3).astype(np.float32).reshape(nseq, -1)
    kc = H.sample(nseq * max_kv * kv_dim, 85).reshape(nseq, max_kv, kv_dim)
    vc = H.sample(nseq * max_kv * kv_dim, 86).reshape(nseq, max_kv, kv_dim)
    lengths = [(max_kv * (s + 1) // nseq) for s in range(nseq)]
    lengths[0] = 1
    check_batch(gpu, q, kc, vc, n_head, n_head_kv, hd, lengths)


@pytest.mark.parametrize("max_kv,lengths", [(2600, (1, 63, 65, 2560, 2561)), (3400, (31, 33, 95, 129, 3072, 3073))])
def test_batched_attention_sum_pieces(gpu, max_kv, lengths):
    """129..256 heads: on 64 dimensions each where a CU's LDS holds two
    workgroups (up to 3300 positions), else on all 128."""
    n_head, n_head_kv, hd, nseq = 32, 4, 128, len(lengths)
    kv_dim = n_head_kv * hd
    q = (H.sample(nseq * n_head * hd, 84) * 3).astype(np.float32).reshape(nseq, -1)
    kc = H.sample(nseq * max_kv * kv_dim, 85).reshape(nseq, max_kv, kv_dim)
    vc = H.sample(nseq * max_kv * kv_dim, 86).reshape(nseq, max_kv, kv_dim)
    check_batch(gpu, q, kc, vc, n_head, n_head_kv, hd, lengths)


def check_batch(gpu, q, kc, vc, n_head, n_head_kv, hd, lengths):
    nseq, max_kv = kc.shape[:2]
    meta = np.array([[7, n - 1] for n in lengths], np.int32)
    L = gpu.lib()
    Q, K, V, M = (gpu.DeviceBuffer.from_array(a) for a in (q, kc, vc, meta))
    out = gpu.DeviceBuffer(q.nbytes)
    L.llamd_b_attention(Q.ptr, K.ptr, V.ptr, out.ptr, None, n_head, n_head_kv, hd, max_kv, M.ptr, nseq)
    assert L.llamd_fwd_sync() == 0 and L.llamd_fwd_last_error() == 0
    got = out.download(np.empty_like(q))
    for s, n in enumerate(lengths):
        assert bits_equal(got[s], O.attend(q[s], kc[s, :n], vc[s, :n], n, n_head, n_head_kv, hd)), (s, n)


@pytest.mark.parametrize("n_head,n_head_kv,hd,max_kv", [
    (32, 4, 128, 70), (32, 4, 128, 300), (16, 8, 128, 300), (12, 12, 64, 80), (16, 1, 64, 400)])
def test_batched_attention_of_few_positions(gpu, n_head, n_head_kv, hd, max_kv):
    """Sequences of up to 56 positions, which one wave takes with V rows 8 at a
    time, beside longer ones, whose blocks of logits are shared out over (kv
    head, sequence) pairs."""
    lengths = (1, 2, 7, 8, 9, 31, 32, 33, 40, 48, 55, 56, 57, 64, 65, max_kv)
    kv_dim = n_head_kv * hd
    q = (H.sample(len(lengths) * n_head * hd, 103) * 3).astype(np.float32).reshape(len(lengths), -1)
    kc = H.sample(len(lengths) * max_kv * kv_dim, 104).reshape(len(lengths), max_kv, kv_dim)
    vc = H.sample(len(lengths) * max_kv * kv_dim, 105).reshape(len(lengths), max_kv, kv_dim)
    check_batch(gpu, q, kc, vc, n_head, n_head_kv, hd, lengths)


def test_batched_attention_more_sequences_than_a_grid_dimension(gpu):
    """66000 sequences of one position: the output is the V row."""
    nseq, hd = 66000, 64
    q = H.sample(nseq * hd, 101).reshape(nseq, hd)
    v = H.sample(nseq * hd, 102).reshape(nseq, hd)
    L = gpu.lib()
    Q, V = (gpu.DeviceBuffer.from_array(a) for a in (q, v))
    M = gpu.DeviceBuffer.from_array(np.zeros((nseq, 2), np.int32))
    out = gpu.DeviceBuffer(q.nbytes)
    L.llamd_b_attention(Q.ptr, V.ptr, V.ptr, out.ptr, None, 1, 1, hd, 1, M.ptr, nseq)
    assert L.llamd_fwd_sync() == 0 and L.llamd_fwd_last_error() == 0
    assert np.array_equal(out.download(np.empty_like(q)), v)


def test_batched_attention_past_its_slice(gpu):
    """A sequence whose position lies past max_kv is attended to over the rows
    that follow its slice's start, as before; one out of range gives NaN."""
    n_head, n_head_kv, hd, max_kv = 8, 2, 128, 96
    kv_dim = n_head_kv * hd
    q = H.sample(3 * n_head * hd, 87).reshape(3, -1)
    kc = H.sample(3 * max_kv * kv_dim, 88).reshape(3 * max_kv, kv_dim)
    vc = H.sample(3 * max_kv * kv_dim, 89).reshape(3 * max_kv, kv_dim)
    meta = np.array([[0, 249], [0, 40000], [0, -1]], np.int32)
    L = gpu.lib()
    Q, K, V, M = (gpu.DeviceBuffer.from_array(a) for a in (q, kc, vc, meta))
    out = gpu.DeviceBuffer(q.nbytes)
    L.llamd_b_attention(Q.ptr, K.ptr, V.ptr, out.ptr, None, n_head, n_head_kv, hd, max_kv, M.ptr, 3)
    assert L.llamd_fwd_sync() == 0 and L.llamd_fwd_last_error() == 0
    got = out.download(np.empty_like(q))
    assert bits_equal(got[0], O.attend(q[0], kc[:250], vc[:250], 250, n_head, n_head_kv, hd))
    assert np.isnan(got[1:]).all()


def test_short_caches_take_no_device_memory(gpu):
    """4096 sequences of one position in slices of 256: the launch forms the
    logits itself, so none of the 256 MiB that they would fill is allocated.
    One position: the output is its V row."""
    nseq, n_head, n_head_kv, hd, max_kv = 4096, 16, 1, 64, 256
    q = H.sample(nseq * n_head * hd, 99).reshape(nseq, n_head, hd)
    v = H.sample(nseq * max_kv * hd, 100).reshape(nseq, max_kv, hd)
    L = gpu.lib()
    Q, K, V = (gpu.DeviceBuffer.from_array(a) for a in (q, v, v))
    M = gpu.DeviceBuffer.from_array(np.zeros((nseq, 2), np.int32))
    out = gpu.DeviceBuffer(q.nbytes)
    assert L.llamd_fwd_sync() == 0
    free = L.llamd_rocm_free_mem()
    L.llamd_b_attention(Q.ptr, K.ptr, V.ptr, out.ptr, None, n_head, n_head_kv, hd, max_kv, M.ptr, nseq)
    assert L.llamd_fwd_sync() == 0 and L.llamd_fwd_last_error() == 0
    assert free - L.llamd_rocm_free_mem() < 64 << 20
    got = out.download(np.empty_like(q))
    assert np.array_equal(got, np.broadcast_to(v[:, :1], got.shape))


@pytest.mark.parametrize("n_kv", [1, 40, 64, 130, 400])
def test_attention_over_its_own_input(gpu, n_kv):
    """out over q, one sequence and two: the bits of a call with a buffer of its own."""
    n_head, n_head_kv, hd, max_kv = 32, 4, 128, 512
    kv_dim = n_head_kv * hd
    q = (H.sample(2 * n_head * hd, 96) * 3).astype(np.float32).reshape(2, -1)
    kc = H.sample(2 * max_kv * kv_dim, 97).reshape(2, max_kv, kv_dim)
    vc = H.sample(2 * max_kv * kv_dim, 98).reshape(2, max_kv, kv_dim)
    L = gpu.lib()
    K, V = gpu.DeviceBuffer.from_array(kc), gpu.DeviceBuffer.from_array(vc)
    M = gpu.DeviceBuffer.from_array(np.array([[0, n_kv - 1]] * 2, np.int32))
    want = [O.attend(q[s], kc[s, :n_kv], vc[s, :n_kv], n_kv, n_head, n_head_kv, hd) for s in range(2)]
    for call in ("fixed", "meta", "batch"):
        Q = gpu.DeviceBuffer.from_array(q)
        if call == "fixed":
            L.llamd_fwd_attention(Q.ptr, K.ptr, V.ptr, Q.ptr, None, n_head, n_head_kv, hd, n_kv)
        elif call == "meta":
            L.llamd_fwd_attention_meta(Q.ptr, K.ptr, V.ptr, Q.ptr, None, n_head, n_head_kv, hd, M.ptr, max_kv)
        else:
            L.llamd_b_attention(Q.ptr, K.ptr, V.ptr, Q.ptr, None, n_head, n_head_kv, hd, max_kv, M.ptr, 2)
        assert L.llamd_fwd_sync() == 0 and L.llamd_fwd_last_error() == 0
        got = Q.download(np.empty_like(q))
        assert bits_equal(got[0], want[0]), call
        assert bits_equal(got[1], want[1] if call == "batch" else q[1]), call


@pytest.mark.parametrize("n_kv", [50, 400])
def test_attention_non_finite_and_lowest_logits(gpu, n_kv):
    """Keys that make a logit -inf, NaN or hugely negative, and a V row of
    infinities right after the last position, which no sum may see."""
    n_head, n_head_kv, hd = 4, 2, 128
    kv_dim = n_head_kv * hd
    q = np.abs(H.sample(n_head * hd, 90)) + np.float32(0.1)
    kc = H.sample((n_kv + 1) * kv_dim, 91).reshape(n_kv + 1, kv_dim)
    vc = H.sample((n_kv + 1) * kv_dim, 92).reshape(n_kv + 1, kv_dim)
    vc[n_kv] = np.inf
    for case in ("lowest", "inf", "nan"):
        k = kc.copy()
        k[3] = {"lowest": -3e37, "inf": -np.inf, "nan": np.nan}[case]
        want = O.attend(q, k[:n_kv], vc[:n_kv], n_kv, n_head, n_head_kv, hd)
        got = run_one(gpu, q, k, vc, n_head, n_head_kv, hd, n_kv)
        if case == "nan":  # NaN payloads are not part of the contract
            assert np.isnan(got).all() and np.isnan(want).all()
        else:
            assert bits_equal(got, want), case


def test_attention_in_a_captured_graph(gpu):
    """Captured with a first use of the scratch inside the capture, replayed at
    other positions with other work between: the eager results every time."""
    n_head, n_head_kv, hd, max_kv = 8, 2, 128, 640
    kv_dim = n_head_kv * hd
    q = H.sample(n_head * hd, 93)
    kc = H.sample(max_kv * kv_dim, 94).reshape(max_kv, kv_dim)
    vc = H.sample(max_kv * kv_dim, 95).reshape(max_kv, kv_dim)
    L = gpu.lib()
    assert L.llamd_fwd_stream_init() == 0
    Q, K, V = (gpu.DeviceBuffer.from_array(a) for a in (q, kc, vc))
    out, M = gpu.DeviceBuffer(q.nbytes), gpu.DeviceBuffer(8)
    assert L.llamd_fwd_begin_capture() == 0
    L.llamd_fwd_attention_meta(Q.ptr, K.ptr, V.ptr, out.ptr, None, n_head, n_head_kv, hd, M.ptr, max_kv)
    assert L.llamd_fwd_end_capture() == 0
    for n_kv in (10, 640, 257, 64):
        M.upload(np.array([0, n_kv - 1], np.int32))
        assert L.llamd_fwd_graph_launch() == 0
        assert L.llamd_fwd_sync() == 0
        got = out.download(np.empty(q.size, np.float32))
        want = O.attend(q, kc[:n_kv], vc[:n_kv], n_kv, n_head, n_head_kv, hd)
        assert bits_equal(got, want), n_kv
        assert bits_equal(run_one(gpu, q, kc, vc, n_head, n_head_kv, hd, 300),
                          O.attend(q, kc[:300], vc[:300], 300, n_head, n_head_kv, hd))
    L.llamd_fwd_graph_destroy()
