"""NaN and infinities in device-resident inputs of the kernels that share out keys or heads.

A special value reaches the rows and columns that read it and no others: key groups merge their
partial results, split backward workgroups add theirs, padded rows are stepped over. Everything not
reached is bitwise what it is without the special value, so these tests need no tolerance except
where a row loses a key (the oracle's).
"""
import numpy as np
import pytest

import oracle
from _inputs import bf16_round, normal
from conftest import assert_close

import flat_attention_amd as fa

pytestmark = pytest.mark.gpu

F32, BF16, F16 = fa.DTYPE_F32, fa.DTYPE_BF16, fa.DTYPE_F16
# heads, positions, head dim, query rows of a workgroup by (no mask, causal)
KERNELS = [(BF16, 8, 300, 64, (64, 64)),     # four key groups
           (F16, 8, 300, 128, (64, 64)),
           (BF16, 64, 500, 64, (128, 128)),  # two
           (F32, 8, 300, 64, (32, 32)),      # key groups of 32 rows
           (F32, 8, 300, 128, (32, 32)),
           (F32, 256, 300, 64, (128, 128))]  # the LDS-staged kernel


def _forward(hip, q, k, v, dims, dtype, causal):
    H, S, D = dims
    shape = fa.GroupedAttentionShape(1, H, H, S, D)
    ex = fa.HipRotaryGroupedAttention(hip, dtype)
    bufs = [fa.DeviceBuffer.from_array(hip, fa.host_storage(x.ravel(), dtype)) for x in (q, k, v)]
    res = ex.download_attention(
        ex.forward_resident(*bufs, shape, fa.FlatAttentionConfig(causal), None), shape)
    return fa.storage_to_f32(res.output, dtype).reshape(H, S, D), res.lse.reshape(H, S)


def _inputs(dims, dtype, seed):
    H, S, D = dims
    rnd = (lambda x: x) if dtype == F32 else bf16_round  # (bf16 values of this size are f16 ones)
    return [rnd(normal(H * S * D, seed + i)).reshape(H, S, D) for i in range(3)]


def _same(a, b):
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.filterwarnings("ignore:invalid value encountered")
@pytest.mark.parametrize("dtype,H,S,D,rows", KERNELS)
@pytest.mark.parametrize("where", ["q", "k", "v"])
@pytest.mark.parametrize("causal", [False, True])
def test_nan_reaches_what_reads_it_and_nothing_else(hip, dtype, H, S, D, rows, where, causal):
    """Q: its row's O and LSE. K: those of every row of the head that sees the key. V: the column of
    those rows (rows before the key multiply it by a probability of 0, which is NaN too)."""
    q, k, v = _inputs((H, S, D), dtype, 900)
    o0, l0 = _forward(hip, q, k, v, (H, S, D), dtype, causal)
    assert hip.last_telemetry().query_rows == rows[causal]
    o0b, l0b = _forward(hip, q, k, v, (H, S, D), dtype, causal)
    _same(o0, o0b)
    _same(l0, l0b)
    head, j, d = H - 2, 203, 9
    {"q": q, "k": k, "v": v}[where][head, j, d] = np.nan
    o1, l1 = _forward(hip, q, k, v, (H, S, D), dtype, causal)
    hit_o, hit_l, free = np.zeros(o0.shape, bool), np.zeros(l0.shape, bool), np.zeros(o0.shape, bool)
    seen = slice(j if causal else 0, None)
    if where == "q":
        hit_o[head, j] = hit_l[head, j] = True
    elif where == "k":
        hit_o[head, seen] = hit_l[head, seen] = True
    else:
        hit_o[head, seen, d] = True
        free[head, :j, d] = True
    assert np.isnan(o1[hit_o]).all() and np.isnan(l1[hit_l]).all()
    _same(o1[~(hit_o | free)], o0[~(hit_o | free)])
    _same(l1[~hit_l], l0[~hit_l])


@pytest.mark.parametrize("dtype,H,S,D,rows", KERNELS[:2] + KERNELS[3:5])
def test_infinite_key_is_masked_or_not_a_number(hip, dtype, H, S, D, rows):
    """K = +inf in one element of one key: a row whose Q is negative there has a score of -inf, as if
    the key were masked (the oracle without that key); a positive one has inf - inf."""
    q, k, v = _inputs((H, S, D), dtype, 920)
    j, d = 203, 9
    k[0, j, d] = np.inf
    o, l = _forward(hip, q, k, v, (H, S, D), dtype, False)
    assert hip.last_telemetry().query_rows == rows[0]
    # S rows over S - 1 keys
    keep = np.arange(S) != j
    eo, el = oracle.forward_projection_asymmetric(
        q[0].ravel(), k[0, keep].ravel(), v[0, keep].ravel(), 1, 1, 1, S, S - 1, D, 0, False, None)
    low, high = q[0, :, d] < 0, q[0, :, d] > 0
    tol = (2e-5, 1e-4) if dtype == F32 else (2e-2, 0.0)
    assert_close("O", o[0][low].ravel(), eo.reshape(S, D)[low].ravel(), *tol)
    assert_close("LSE", l[0][low], el.ravel()[low], *tol)
    assert np.isnan(o[0][high]).all() and not np.isfinite(l[0][high]).any()


@pytest.mark.filterwarnings("ignore:invalid value encountered")
@pytest.mark.parametrize("dtype", [F32, BF16, F16])
@pytest.mark.parametrize("D", [64, 128, 80])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
def test_padding_is_never_read(hip, dtype, D, causal, bad):
    """Padded rows of Q, K and V that are NaN or infinite: bitwise the result for zeros there."""
    shape = fa.AsymmetricGroupedAttentionShape(3, 8, 2, 150, 400, D, 0)
    meta = [fa.VariableLengthSequenceMetadata(aq, ak, ak - aq, ak - aq)
            for aq, ak in ((150, 333), (37, 400), (1, 65))]
    rnd = (lambda x: x) if dtype == F32 else bf16_round
    q, k, v = (rnd(normal(n, 940 + i)) for i, n in enumerate(
        (shape.q_tensor_len(), shape.kv_tensor_len(), shape.kv_tensor_len())))
    pipe = fa.HipVariableProjectionPipeline(hip, dtype)
    got = []
    for pad in (0.0, bad):
        for b, m in enumerate(meta):
            q.reshape(3, 150, -1)[b, m.active_query_len:] = pad
            k.reshape(3, 400, -1)[b, m.active_kv_len:] = pad
            v.reshape(3, 400, -1)[b, m.active_kv_len:] = pad
        out = pipe.create_output_buffer(shape)
        bufs = [fa.DeviceBuffer.from_array(hip, fa.host_storage(x, dtype)) for x in (q, k, v)]
        lay = pipe.encode(*bufs, out, shape, meta, fa.FlatAttentionConfig(causal),
                          fa.VariableLengthRotaryEmbeddingConfig(10000.0, 0))
        got.append(fa.download_attention(out, lay, dtype))
    _same(got[0].lse, got[1].lse)
    assert np.array_equal(got[0].output.view(np.uint8), got[1].output.view(np.uint8))
    assert np.isfinite(fa.storage_to_f32(got[1].output, dtype)).all()


@pytest.mark.filterwarnings("ignore:invalid value encountered")
@pytest.mark.parametrize("dtype,H,S,D", [(F32, 4, 300, 64), (F32, 4, 300, 128),   # split f32
                                         (F32, 96, 300, 128),                     # LDS-staged f32
                                         (BF16, 4, 600, 64), (BF16, 4, 600, 128),  # split key blocks
                                         (F16, 200, 300, 64)])                    # whole ones
@pytest.mark.parametrize("causal", [False, True])
def test_nan_stays_in_its_heads_gradients(hip, dtype, H, S, D, causal):
    """A NaN in one head's dO: that head's dQ row and dK are NaN, every other head bitwise the same."""
    q, k, v = _inputs((H, S, D), dtype, 960)
    do = _inputs((H, S, D), dtype, 970)[0]
    shape, cfg = fa.GroupedAttentionShape(1, H, H, S, D), fa.FlatAttentionConfig(causal)
    o, l = _forward(hip, q, k, v, (H, S, D), dtype, causal)
    fwd = fa.FlatAttentionOutput(o.ravel(), l.ravel())
    pipe = fa.HipGroupedBackwardRecomputePipeline(hip, dtype)
    bufs = [fa.DeviceBuffer.from_array(hip, fa.host_storage(x.ravel(), dtype)) for x in (q, k, v)]
    out = [fa.DeviceBuffer.from_array(hip, fa.host_storage(fwd.output, dtype)),
           fa.DeviceBuffer.from_array(hip, fwd.lse)]
    store = fa.host_storage(do.ravel(), dtype).dtype
    grads = []
    for bad in (False, True):
        if bad:
            do[H - 2, 201, 5] = np.nan
        g = [fa.DeviceBuffer(hip, H * S * D * store.itemsize) for _ in range(3)]
        db = fa.DeviceBuffer.from_array(hip, fa.host_storage(do.ravel(), dtype))
        pipe.encode_tensors(*bufs, db, out[0], out[1].ptr, *g, shape, cfg)
        grads.append([fa.storage_to_f32(x.download(store, H * S * D), dtype).reshape(H, S, D)
                      for x in g])
    others = np.arange(H) != H - 2
    for a, b in zip(*grads):
        _same(a[others], b[others])
    dq, dk, dv = (x[H - 2] for x in grads[1])
    assert np.isnan(dq[201]).all()
    seen = slice(0, 202 if causal else None)
    assert np.isnan(dk[seen]).all() and np.isnan(dv[seen, 5]).all()
