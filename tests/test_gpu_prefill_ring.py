"""The two-tile causal prefill kernel where its rings and lazy maximum can go
wrong, against the CPU oracle: more key blocks than the ring holds (4), rows
past the end (waves that only keep the barriers), scores that outgrow the
softmax reference in a late block, and scales from one that makes every
visible key weigh the same to one that picks a single key.

P is rounded to bf16 (half an ulp, 2^-9 = 2.0e-3 of each weight) and nothing
else is below f32, so a row is within 2^-9 of its values' scale; 4e-3 leaves a
factor of two for the norm that rel_err divides by."""
import numpy as np
import pytest

import oracle
from conftest import rel_err
from test_gpu_prefill import make

pytestmark = pytest.mark.gpu

TOL = 4e-3


def reference(q, kc, vc, starts, scale):
    k, v = oracle.bf16_to_f32(kc).astype(np.float64), oracle.bf16_to_f32(vc).astype(np.float64)
    group = q.shape[2] // k.shape[1]
    out = np.empty(q.shape)
    for b in range(q.shape[0]):
        for h in range(q.shape[2]):
            s = q[b, :, h].astype(np.float64) @ k[b, h // group].T * scale
            pos = starts[b] + np.arange(q.shape[1])
            s[np.arange(k.shape[2])[None, :] > pos[:, None]] = -np.inf
            p = np.exp(s - s.max(axis=1, keepdims=True))
            out[b, :, h] = p / p.sum(axis=1, keepdims=True) @ v[b, h // group]
    return out


@pytest.mark.parametrize("q_bf16", [True, False])
@pytest.mark.parametrize("group,rows,starts,scale", [
    (1, 129, [0, 200], None), (2, 1, [319, 0], None), (2, 129, [447, 60], 1.5),
    (4, 33, [255, 256], None), (4, 300, [150, 0], 1e-38), (8, 160, [63, 300], None)])
def test_rings_and_late_maxima(rt, group, rows, starts, scale, q_bf16):
    import rxla_amd as r
    rng = np.random.default_rng(rows + group)
    q, kc, vc = make(rng, 2, rows, 2 * group, 2, 600)
    k = oracle.bf16_to_f32(kc)
    k[:, :, 64:] *= 2  # scores grow from the second block on, past the lazy reference
    k[:, :, 256:] *= 2
    kc = oracle.bf16_bits(k)
    if q_bf16:
        q = oracle.round_bf16(q)
    qb = rt.buffer(oracle.bf16_bits(q), r.DType.BF16) if q_bf16 else rt.buffer(q)
    out = r.grouped_query_attention_prefill(
        rt, qb, rt.buffer(kc, r.DType.BF16), rt.buffer(vc, r.DType.BF16),
        rt.buffer(np.asarray(starts, np.int32)), out_dtype=r.DType.F32,
        **({} if scale is None else {"scale": scale})).to_numpy()
    ref = reference(q, kc, vc, starts, 128 ** -0.5 if scale is None else scale)
    assert np.isfinite(out).all()
    assert rel_err(out, ref) <= TOL


@pytest.mark.parametrize("group", [1, 2, 4, 8])
@pytest.mark.parametrize("rows,start", [(1, 0), (1, 63), (17, 40), (64, 0), (64, 1), (65, 0)])
@pytest.mark.parametrize("q_bf16", [True, False])
def test_one_and_two_blocks(rt, group, rows, start, q_bf16):
    """A single block of 64 keys runs both heads of a workgroup in step, two
    run them half a step apart."""
    import rxla_amd as r
    rng = np.random.default_rng(64 * rows + start + group)
    q, kc, vc = make(rng, 2, rows, 2 * group, 2, 130)
    if q_bf16:
        q = oracle.round_bf16(q)
    qb = rt.buffer(oracle.bf16_bits(q), r.DType.BF16) if q_bf16 else rt.buffer(q)
    starts = np.array([start, max(0, start - 3)], np.int32)
    out = r.grouped_query_attention_prefill(rt, qb, rt.buffer(kc, r.DType.BF16), rt.buffer(vc, r.DType.BF16),
                                            rt.buffer(starts), out_dtype=r.DType.F32).to_numpy()
    assert rel_err(out, reference(q, kc, vc, starts, 128 ** -0.5)) <= TOL
