"""GPU parity of the training step: the HIP kernels behind the MatrixHIP training overloads,
and FreeML's own Model::Run(input, target) + AdamW on MatrixHIP against the reference.

Op level (C ABI, against the oracle's restatements, which tests/test_oracle_training.py pins
bit for bit to the compiled reference): data movement and the element-wise optimiser are
bit-exact (same operation order, no FMA contraction, correctly rounded divide and sqrt);
reductions whose order differs (row dots, LayerNorm sums, softmax sums) are within 1e-5
normwise; the transcendental element ops (erf/exp) within 2e-6 absolute.

Model level (oracle/_ref/nanollm_dropin, the reference's Model / Layer / loss / optimiser code
running on either backend): losses per iteration within 1e-5 relative of MatrixCPU's, every
gradient and error matrix after one backward within 1e-4 normwise, and no host copy inside an
iteration except the 4-byte loss readback that storeLoss asks for.
"""
import os
import re
import subprocess

import numpy as np
import pytest

import freeml_amd as fh
import oracle
from freeml_amd import checkpoint, synth
from freeml_amd.dropin import DROPIN, read_train, write_params

pytestmark = pytest.mark.gpu
# The comparisons with the reference's own training step run its code (test_dropin.py skips likewise).
needs_dropin = pytest.mark.skipif(not os.path.exists(DROPIN), reason="drop-in driver not built")


@pytest.fixture(scope="module", autouse=True)
def device():
    fh.init(0)


def rel(got, ref):
    ref = np.asarray(ref, np.float64)
    s = np.max(np.abs(ref))
    d = np.max(np.abs(np.asarray(got, np.float64) - ref))
    return d / s if s > 0 else d


def dev(a):
    return fh.DeviceArray.from_host(np.ascontiguousarray(a))


def rng(seed):
    return np.random.default_rng(seed)


@pytest.mark.parametrize("rows,cols", [(1, 1), (7, 1000), (256, 256), (33, 65)])
def test_softmax_backward(rows, cols):
    print(f"softmax_backward rows={rows} cols={cols}", flush=True)
    r = rng(rows + cols)
    x = r.standard_normal((rows, cols))
    p = (np.exp(x - x.max(1, keepdims=True)) / np.exp(x - x.max(1, keepdims=True)).sum(1, keepdims=True)).astype(np.float32)
    dp = r.standard_normal((rows, cols)).astype(np.float32)
    dP, dG, dO = dev(p), dev(dp), fh.DeviceArray((rows, cols))
    fh.softmax_backward(dO.ptr, dP.ptr, dG.ptr, rows, cols)
    assert rel(dO.numpy(), oracle.softmax_backward(p, dp)) <= 1e-5
    fh.softmax_backward(dG.ptr, dP.ptr, dG.ptr, rows, cols)  # out aliasing grad_in
    assert rel(dG.numpy(), oracle.softmax_backward(p, dp)) <= 1e-5


@pytest.mark.parametrize("rows,cols", [(1, 8), (5, 1000), (256, 384), (61, 64)])
@pytest.mark.parametrize("with_xhat", [True, False])
@pytest.mark.parametrize("with_beta", [True, False])
def test_layernorm_backward(rows, cols, with_xhat, with_beta):
    print(f"layernorm_backward rows={rows} cols={cols} xhat={with_xhat} beta={with_beta}", flush=True)
    r = rng(rows * cols)
    x = (r.standard_normal((rows, cols)) * 2 + 0.5).astype(np.float32)
    dy = r.standard_normal((rows, cols)).astype(np.float32)
    g = (1 + 0.1 * r.standard_normal(cols)).astype(np.float32)
    xhat = None
    if with_xhat:
        mu = x.mean(1, keepdims=True, dtype=np.float64)
        xhat = ((x - mu) / np.sqrt(x.var(1, keepdims=True, dtype=np.float64) + 1e-5)).astype(np.float32)
    ex, eg, eb = oracle.layernorm_backward(dy, x, g, xhat, with_beta)
    dX, dDY, dIN, dGm = fh.DeviceArray((rows, cols)), dev(dy), dev(x), dev(g)
    dDG = fh.DeviceArray(cols)
    dDB = fh.DeviceArray(cols) if with_beta else None
    dXH = dev(xhat) if with_xhat else None
    ws = None if with_xhat else fh.DeviceArray(2 * rows)
    fh.layernorm_backward(dX.ptr, dDY.ptr, dIN.ptr, dGm.ptr, dDG.ptr, dDB.ptr if dDB else None,
                          dXH.ptr if dXH else None, ws.ptr if ws else None, rows, cols)
    assert rel(dX.numpy(), ex) <= 1e-5
    assert rel(dDG.numpy(), eg) <= 1e-5
    if with_beta:
        assert rel(dDB.numpy(), eb) <= 1e-5


def test_layernorm_backward_rejects_missing_workspace():
    a = fh.DeviceArray((4, 8))
    g = fh.DeviceArray(8)
    with pytest.raises(fh.FreeMLHipError, match="workspace"):
        fh.layernorm_backward(a.ptr, a.ptr + 0, a.ptr, g.ptr, g.ptr, None, None, None, 4, 8)


def test_gelu_derivative():
    x = np.concatenate([np.linspace(-9, 9, 4001), rng(1).standard_normal(100000) * 3]).astype(np.float32)
    dx, do = dev(x), fh.DeviceArray(x.shape)
    fh.gelu_derivative(do.ptr, dx.ptr, x.size)
    np.testing.assert_allclose(do.numpy(), oracle.gelu_derivative(x), atol=2e-6, rtol=0)


@pytest.mark.parametrize("src_batch,out_batch,width,src_rows,out_rows",
                         [(1, 1, 384, 256, 65), (3, 1, 37, 50, 9), (3, 3, 37, 50, 9),
                          (1, 1, 2500, 300, 4), (1, 1, 64, 700, 700)])
def test_scatter_add_rows_bit_exact(src_batch, out_batch, width, src_rows, out_rows):
    """Same per-row summation order as the reference: identical bits, also with every source
    row going to the same few destinations and with widths beyond one pass of the block."""
    print(f"scatter_add_rows {src_batch}/{out_batch} w={width} src={src_rows} out={out_rows}", flush=True)
    r = rng(width + src_rows)
    out = r.standard_normal((out_batch, out_rows, width)).astype(np.float32)
    src = r.standard_normal((src_batch, src_rows, width)).astype(np.float32)
    idx = r.integers(0, out_rows, (src_batch, src_rows)).astype(np.float32)
    dO, dS, dI = dev(out), dev(src), dev(idx)
    fh.scatter_add_rows(dO.ptr, dS.ptr, dI.ptr, width, src_rows, src_batch, out_rows, out_batch)
    np.testing.assert_array_equal(dO.numpy(), oracle.scatter_add_rows(out, src, idx))


def test_scatter_add_rows_skips_out_of_range_ids():
    out = np.zeros((1, 4, 8), np.float32)
    src = np.ones((1, 5, 8), np.float32)
    idx = np.array([[0, 7, -1, 3, 4.0]], np.float32)  # 7, -1 and 4 are outside [0, 4)
    dO, dS, dI = dev(out), dev(src), dev(idx)
    fh.scatter_add_rows(dO.ptr, dS.ptr, dI.ptr, 8, 5, 1, 4, 1)
    expect = np.zeros((1, 4, 8), np.float32)
    expect[0, 0] = 1
    expect[0, 3] = 1
    np.testing.assert_array_equal(dO.numpy(), expect)


def test_merge_qkv_bit_exact():
    r = rng(3)
    q, k, v = (r.standard_normal((6, 256, 64)).astype(np.float32) for _ in range(3))
    dq, dk, dv, dp = dev(q), dev(k), dev(v), fh.DeviceArray((256, 3 * 384))
    fh.merge_qkv(dp.ptr, dq.ptr, dk.ptr, dv.ptr, 64, 256, 6)
    np.testing.assert_array_equal(dp.numpy(), oracle.merge_qkv(q, k, v))


# merge_qkv: four columns of a head per thread where head_dim and every pointer allow it: one and several
# passes of the block over a row, head_dims of 4 and not, and a pointer off by one float.
@pytest.mark.parametrize("heads,tokens,hd", [(1, 1, 4), (3, 33, 64), (12, 5, 64), (5, 7, 3), (2, 9, 600)])
@pytest.mark.parametrize("off", [0, 1])
def test_split_and_merge_qkv_bit_exact(heads, tokens, hd, off):
    r, C = rng(heads + tokens), heads * hd
    print(f"split / merge qkv heads={heads} tokens={tokens} hd={hd} offset={off}", flush=True)
    q, k, v = (r.standard_normal((heads, tokens, hd)).astype(np.float32) for _ in range(3))
    dq, dk, dv = dev(np.concatenate([np.zeros(off, np.float32), q.ravel()])), dev(k), dev(v)
    dp = fh.DeviceArray((tokens, 3 * C))
    fh.merge_qkv(dp.ptr, dq.ptr + 4 * off, dk.ptr, dv.ptr, hd, tokens, heads)
    rows = [np.ascontiguousarray(t.transpose(1, 0, 2).reshape(tokens, C)) for t in (q, k, v)]
    np.testing.assert_array_equal(dp.numpy(), np.concatenate(rows, 1))
    sq, sk, sv = dev(np.full(tokens * C + off, 7.0, np.float32)), fh.DeviceArray((tokens, C)), fh.DeviceArray((tokens, C))
    fh.split_qkv(sq.ptr + 4 * off, sk.ptr, sv.ptr, dp.ptr, tokens, C)
    got = sq.numpy()
    np.testing.assert_array_equal(got[off:].reshape(tokens, C), rows[0])
    assert np.all(got[:off] == 7.0)
    np.testing.assert_array_equal(sk.numpy(), rows[1])
    np.testing.assert_array_equal(sv.numpy(), rows[2])


# Rows held in registers: the widest of each register count and one more, LayerNorm rows of 8 and 16
# values per lane and longer ones, one row, and rows around the 64 a block's lanes take at once.
@pytest.mark.parametrize("rows,cols", [(63, 512), (65, 513), (64, 1024), (3, 1025), (1, 17)])
def test_layernorm_backward_register_rows(rows, cols):
    test_layernorm_backward(rows, cols, True, True)
    test_layernorm_backward(rows, cols, False, True)


@pytest.mark.parametrize("vocab", [1, 1024, 1025, 4096, 4097, 32768, 32769, 65536, 65537])
def test_cce_logits_register_rows(vocab):
    test_cce_logits("index_ignore", 1, 5, vocab)


@pytest.mark.parametrize("kind,batch,steps,vocab",
                         [("index", 1, 256, 65), ("index_ignore", 1, 64, 65), ("index", 4, 128, 50304),
                          ("onehot", 1, 31, 65), ("index_all_ignored", 1, 8, 65)])
def test_cce_logits(kind, batch, steps, vocab):
    print(f"cce {kind} batch={batch} steps={steps} vocab={vocab}", flush=True)
    r = rng(steps + vocab)
    z = (r.standard_normal((batch, steps, vocab)) * 3).astype(np.float32)
    if kind == "onehot":
        t = np.zeros((1, steps, vocab), np.float32)
        t[0, np.arange(steps), r.integers(0, vocab, steps)] = 1
        tcols = vocab
    else:
        t = r.integers(0, vocab, (batch, steps)).astype(np.float32)
        if kind == "index_ignore":
            t[0, ::3] = -1
        if kind == "index_all_ignored":
            t[:] = -1
        tcols = 1
    eg, el = oracle.cce_logits(t, z)
    dT, dZ, dG = dev(t), dev(z), fh.DeviceArray(z.shape)
    dL, ws = fh.DeviceArray(1), fh.DeviceArray(batch * steps)
    fh.cce_logits(dG.ptr, dL.ptr, ws.ptr, dT.ptr, dZ.ptr, vocab, steps, batch, tcols, t.shape[0])
    got, loss = dG.numpy(), float(dL.numpy()[0])
    # The exact (float64) gradient and loss.  The reference sums exp(z - max) sequentially in
    # fp32, whose rounding grows with the vocabulary; the device sums by a tree.  So the device
    # must be within 1e-5 of the exact values and no further from the reference than the
    # reference itself is from them (plus 1e-5).
    z64 = z.astype(np.float64)
    e = np.exp(z64 - z64.max(-1, keepdims=True))
    p64 = e / e.sum(-1, keepdims=True)
    lse = np.log(e.sum(-1)) + z64.max(-1)
    if tcols == 1:
        ids = np.broadcast_to(t, (batch, steps)).astype(np.int64)
        valid = ids != -1
        onehot = np.zeros_like(p64)
        b_, s_ = np.nonzero(valid)
        onehot[b_, s_, ids[valid]] = 1
        n_valid = max(int(valid.sum()), 1)
        g64 = np.where(valid[..., None], (onehot - p64) / n_valid, 0.0)
        l64 = float((lse[valid] - z64[b_, s_, ids[valid]]).sum() / n_valid) if valid.any() else 0.0
    else:
        g64 = t.astype(np.float64) - p64
        first = np.argmax(t > 0.5, axis=-1)
        l64 = float((lse - np.take_along_axis(z64, first[..., None], -1)[..., 0]).sum())
    assert rel(got, g64) <= 1e-5
    assert rel(got, eg) <= rel(eg, g64) + 1e-5
    assert abs(loss - l64) <= 1e-5 * max(1.0, abs(l64)), (loss, l64)
    assert abs(loss - el) <= abs(el - l64) + 1e-5 * max(1.0, abs(l64)), (loss, el, l64)


@pytest.mark.parametrize("t", [1, 2, 50])
def test_adamw_bit_exact(t):
    r = rng(t)
    n = 100003
    p = (r.standard_normal(n) * 0.02).astype(np.float32)
    g = (r.standard_normal(n) * 1e-3).astype(np.float32)
    g[:7] = 0
    m = (r.standard_normal(n) * 1e-4).astype(np.float32)
    v = (r.random(n) * 1e-6).astype(np.float32)
    ep, em, ev = oracle.adamw_update(p, g, m, v, 1e-4, 0.9, 0.999, t, 1e-8, 0.01)
    b1t, b2t = oracle.adam_powers(0.9, 0.999, t)
    dp_, dg, dm, dv = dev(p), dev(g), dev(m), dev(v)
    fh.adamw_update(dp_.ptr, dg.ptr, dm.ptr, dv.ptr, n, 1e-4, 0.9, 0.999, b1t, b2t, 1e-8, 0.01)
    np.testing.assert_array_equal(dm.numpy(), em)
    np.testing.assert_array_equal(dv.numpy(), ev)
    np.testing.assert_array_equal(dp_.numpy(), ep)


@pytest.mark.parametrize("n_head,T", [(6, 256), (4, 64), (3, 100), (32, 16)])
def test_attention_softmax_heads(n_head, T):
    """Scale + causal mask + Softmax for all heads = the layer's ScaleAdd and Softmax per head
    (oracle restatements, pinned to the compiled reference), into per-head matrices at a batch
    plane offset and into the contiguous all-heads buffer."""
    print(f"attention_softmax_heads heads={n_head} T={T}", flush=True)
    r = rng(n_head * T)
    scores = (r.standard_normal((n_head, T, T)) * 4).astype(np.float32)
    scale = np.float32(1 / np.sqrt(64))
    mask = oracle.triangle_lower(T, T, 0.0, -np.inf)
    expect = np.stack([oracle.softmax(oracle.scale_add(scores[h], float(scale), mask)) for h in range(n_head)])
    dS, dScale, dAll = dev(scores), dev(np.array([scale])), fh.DeviceArray((n_head, T, T))
    heads = [fh.DeviceArray((2, T, T)) for _ in range(n_head)]  # two batch planes; write plane 1
    fh.attention_softmax_heads([hh.ptr for hh in heads], T * T, dAll.ptr, dS.ptr, dScale.ptr, n_head, T)
    got_all = dAll.numpy()
    assert rel(got_all, expect) <= 1e-6
    for h in range(n_head):
        np.testing.assert_array_equal(heads[h].numpy()[1], got_all[h])
        assert np.all(np.triu(got_all[h], 1) == 0)


@pytest.mark.parametrize("n_head,T", [(6, 256), (3, 100)])
def test_attention_softmax_backward_heads(n_head, T):
    """SoftmaxBackwards, mask and scale for all heads = the layer's three per-head ops."""
    print(f"attention_softmax_backward_heads heads={n_head} T={T}", flush=True)
    r = rng(n_head + T)
    mask = oracle.triangle_lower(T, T, 0.0, -np.inf)
    fin = oracle.triangle_lower(T, T, 1.0, 0.0)
    P = np.stack([oracle.softmax(oracle.scale_add(r.standard_normal((T, T)).astype(np.float32), 1.0, mask))
                  for _ in range(n_head)])
    dA = r.standard_normal((n_head, T, T)).astype(np.float32)
    scale = np.float32(0.125)
    expect = np.stack([(oracle.softmax_backward(P[h], dA[h]) * fin) * scale for h in range(n_head)])
    heads = [dev(P[h]) for h in range(n_head)]
    dDA, dScale, dOut = dev(dA), dev(np.array([scale])), fh.DeviceArray((n_head, T, T))
    fh.attention_softmax_backward_heads(dOut.ptr, [hh.ptr for hh in heads], dDA.ptr, dScale.ptr, n_head, T)
    assert rel(dOut.numpy(), expect) <= 1e-5


# ---- the reference's training step on MatrixHIP -------------------------------------------

def train(backend, name, iters, tmp, *extra, env=None):
    w = synth.make_weights(synth.CONFIGS[name]["shape"], 0)
    corpus = synth.prompt_tokens(w.shape.vocab, 4 * w.shape.block_size, 5)
    inp, out = os.path.join(tmp, f"in_{backend}.bin"), os.path.join(tmp, f"out_{backend}.bin")
    write_params(inp, w, corpus, 0)
    print(f"nanollm_dropin {backend} --train {iters} {' '.join(extra)} ({name})", flush=True)
    r = subprocess.run([DROPIN, backend, inp, out, "--train", str(iters), *extra], capture_output=True,
                       text=True, timeout=600, env=dict(os.environ, **(env or {})))
    assert r.returncode == 0, r.stderr
    print(r.stdout.strip(), flush=True)
    if backend == "hip":
        path = "per-head" if env else "batched"
        m = re.search(r"(\d+) batched / (\d+) per-head forwards, (\d+) batched / (\d+) per-head backwards",
                      r.stdout)
        counts = dict(zip(("bf", "pf", "bb", "pb"), map(int, m.groups())))
        # Every attention layer of every iteration took the expected path.
        if path == "batched":
            assert counts["pf"] == 0 and counts["pb"] == 0 and counts["bf"] > 0, counts
        else:
            assert counts["bf"] == 0 and counts["bb"] == 0 and counts["pf"] > 0, counts
    losses, _, copies = read_train(out, iters)
    return losses, copies


@needs_dropin
@pytest.mark.parametrize("name,iters,per_head", [("c1", 12, False), ("c2", 4, False), ("c2", 4, True)])
def test_training_iterations_match_reference(name, iters, per_head, tmp_path):
    """K iterations of TrainLoop's step (window + shifted target, forward, CCE gradient,
    backward, AdamW) on both backends from the same weights; the MatrixHIP attention layer on
    its all-heads path and, forced, on its head-by-head path."""
    ref, _ = train("cpu", name, iters, str(tmp_path))
    env = {"FMLH_ATTENTION_PER_HEAD": "1"} if per_head else None
    got, copies = train("hip", name, iters, str(tmp_path), env=env)
    np.testing.assert_allclose(got, ref, rtol=1e-5, atol=0)
    if iters >= 10:
        assert ref[-1] < ref[0]  # it trains
    assert copies.tolist() == [iters - 1, 0], copies  # only the loss readback per iteration


GRADS = re.compile(r"(Grad|WUpdate|Delta|ErrorOutput_\d+|ErrorInput_\d+|Scratch_d\w+|Scratch_QKVGrad)$")


def _walk(rec, prefix=""):
    for k, m in rec.matrices.items():
        yield f"{prefix}{rec.name}/{k}", m
    for k, sub in rec.sublayers.items():
        yield from _walk(sub, f"{prefix}{rec.name}/{k}:")


@needs_dropin
@pytest.mark.parametrize("name", ["c1", "c2"])
def test_backward_gradients_match_reference(name, tmp_path):
    """One backward without optimiser on each backend, saved with Model::Save: every weight
    gradient and error signal within 1e-4 normwise of the reference's."""
    mats = {}
    for be in ("cpu", "hip"):
        d = str(tmp_path / be)
        os.makedirs(d)
        train(be, name, 1, d, "--grads", "--save", os.path.join(d, "ck"))
        ck = checkpoint.read_checkpoint(os.path.join(d, "ck", "NanoLLM_dropin"))
        mats[be] = dict(kv for rec in ck.layers for kv in _walk(rec))
    checked = 0
    for key, m in mats["cpu"].items():
        if not GRADS.search(key):
            continue
        e = rel(mats["hip"][key].array(), m.array())
        assert e <= 1e-4, (key, e)
        checked += 1
    assert checked >= (90 if name == "c1" else 250), checked


@pytest.mark.parametrize("rows,cols", [(1, 1), (256, 384), (1000, 65), (3, 5000)])
def test_sum_columns_bit_exact(rows, cols):
    """SumColumns (the Dense bias gradient) on the device: each column's rows added in row
    order, bit-identical to the oracle (which the CPU suite pins to the reference)."""
    x = (rng(rows + cols).standard_normal((rows, cols)) * 3).astype(np.float32)
    dX, dO = dev(x), fh.DeviceArray(cols)
    fh.sum_columns(dO.ptr, dX.ptr, rows, cols)
    np.testing.assert_array_equal(dO.numpy(), oracle.sum_columns(x))


@pytest.mark.parametrize("n,start,prob", [(1, 0, 0.1), (100003, 7, 0.1), (5000, 999_000, 0.5)])
def test_dropout_mask_bit_exact(n, start, prob):
    """UpdateMask's draws on the device from a uniform buffer (1e6 floats here), starting at a
    running index and wrapping at the buffer's end, equal to the restatement."""
    u = rng(n).random(1_000_000).astype(np.float32)
    dU, dM = dev(u), fh.DeviceArray(n)
    fh.dropout_mask(dM.ptr, n, dU.ptr, u.size, start, prob)
    np.testing.assert_array_equal(dM.numpy(), oracle.dropout_mask(n, u, start, prob)[0])


@needs_dropin
def test_training_with_biases_and_dropout_matches_reference(tmp_path):
    """The reference's training step with use_bias = true (Dense biases, their SumColumns
    gradient) and dropout 0.1 (embedding, attention-residual and MLP dropout; masks drawn on the
    device from RandomUtils' own uniform buffer) on MatrixHIP, against MatrixCPU run first in
    the same process so both draw from the same buffer: losses within 1e-5 relative, and no
    host copy inside an iteration but the loss readback."""
    name, iters = "c1", 8
    w = synth.make_weights(synth.CONFIGS[name]["shape"], 0)
    corpus = synth.prompt_tokens(w.shape.vocab, 4 * w.shape.block_size, 5)
    inp, out = str(tmp_path / "in.bin"), str(tmp_path / "out.bin")
    write_params(inp, w, corpus, 0)
    print(f"nanollm_dropin cpuhip --train {iters} --bias --dropout 0.1", flush=True)
    r = subprocess.run([DROPIN, "cpuhip", inp, out, "--train", str(iters), "--bias", "--dropout", "0.1"],
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr
    print(r.stdout.strip(), flush=True)
    got, _, copies = read_train(out, iters)
    ref, _, _ = read_train(out + ".cpu", iters)
    np.testing.assert_allclose(got, ref, rtol=1e-5, atol=0)
    assert copies.tolist() == [iters - 1, 0], copies
    # dropout is really on: the same run without it gives other losses
    r0 = subprocess.run([DROPIN, "cpu", inp, out + ".nodrop", "--train", str(iters), "--bias"],
                        capture_output=True, text=True, timeout=600)
    assert r0.returncode == 0, r0.stderr
    nodrop, _, _ = read_train(out + ".nodrop", iters)
    assert np.max(np.abs(nodrop - ref)) > 1e-4
