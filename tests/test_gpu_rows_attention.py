"""GPU parity: fused row kernels, attention and dense matmuls against the oracle (and the reference C library's
recorded vectors). Tolerances: the reference's own for fused rows (rel 1e-4, abs 1e-5, NativeFusedKernelsTest.kt:166-218);
2e-2 normalised is the task's bound for attention, the fp32 kernels here are held to 1e-4.
"""
import os

import numpy as np
import pytest

from oracle import lib as L
from gpu_util import dev, launches, normalized_err
from test_oracle_golden import SDPA_GRID, fill, sdpa_fp64, sdpa_inputs

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))


def close(got, want, rel=1e-4, abs_=1e-5):
    """assertClose of NativeFusedKernelsTest.kt:53-61: |d| <= max|want| * rel + abs."""
    tol = np.abs(want).max() * rel + abs_
    d = np.abs(np.asarray(got, np.float64) - want).max()
    assert d <= tol, (d, tol)


def gpu_sdpa(kernels, torch, q, k, v, scale, causal=False, window=0, rc=0, lengths=None, mask=None):
    b, h, sq, d = q.shape
    hkv, skv = k.shape[1], k.shape[2]
    out = torch.full(q.shape, float("nan"), dtype=torch.float32, device="cuda")
    md = (0, 0, 0, 0)
    dm = None
    if mask is not None:
        md = tuple([1] * (4 - mask.ndim) + list(mask.shape))
        dm = dev(torch, mask)
    dl = None if lengths is None else dev(torch, np.asarray(lengths, np.int32))
    kernels.sdpa_dev(dev(torch, q), dev(torch, k), dev(torch, v), out, b, h, hkv, sq, skv, d, scale, causal, window, rc, dl, dm, md)
    return out.cpu().numpy()


@pytest.mark.parametrize("case", SDPA_GRID)
def test_attention_every_mask_rule(hip_backend, torch_cuda, case):
    h, hkv, sq, skv, causal, use_len, win, rc = case
    q, k, v = sdpa_inputs(3, h, hkv, sq, skv, 8)
    lengths = np.array([skv, (skv + 1) // 2, 1], np.int32) if use_len else None
    scale = float(1.0 / np.sqrt(8))
    got = gpu_sdpa(hip_backend, torch_cuda, q, k, v, scale, causal, win, rc, lengths)
    close(got, L.sdpa(q, k, v, scale, causal, win, rc, lengths))
    recorded = np.load(os.path.join(HERE, "golden", "ref_vectors.npz"))[f"sdpa/{SDPA_GRID.index(case)}"]
    close(got, recorded)
    # the structured rules equal the dense -1e30 mask (AttentionMask.additive)
    dense = np.full((3, 1, sq, skv), -1e30, np.float32)
    for b in range(3):
        for qi in range(sq):
            absq = skv - sq + qi
            first = max(0, absq - win + 1) if win > 0 else 0
            end = min(skv, lengths[b] if use_len else skv)
            if causal:
                end = min(end, absq + 1)
            if win > 0:
                end = min(end, absq + rc + 1)
            dense[b, 0, qi, first:max(end, first)] = 0.0
    close(gpu_sdpa(hip_backend, torch_cuda, q, k, v, scale, mask=dense), got, rel=1e-5, abs_=1e-6)


def test_attention_masks_padding_and_host_entry(hip_backend, torch_cuda):
    q, k, v = sdpa_inputs(2, 4, 2, 5, 9, 16, seed=4)
    for mask in (fill(9, 6).reshape(1, 1, 1, 9), fill(45, 7).reshape(5, 9), fill(2 * 4 * 5 * 9, 8).reshape(2, 4, 5, 9),
                 fill(2 * 2 * 5 * 9, 9).reshape(2, 2, 5, 9)):
        close(gpu_sdpa(hip_backend, torch_cuda, q, k, v, 0.3, True, mask=mask), L.sdpa(q, k, v, 0.3, True, mask=mask))
    q, k, v = sdpa_inputs(2, 2, 2, 3, 5, 4)
    out = gpu_sdpa(hip_backend, torch_cuda, q, k, v, 0.5, lengths=[0, 5])
    assert np.isfinite(out).all()
    close(out, L.sdpa(q, k, v, 0.5, lengths=np.array([0, 5], np.int32)), rel=1e-5, abs_=1e-6)
    # seq_kv == 0 zeroes the output; the SPI kernel on host arrays goes through the same path
    attn = hip_backend.HipKernelProvider().attention_fp32()
    o = np.full(q.shape, 5, np.float32)
    attn.sdpa(q, k[:, :, :0].copy(), v[:, :, :0].copy(), o, 2, 2, 2, 3, 0, 4, 0.5, False, 0, 0)
    assert not o.any()
    q, k, v = sdpa_inputs(1, 12, 12, 150, 150, 64, seed=9)     # the reference's threaded shape (NativeFusedKernelsTest.kt:211)
    o = np.empty_like(q)
    want = L.sdpa(q, k, v, 1 / np.sqrt(64.0), True)
    hip_backend.set_tuning("sdpa_decode_prompts", 0)              # on the prompt kernel: bf16 operands on the matrix cores
    try:
        attn.sdpa(q, k, v, o, 1, 12, 12, 150, 150, 64, float(1 / np.sqrt(64.0)), True, 0, 0)
        assert hip_backend.last_kernel() == "sdpa_prefill_kernel"
    finally:
        hip_backend.set_tuning("sdpa_decode_prompts", 1)
    assert normalized_err(o, want, eps=1.0) <= 2e-2
    hip_backend.set_tuning("sdpa_prefill_mfma", 0)                # the same call on the fp32 kernel: the reference's tolerance
    try:
        attn.sdpa(q, k, v, o, 1, 12, 12, 150, 150, 64, float(1 / np.sqrt(64.0)), True, 0, 0)
    finally:
        hip_backend.set_tuning("sdpa_prefill_mfma", 1)
    close(o, want)
    with pytest.raises(ValueError):
        attn.sdpa(q, k, v, o, 1, 12, 12, 150, 150, 64, 0.1, True, 0, 2)


@pytest.mark.parametrize("batch", [1, 8])
def test_attention_decode_config(hip_backend, torch_cuda, batch):
    """Decode: one query token against a KV cache of 4096, 32 query / 8 KV heads, head_dim 128."""
    rng = np.random.default_rng(50 + batch)
    q = rng.standard_normal((batch, 32, 1, 128)).astype(np.float32)
    k = rng.standard_normal((batch, 8, 4096, 128)).astype(np.float32)
    v = rng.standard_normal((batch, 8, 4096, 128)).astype(np.float32)
    scale = float(1 / np.sqrt(128.0))
    got = gpu_sdpa(hip_backend, torch_cuda, q, k, v, scale, True)
    want = L.sdpa(q, k, v, scale, True)
    err = normalized_err(got, want)
    print(f"decode attention batch {batch}: normalized max err {err:.2e}")
    assert err <= 2e-2
    lengths = np.arange(1, batch + 1, dtype=np.int32) * 500
    close(gpu_sdpa(hip_backend, torch_cuda, q, k, v, scale, True, 1024, 0, lengths), L.sdpa(q, k, v, scale, True, 1024, 0, lengths))


@pytest.mark.parametrize("heads,kv_heads,d,skv,batch", [(8, 2, 64, 700, 2), (4, 4, 128, 33, 3), (16, 2, 128, 1500, 1),
                                                         (6, 3, 256, 260, 2), (2, 1, 64, 16, 1), (32, 8, 128, 2048, 1),
                                                         (12, 4, 64, 5000, 1), (5, 5, 96, 300, 2)])
def test_attention_decode_kernel_shapes_and_rules(hip_backend, torch_cuda, heads, kv_heads, d, skv, batch):
    """The one-query kernel over its head shapes (group sizes 1 / 2 / 4 / 8-as-2x4, head_dim 64 / 128 / 256; 96 stays
    on the general kernel), split and unsplit key ranges, key lengths (one of them 0: uniform weights), windows,
    and twice in a row so the split counters are known to come back to zero."""
    rng = np.random.default_rng(heads * d + skv)
    q = rng.standard_normal((batch, heads, 1, d)).astype(np.float32)
    k = rng.standard_normal((batch, kv_heads, skv, d)).astype(np.float32)
    v = rng.standard_normal((batch, kv_heads, skv, d)).astype(np.float32)
    scale = float(1 / np.sqrt(d))
    lengths = np.array([skv, 0, skv // 3][:batch], np.int32)
    for causal, win, rc, lens in ((True, 0, 0, None), (False, 0, 0, lengths), (True, max(1, skv // 5), 0, None),
                                  (True, max(2, skv // 2), 1, lengths), (True, 0, 0, None)):
        got = gpu_sdpa(hip_backend, torch_cuda, q, k, v, scale, causal, win, rc, lens)
        close(got, L.sdpa(q, k, v, scale, causal, win, rc, lens), rel=2e-5, abs_=2e-6)


@pytest.mark.parametrize("one_launch", [1, 0])
@pytest.mark.parametrize("batch,heads,kv_heads,d,sq,skv", [(1, 8, 2, 128, 2, 65), (2, 6, 2, 64, 3, 300), (1, 4, 4, 128, 8, 8), (1, 3, 1, 64, 15, 700),
                                                           (3, 2, 1, 256, 5, 129), (1, 32, 8, 128, 4, 1500), (2, 1, 1, 64, 2, 40)])
def test_attention_of_a_few_queries_over_a_cache(hip_backend, torch_cuda, batch, heads, kv_heads, d, sq, skv, one_launch):
    """2 to 15 queries per sequence on the cache-streaming kernel: rows of several queries and heads share a workgroup, each
    with a key range of its own (causal and window move with the query, lengths cut some of them to nothing, one sequence
    to no key at all), padded last workgroups, one split and several."""
    rng = np.random.default_rng(heads * d + skv + sq)
    q = rng.standard_normal((batch, heads, sq, d)).astype(np.float32)
    k = rng.standard_normal((batch, kv_heads, skv, d)).astype(np.float32)
    v = rng.standard_normal((batch, kv_heads, skv, d)).astype(np.float32)
    scale = float(1 / np.sqrt(d))
    lengths = np.array([skv - sq // 2, 0, skv // 3][:batch], np.int32)
    hip_backend.set_tuning("sdpa_decode_one_launch", one_launch)
    try:
        for causal, win, rc, lens in ((True, 0, 0, None), (False, 0, 0, None), (True, 0, 0, lengths), (True, max(1, skv // 5), 0, None),
                                      (False, 3, 2, lengths), (True, 2, 0, lengths)):
            got = gpu_sdpa(hip_backend, torch_cuda, q, k, v, scale, causal, win, rc, lens)
            assert hip_backend.last_kernel() == "sdpa_decode_kernel"
            close(got, L.sdpa(q, k, v, scale, causal, win, rc, lens), rel=2e-5, abs_=2e-6)
    finally:
        hip_backend.set_tuning("sdpa_decode_one_launch", 1)


@pytest.mark.parametrize("one_launch", [1, 0])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("heads,kv_heads,d,sq,skv", [(8, 2, 128, 2, 65), (6, 2, 64, 3, 300), (3, 1, 64, 15, 700), (2, 1, 256, 5, 129), (4, 4, 128, 5, 1500),
                                                     (1, 1, 64, 2, 40)])
def test_a_draft_query_takes_nothing_from_keys_that_are_hidden_from_it(hip_backend, torch_cuda, heads, kv_heads, d, sq, skv, bad, one_launch):
    """Rows with different key ranges share a workgroup that walks the union of the ranges. Infinite or undefined K and V at
    keys that some rows attend and others do not: the later tokens of the draft, the first query's oldest window key, the
    padding past a short length beside a row that the window and the length leave no key (that row weighs every key). Rows
    that do not attend the bad keys give the oracle's result on finite values there."""
    rng = np.random.default_rng(heads * d + skv + sq)
    q = rng.standard_normal((1, heads, sq, d)).astype(np.float32)
    k = rng.standard_normal((1, kv_heads, skv, d)).astype(np.float32)
    v = rng.standard_normal((1, kv_heads, skv, d)).astype(np.float32)
    scale = float(1 / np.sqrt(d))
    pos, key = np.arange(skv - sq, skv)[:, None], np.arange(skv)[None, :]
    win = min(3, sq)
    hip_backend.set_tuning("sdpa_decode_one_launch", one_launch)
    try:
        # (window, length, bad keys): the last token, every later token than the first query's, the first query's oldest key, padding
        for w, length, keys in ((0, None, [skv - 1]), (0, None, range(skv - sq + 1, skv)), (win, None, [skv - sq - win + 1]),
                                (win, skv - win, range(skv - win, skv))):
            lens = None if length is None else np.array([length], np.int32)
            attended = (key <= pos) & (key > pos - w if w else True) & (key < (skv if length is None else length))
            attended[~attended.any(1)] = True
            kb, vb = k.copy(), v.copy()
            kb[:, :, list(keys)], vb[:, :, list(keys)] = bad, bad
            clean = ~attended[:, list(keys)].any(1)
            assert 0 < clean.sum() < sq
            got = gpu_sdpa(hip_backend, torch_cuda, q, kb, vb, scale, True, w, 0, lens)
            assert hip_backend.last_kernel() == "sdpa_decode_kernel"
            close(got[:, :, clean], L.sdpa(q, k, v, scale, True, w, 0, lens)[:, :, clean], rel=2e-5, abs_=2e-6)
    finally:
        hip_backend.set_tuning("sdpa_decode_one_launch", 1)


@pytest.mark.parametrize("one_launch", [1, 0])
@pytest.mark.parametrize("heads,kv_heads,d,sq,skv", [(8, 2, 128, 1, 40), (8, 2, 128, 1, 200), (4, 1, 64, 1, 1000), (6, 2, 64, 3, 200), (2, 1, 256, 5, 129), (4, 4, 128, 4, 900)])
def test_an_undefined_score_makes_the_output_undefined(hip_backend, torch_cuda, heads, kv_heads, d, sq, skv, one_launch):
    """A NaN in the K row of an attended key reaches every query that attends it, with one split of the keys and with several:
    no zeros in its place. V is finite."""
    rng = np.random.default_rng(heads * d + skv + sq)
    q = rng.standard_normal((1, heads, sq, d)).astype(np.float32)
    k = rng.standard_normal((1, kv_heads, skv, d)).astype(np.float32)
    v = rng.standard_normal((1, kv_heads, skv, d)).astype(np.float32)
    hip_backend.set_tuning("sdpa_decode_one_launch", one_launch)
    try:
        for key in (0, skv // 2, skv - sq):
            kb = k.copy()
            kb[:, :, key, 1] = np.nan
            got = gpu_sdpa(hip_backend, torch_cuda, q, kb, v, float(1 / np.sqrt(d)), True)
            assert hip_backend.last_kernel() == "sdpa_decode_kernel"
            assert np.isnan(got).all()
    finally:
        hip_backend.set_tuning("sdpa_decode_one_launch", 1)


def test_attention_prefill_config_against_torch_fp32(hip_backend, torch_cuda):
    """Prefill: seq 2048 causal, 32 / 8 heads, head_dim 128. The oracle checks a 256-long prefix problem exactly;
    the full size is compared with torch's fp32 attention on the same device (textbook softmax(QK^T)V)."""
    torch = torch_cuda
    rng = np.random.default_rng(60)
    s = 2048
    q = rng.standard_normal((1, 32, s, 128)).astype(np.float32)
    k = rng.standard_normal((1, 8, s, 128)).astype(np.float32)
    v = rng.standard_normal((1, 8, s, 128)).astype(np.float32)
    scale = float(1 / np.sqrt(128.0))
    got = gpu_sdpa(hip_backend, torch, q, k, v, scale, True)
    tq, tk, tv = dev(torch, q), dev(torch, k).repeat_interleave(4, 1), dev(torch, v).repeat_interleave(4, 1)
    sc = torch.matmul(tq, tk.transpose(-1, -2)) * scale
    sc = sc.masked_fill(~torch.ones(s, s, dtype=torch.bool, device="cuda").tril(), -1e30)
    want = torch.matmul(torch.softmax(sc, -1), tv).cpu().numpy()
    # bf16 operands: the bound is on the error against the largest output magnitude (per-element relative error of a
    # near-zero output is unbounded for any reordered or reduced-precision sum), plus an RMS bound
    err = normalized_err(got, want, eps=1.0)
    rms = float(np.sqrt(np.mean((got - want) ** 2)) / np.abs(want).max())
    print(f"prefill attention 2048: max err / max |ref| vs torch fp32 {err:.2e}, rms {rms:.2e}")
    assert err <= 2e-2 and rms <= 5e-3
    sp = 256
    qs, ks, vs = q[:, :, :sp].copy(), k[:, :, :sp].copy(), v[:, :, :sp].copy()
    want_s = L.sdpa(qs, ks, vs, scale, True)
    e_mfma = normalized_err(gpu_sdpa(hip_backend, torch, qs, ks, vs, scale, True), want_s, eps=1.0)
    assert hip_backend.last_kernel() == "sdpa_prefill_kernel"
    print(f"prefill attention 256 (matrix cores): max err / max |ref| vs oracle {e_mfma:.2e}")
    assert e_mfma <= 2e-2
    hip_backend.set_tuning("sdpa_prefill_mfma", 0)                # the fp32 kernel on the same problem, reference tolerance
    try:
        close(gpu_sdpa(hip_backend, torch, qs, ks, vs, scale, True), want_s)
    finally:
        hip_backend.set_tuning("sdpa_prefill_mfma", 1)
    # causal prefix property: the first 256 rows of the long problem are the short problem
    assert normalized_err(got[:, :, :sp], want_s, eps=1.0) <= 2e-2


@pytest.mark.parametrize("batch,heads,kv_heads,d,sq,skv,causal", [
    (1, 8, 2, 128, 200, 200, True), (2, 4, 4, 64, 97, 97, True), (1, 6, 3, 128, 64, 333, True), (1, 16, 2, 64, 130, 130, False),
    (1, 2, 1, 128, 31, 1000, True), (2, 8, 8, 64, 512, 512, True), (1, 4, 1, 128, 16, 16, True), (1, 3, 3, 128, 100, 257, False)])
def test_attention_prefill_mfma_shapes(hip_backend, torch_cuda, batch, heads, kv_heads, d, sq, skv, causal):
    """The matrix-core prompt kernel over its shape range: group sizes 1 / 2 / 4 / 8, head_dim 64 / 128, lengths that
    are not multiples of the 32-query or 64-key tiles, a query block shorter than the keys (a later prompt chunk),
    causal and full; the short ones would go to the streaming kernel, which is kept out. Bound: 2e-2 of the largest reference magnitude (bf16 operands); the RMS error is held to 5e-3."""
    rng = np.random.default_rng(sq * skv + d)
    q = rng.standard_normal((batch, heads, sq, d)).astype(np.float32)
    k = rng.standard_normal((batch, kv_heads, skv, d)).astype(np.float32)
    v = rng.standard_normal((batch, kv_heads, skv, d)).astype(np.float32)
    scale = float(1 / np.sqrt(d))
    hip_backend.set_tuning("sdpa_decode_prompts", 0)
    try:
        got = gpu_sdpa(hip_backend, torch_cuda, q, k, v, scale, causal)
        assert hip_backend.last_kernel() == "sdpa_prefill_kernel"
        # rows of P sum to 1: with v = 1 everywhere the output is 1 (bf16 P entries: 1e-2)
        assert np.abs(gpu_sdpa(hip_backend, torch_cuda, q, k, np.ones_like(v), scale, causal) - 1.0).max() <= 1e-2
    finally:
        hip_backend.set_tuning("sdpa_decode_prompts", 1)
    want = L.sdpa(q, k, v, scale, causal)
    assert np.isfinite(got).all()
    assert normalized_err(got, want, eps=1.0) <= 2e-2
    assert np.sqrt(np.mean((got - want) ** 2)) <= 5e-3 * np.abs(want).max()


@pytest.mark.parametrize("batch,heads,kv_heads,d,sq,skv,causal,window,rc,lengths", [
    (1, 1, 1, 64, 16, 16, True, 0, 0, None), (1, 3, 1, 128, 17, 17, True, 0, 0, None),       # rows that are no multiple of a workgroup's four
    (1, 8, 2, 128, 33, 97, True, 0, 0, None), (1, 2, 2, 64, 31, 400, True, 0, 0, None),      # a later chunk; keys split over workgroups
    (2, 4, 2, 64, 40, 40, True, 0, 0, [40, 7]), (3, 4, 4, 64, 20, 30, True, 10, 0, [30, 9, 0]),   # key lengths, sequences without a key
    (1, 6, 3, 128, 50, 50, False, 12, 5, None), (1, 4, 1, 64, 24, 64, False, 0, 0, None),
    (1, 1, 1, 128, 100, 900, True, 128, 0, None), (2, 2, 1, 64, 90, 90, True, 0, 0, None)])
def test_attention_short_prompts_stream_the_cache(hip_backend, torch_cuda, batch, heads, kv_heads, d, sq, skv, causal, window, rc, lengths):
    """Prompts that the streaming kernel is the faster one for: fp32 operands, so the reference's own tolerance; as token rows the same bits;
    values of excluded keys do not reach the output."""
    torch = torch_cuda
    rng = np.random.default_rng(sq * skv + d)
    q, k, v = (rng.standard_normal(s).astype(np.float32) for s in ((batch, heads, sq, d), (batch, kv_heads, skv, d), (batch, kv_heads, skv, d)))
    scale = float(1 / np.sqrt(d))
    ln = None if lengths is None else np.asarray(lengths, np.int32)
    got = gpu_sdpa(hip_backend, torch, q, k, v, scale, causal, window, rc, ln)
    assert hip_backend.last_kernel() == "sdpa_decode_kernel"
    close(got, L.sdpa(q, k, v, scale, causal, window, rc, ln))
    rows = torch.full((batch, sq, heads, d), float("nan"), device="cuda")
    hip_backend.sdpa_cache_rows_dev(*(dev(torch, a) for a in (q, k, v)), rows, batch, heads, kv_heads, sq, skv, skv, d, scale, causal, window, rc,
                                    None if ln is None else dev(torch, ln))
    assert hip_backend.last_kernel() == "sdpa_decode_kernel"
    assert np.array_equal(rows.cpu().numpy(), got.transpose(0, 2, 1, 3))
    spare = [np.full((batch, kv_heads, skv + 5, d), np.nan, np.float32) for _ in range(2)]      # rows of a cache past its keys
    spare[0][:, :, :skv], spare[1][:, :, :skv] = k, v
    out = torch.full((batch, heads, sq, d), float("nan"), device="cuda")
    hip_backend.sdpa_cache_dev(dev(torch, q), dev(torch, spare[0]), dev(torch, spare[1]), out, batch, heads, kv_heads, sq, skv, skv + 5, d, scale,
                               causal, window, rc, None if ln is None else dev(torch, ln))
    assert np.array_equal(out.cpu().numpy(), got)
    if causal and window == 0 and ln is None:
        v[:, :, -1] = np.nan                                        # the last key: only the last query's
        late = gpu_sdpa(hip_backend, torch, q, k, v, scale, causal)
        assert np.array_equal(late[:, :, :-1], got[:, :, :-1]) and np.isnan(late[:, :, -1]).all()


@pytest.mark.parametrize("heads,kv_heads,d,sq", [(4, 1, 64, 385), (8, 2, 128, 101), (8, 1, 128, 51)])
def test_attention_short_prompt_rows_share_a_workgroup_with_their_own_query_only(hip_backend, torch_cuda, heads, kv_heads, d, sq):
    """Four heads or more to a KV head: all rows of a workgroup belong to one query, so what it walks, and the order of a row's sums, do not depend on
    how many queries the call has: the last 18 alone give the same bits. Head by head, with a count of queries that four does not divide, they
    would share workgroups with other queries, and with the next head's first ones, which have no key in common with them under the window."""
    q, k, v = sdpa_inputs(1, heads, kv_heads, sq, sq + 15, d, seed=sq)
    got = gpu_sdpa(hip_backend, torch_cuda, q, k, v, 0.1, True, 60)
    assert hip_backend.last_kernel() == "sdpa_decode_kernel"
    last = gpu_sdpa(hip_backend, torch_cuda, q[:, :, -18:].copy(), k, v, 0.1, True, 60)
    assert hip_backend.last_kernel() == "sdpa_decode_kernel"
    assert np.array_equal(got[:, :, -18:], last)
    close(got, L.sdpa(q, k, v, 0.1, True, 60))


@pytest.mark.parametrize("heads,kv_heads,d,sq,skv", [(32, 8, 128, 512, 512), (8, 1, 64, 300, 2000)])
def test_attention_long_prompts_stay_on_the_matrix_cores(hip_backend, torch_cuda, heads, kv_heads, d, sq, skv):
    q, k, v = (np.zeros(s, np.float32) for s in ((1, heads, sq, d), (1, kv_heads, skv, d), (1, kv_heads, skv, d)))
    gpu_sdpa(hip_backend, torch_cuda, q, k, v, 1.0, True)
    assert hip_backend.last_kernel() == "sdpa_prefill_kernel"


@pytest.mark.parametrize("heads,kv_heads,d,sq,skv,window,streams", [
    (8, 1, 128, 16, 8192, 0, False), (8, 1, 128, 16, 32768, 0, False), (1, 1, 128, 128, 16384, 0, False), (4, 1, 128, 23, 21041, 0, False),
    (1, 1, 64, 8000, 8000, 128, False),                                   # a window: the prompt kernel walks a query group's keys, not all queries'
    (1, 1, 128, 16, 8192, 0, True), (8, 1, 64, 40, 20000, 300, True), (16, 2, 128, 60, 60, 0, True)])
def test_attention_prompts_over_long_caches_take_the_shorter_kernel(hip_backend, torch_cuda, heads, kv_heads, d, sq, skv, window, streams):
    q, k, v = (torch_cuda.zeros(s, device="cuda") for s in ((1, heads, sq, d), (1, kv_heads, skv, d), (1, kv_heads, skv, d)))
    hip_backend.sdpa_dev(q, k, v, torch_cuda.empty_like(q), 1, heads, kv_heads, sq, skv, d, 1.0, True, window)
    assert hip_backend.last_kernel() == ("sdpa_decode_kernel" if streams else "sdpa_prefill_kernel")


@pytest.mark.parametrize("batch,heads,kv_heads,d,sq,skv,causal,window,rc,lengths", [
    (1, 8, 2, 128, 300, 300, True, 64, 0, None),            # sliding window shorter than a key block ... 
    (1, 8, 2, 128, 300, 300, True, 100, 0, None),           # ... and one that straddles blocks
    (2, 4, 2, 64, 200, 200, True, 0, 0, [200, 77]),         # key lengths: the second sequence ends inside a block
    (3, 4, 4, 64, 130, 130, True, 50, 0, [130, 40, 0]),     # window + lengths: late queries of sequence 1 and all of 2 keep no key
    (1, 4, 1, 128, 96, 400, True, 128, 0, None),            # a later prompt chunk with a window
    (1, 6, 3, 128, 150, 150, False, 40, 7, None),           # bidirectional window with right context
    (2, 2, 2, 64, 64, 64, False, 0, 0, [1, 64]),            # full attention, one key
    (1, 32, 8, 128, 512, 512, True, 256, 0, None),          # the Llama-3 head shape with a 256-key window
])
def test_attention_prefill_mfma_window_and_key_lengths(hip_backend, torch_cuda, batch, heads, kv_heads, d, sq, skv, causal, window,
                                                       rc, lengths):
    """The matrix-core prompt kernel under the structured rules (sliding window, right context, per-sequence key
    lengths), including queries the rules leave without a key (equal weight on every key, as the reference's row of
    equal -1e30 scores). Against the oracle, 2e-2 of the largest reference magnitude; the fp32 kernel on the same call
    stays within the reference's own tolerance."""
    rng = np.random.default_rng(sq * skv + d + window)
    q = rng.standard_normal((batch, heads, sq, d)).astype(np.float32)
    k = rng.standard_normal((batch, kv_heads, skv, d)).astype(np.float32)
    v = rng.standard_normal((batch, kv_heads, skv, d)).astype(np.float32)
    scale = float(1 / np.sqrt(d))
    ln = None if lengths is None else np.asarray(lengths, np.int32)
    want = L.sdpa(q, k, v, scale, causal, window, rc, ln)
    try:
        for teams in (1, 2):        # one query group per workgroup; a late and an early (or two neighbouring) groups paired
            hip_backend.set_tuning("sdpa_prefill_teams", teams)
            got = gpu_sdpa(hip_backend, torch_cuda, q, k, v, scale, causal, window, rc, ln)
            assert hip_backend.last_kernel() == "sdpa_prefill_kernel"
            assert np.isfinite(got).all()
            assert normalized_err(got, want, eps=1.0) <= 2e-2
            assert np.sqrt(np.mean((got - want) ** 2)) <= 5e-3 * np.abs(want).max()
            assert np.abs(gpu_sdpa(hip_backend, torch_cuda, q, k, np.ones_like(v), scale, causal, window, rc, ln) - 1.0).max() <= 1e-2
    finally:
        hip_backend.set_tuning("sdpa_prefill_teams", 0)
    hip_backend.set_tuning("sdpa_prefill_mfma", 0)
    try:
        close(gpu_sdpa(hip_backend, torch_cuda, q, k, v, scale, causal, window, rc, ln), want)
        assert hip_backend.last_kernel() != "sdpa_prefill_kernel"
    finally:
        hip_backend.set_tuning("sdpa_prefill_mfma", 1)


@pytest.mark.parametrize("batch,heads,kv_heads,d,sq,skv,causal,window,lengths,mask_dims", [
    (2, 8, 2, 64, 200, 200, True, 0, None, (1, 1, 200, 200)),        # one bias matrix for every head (ALiBi-like), causal
    (2, 8, 2, 128, 96, 160, False, 0, [160, 70], (2, 8, 96, 160)),   # a bias per batch and head, ragged key lengths, a prompt chunk
    (1, 4, 4, 64, 130, 132, True, 48, None, (1, 4, 1, 132)),         # per-head key bias broadcast over queries, window (late queries lose keys)
    (3, 6, 3, 128, 64, 64, True, 0, [64, 10, 0], (3, 3, 64, 64)),    # a bias per KV head; sequence 2 has no key at all
    (2, 4, 2, 64, 80, 80, False, 0, None, (2, 1, 80, 1)),            # one value per query row: shifts every score of the row alike
    (1, 32, 8, 128, 512, 512, True, 0, None, (1, 1, 512, 512)),      # the Llama-3 head shape with a padding-style mask of -1e9 entries
])
def test_attention_prefill_mfma_with_an_additive_mask(hip_backend, torch_cuda, batch, heads, kv_heads, d, sq, skv, causal, window,
                                                      lengths, mask_dims):
    """The matrix-core prompt kernel with an additive mask in every broadcast form the reference accepts, alone and on
    top of the structured rules: the mask is added to every score, an excluded key's -1e30 included, so a row the rules
    leave without a key weighs the keys by its mask values' softmax only if those differ by less than fp32 resolves at
    1e30 -- i.e. equally. Against the oracle, 2e-2 of the largest reference magnitude; masks whose rows are not a
    multiple of four keys stay on the fp32 kernel."""
    rng = np.random.default_rng(sq * skv + d + mask_dims[0])
    q = rng.standard_normal((batch, heads, sq, d)).astype(np.float32)
    k = rng.standard_normal((batch, kv_heads, skv, d)).astype(np.float32)
    v = rng.standard_normal((batch, kv_heads, skv, d)).astype(np.float32)
    scale = float(1 / np.sqrt(d))
    mask = (rng.standard_normal(mask_dims) * 2).astype(np.float32)
    if mask_dims[3] > 1:
        mask[..., rng.random(mask_dims[3]) < 0.2] = -1e9              # some keys switched off for everyone, as a padding mask does
        mask[..., 0] = np.minimum(mask[..., 0], 3.0)                   # and key 0 stays available
        mask[..., 0] = np.maximum(mask[..., 0], -3.0)
    ln = None if lengths is None else np.asarray(lengths, np.int32)
    want = L.sdpa(q, k, v, scale, causal, window, 0, ln, mask)
    try:
        for teams in (1, 2):
            hip_backend.set_tuning("sdpa_prefill_teams", teams)
            got = gpu_sdpa(hip_backend, torch_cuda, q, k, v, scale, causal, window, 0, ln, mask)
            assert hip_backend.last_kernel() == "sdpa_prefill_kernel"
            assert np.isfinite(got).all()
            assert normalized_err(got, want, eps=1.0) <= 2e-2
            assert np.sqrt(np.mean((got - want) ** 2)) <= 5e-3 * np.abs(want).max()
    finally:
        hip_backend.set_tuning("sdpa_prefill_teams", 0)
    hip_backend.set_tuning("sdpa_prefill_mfma", 0)
    try:
        close(gpu_sdpa(hip_backend, torch_cuda, q, k, v, scale, causal, window, 0, ln, mask), want)
        assert hip_backend.last_kernel() != "sdpa_prefill_kernel"
    finally:
        hip_backend.set_tuning("sdpa_prefill_mfma", 1)
    if mask_dims[3] > 4:
        odd = np.ascontiguousarray(mask[..., : mask_dims[3] - 1])     # rows of skv - 1 keys: not the layout the kernel reads
        got_odd = gpu_sdpa(hip_backend, torch_cuda, q, k[:, :, : skv - 1], v[:, :, : skv - 1], scale, causal, window, 0,
                           None if ln is None else np.minimum(ln, skv - 1), odd) if sq <= skv - 1 else None
        if got_odd is not None:
            assert hip_backend.last_kernel() != "sdpa_prefill_kernel" or (skv - 1) % 4 == 0
            close(got_odd, L.sdpa(q, k[:, :, : skv - 1], v[:, :, : skv - 1], scale, causal, window, 0,
                                  None if ln is None else np.minimum(ln, skv - 1), odd))


def test_norms_softmax_and_glue(hip_backend, torch_cuda):
    torch = torch_cuda
    kx = hip_backend
    rows, cols = 5, 4096
    x = (np.random.default_rng(1).standard_normal((rows, cols)) * 3).astype(np.float32)
    g = np.random.default_rng(2).standard_normal(cols).astype(np.float32)
    bta = np.random.default_rng(3).standard_normal(cols).astype(np.float32)
    xd = x.astype(np.float64)
    out = torch.empty(rows, cols, device="cuda")
    kx.rms_norm_dev(dev(torch, x), dev(torch, g), out, rows, cols, 1e-5)
    close(out.cpu().numpy(), xd / np.sqrt((xd * xd).mean(1, keepdims=True) + 1e-5) * g, abs_=1e-4)
    ref = np.empty_like(x)
    L.oracle().orc_f32_rms_norm(L.fp(x), L.fp(g), L.fp(ref), rows, cols, 1e-5)
    close(out.cpu().numpy(), ref, rel=1e-5)
    kx.rms_norm_dev(dev(torch, x), None, out, rows, cols, 1e-5)
    close(out.cpu().numpy(), xd / np.sqrt((xd * xd).mean(1, keepdims=True) + 1e-5), abs_=1e-4)
    kx.layer_norm_dev(dev(torch, x), dev(torch, g), dev(torch, bta), out, rows, cols, 1e-5)
    mu, var = xd.mean(1, keepdims=True), xd.var(1, keepdims=True)
    close(out.cpu().numpy(), (xd - mu) / np.sqrt(var + 1e-5) * g + bta, abs_=1e-4)
    for log in (False, True):
        kx.softmax_rows_dev(dev(torch, x), out, rows, cols, log)
        want = np.empty_like(x)
        L.oracle().orc_f32_softmax_rows(L.fp(x), L.fp(want), rows, cols, int(log))
        close(out.cpu().numpy(), want, rel=1e-5, abs_=1e-6)
    n = 14336 * 3 + 5
    a = np.random.default_rng(4).standard_normal(n).astype(np.float32) * 4
    b = np.random.default_rng(5).standard_normal(n).astype(np.float32)
    o = torch.empty(n, device="cuda")
    kx.silu_mul_dev(dev(torch, a), dev(torch, b), o, n)
    ad = a.astype(np.float64)
    close(o.cpu().numpy(), ad * (1 / (1 + np.exp(-ad))) * b, rel=1e-6, abs_=1e-6)
    if L.ref() is not None:   # the reference's silu (f32_ops.c) then its multiply
        s = np.empty_like(a)
        L.ref().skainet_f32_unary(2, L.fp(a), L.fp(s), n)
        close(o.cpu().numpy(), s * b, rel=1e-6, abs_=1e-6)
    kx.add_dev(dev(torch, a), dev(torch, b), o, n)
    assert np.array_equal(o.cpu().numpy(), a + b)
    # arg-max: first maximum wins (TensorOps.argMax)
    lg = np.random.default_rng(6).standard_normal((4, 128256)).astype(np.float32)
    lg[1, 77] = lg[1, 90000] = 50.0
    lg[2, :] = -3.0
    lg[3, 128255] = 60.0
    idx = torch.empty(4, dtype=torch.int32, device="cuda")
    kx.argmax_rows_dev(dev(torch, lg), 4, 128256, idx)
    assert idx.cpu().tolist() == [int(lg[0].argmax()), 77, 0, 128255]
    # SPI kernels on host arrays
    norm, soft = kx.HipKernelProvider().norm_fp32(), kx.HipKernelProvider().softmax_fp32()
    ho = np.zeros((rows + 1, cols), np.float32)
    norm.rms_norm(x, cols, g, ho, cols, rows - 1, cols, 1e-5)     # offsets: skip the first row of both
    close(ho[1:rows], ref[1:rows], rel=1e-5)
    assert not ho[0].any() and not ho[rows].any()
    norm.layer_norm(x, 0, None, None, ho, 0, rows, cols, 1e-5)
    close(ho[:rows], (xd - mu) / np.sqrt(var + 1e-5), abs_=1e-4)
    soft.softmax_rows(x, 0, ho, 0, rows, cols, False)
    close(ho[:rows].sum(1), np.ones(rows), rel=1e-5)


@pytest.mark.parametrize("rows,cols", [(1, 8192), (3, 4099), (2, 100), (7, 6144), (1, 12288)])
def test_rms_norm_row_shapes(hip_backend, torch_cuda, rows, cols):
    """Register-cached rows (cols % 4 == 0 up to 8192) and the looping kernel (everything else) against the oracle."""
    torch, kx = torch_cuda, hip_backend
    x = (np.random.default_rng(cols).standard_normal((rows, cols)) * 2).astype(np.float32)
    g = np.random.default_rng(cols + 1).standard_normal(cols).astype(np.float32)
    out = torch.empty(rows, cols, device="cuda")
    kx.rms_norm_dev(dev(torch, x), dev(torch, g), out, rows, cols, 1e-6)
    ref = np.empty_like(x)
    L.oracle().orc_f32_rms_norm(L.fp(x), L.fp(g), L.fp(ref), rows, cols, 1e-6)
    close(out.cpu().numpy(), ref, rel=2e-5, abs_=1e-6)


@pytest.mark.parametrize("rows,cols", [(1, 16384), (64, 20000), (65, 20000), (2, 16383), (3, 128256)])
def test_argmax_split_and_single_kernels(hip_backend, torch_cuda, rows, cols):
    """Few long rows take the many-workgroups-per-row kernel (twice in a row: its counters must come back to zero),
    other shapes the one-workgroup-per-row kernel; ties keep the lowest index, also across slice borders."""
    torch, kx = torch_cuda, hip_backend
    lg = np.random.default_rng(rows * cols).standard_normal((rows, cols)).astype(np.float32)
    lg[0, cols - 1] = lg[0, cols // 2] = 40.0          # tie in two different slices
    if rows > 1:
        lg[1, :] = 1.5                                  # all equal: index 0
    idx = torch.full((rows,), -1, dtype=torch.int32, device="cuda")
    want = [int(r.argmax()) for r in lg]
    assert want[0] == cols // 2
    d = dev(torch, lg)
    for _ in range(2):
        idx.fill_(-1)
        kx.argmax_rows_dev(d, rows, cols, idx)
        assert idx.cpu().tolist() == want


def test_dense_matmuls(hip_backend, torch_cuda):
    prov = hip_backend.HipKernelProvider()
    # capability answers of KernelProvider.supports (KernelProvider.kt:161-190)
    for op in ("softmax", "layer_norm", "rms_norm", "sdpa"):
        assert prov.supports(op, ["Float32"]) and not prov.supports(op, ["Float16"])
    assert prov.supports("matmul_wt", ["Float32", "Float32"]) and not prov.supports("matmul_wt", ["Float32", "Q4_K"])
    assert not prov.supports("matmul", ["Float16", "Float32"]) and not prov.supports("matmul", ["Float32", "Q3_K"])
    assert not prov.supports("gather", ["Float32"]) and not prov.supports("matmul", ["Float32"])
    rng = np.random.default_rng(9)
    a = rng.standard_normal((70, 130)).astype(np.float32)
    b = rng.standard_normal((130, 90)).astype(np.float32)
    c = np.full((70, 100), 3.0, np.float32)
    # strided views: A rows 2.., 100 of 130 columns; C written into a wider matrix at an offset
    prov.matmul_fp32().matmul(a, 2 * 130 + 5, 130, b, 7, 90, c, 100 + 4, 100, 60, 80, 100)
    bb = np.lib.stride_tricks.as_strided(b.reshape(-1)[7:], (100, 80), (360, 4))
    want = a[2:62, 5:105].astype(np.float64) @ bb
    close(c[1:61, 4:84], want, rel=1e-5, abs_=1e-4)
    assert (c[0] == 3).all() and (c[1:61, :4] == 3).all() and (c[1:61, 84:] == 3).all() and (c[61:] == 3).all()
    ref = np.full((70, 100), 3.0, np.float32)
    L.oracle().orc_fp32_matmul(L.fp(a), 2 * 130 + 5, 130, L.fp(b), 7, 90, L.fp(ref), 104, 100, 60, 80, 100)
    close(c, ref, rel=1e-5, abs_=1e-4)
    z = np.full((4, 6), 9.0, np.float32)
    prov.matmul_fp32().matmul(a, 0, 130, b, 0, 90, z, 0, 6, 4, 6, 0)     # k == 0 zeroes C
    assert not z.any()
    w = rng.standard_normal((33, 130)).astype(np.float32)
    o = np.zeros((70, 33), np.float32)
    prov.matmul_fp32_wt().matmul_wt(a, 0, w, 0, o, 0, 70, 33, 130)
    close(o, a.astype(np.float64) @ w.T, rel=1e-5, abs_=1e-4)


@pytest.mark.parametrize("m,n,k,wt", [(512, 1024, 768, False), (200, 300, 260, False), (64, 32, 4, True), (130, 4096, 516, True),
                                      (1000, 132, 2048, False), (65, 257, 100, True), (1030, 2052, 100, True), (1030, 2052, 36, False),
                                      (2100, 2100, 20, True), (2100, 2100, 132, False), (232, 7124, 20, True), (232, 7124, 36, True), (948, 1164, 32, False), (500, 1284, 28, False),
                                      (948, 1164, 36, False)])
def test_dense_fp32_matmul_on_the_matrix_cores(hip_backend, torch_cuda, m, n, k, wt):
    """fp32 operands on the fp32 matrix instruction (exact products, fp32 accumulation in the instruction's order):
    resident operands through the device entries, ragged tiles in every direction, K from one instruction step to many
    slices, both layouts of B: shapes whose 64 x 128 tiles leave CUs idle run the kernel that splits K over waves, the others
    64- or 128-row tiles; against fp64 and against the tile kernel that takes the same call when the matrix-core
    ones are switched off. Products whose strides or alignment the matrix-core kernel does not read stay on the tile
    kernel."""
    torch = torch_cuda
    rng = np.random.default_rng(m + n + k)
    a = rng.standard_normal((m, k)).astype(np.float32)
    b = rng.standard_normal((n, k) if wt else (k, n)).astype(np.float32)
    want = a.astype(np.float64) @ (b.astype(np.float64).T if wt else b.astype(np.float64))

    def run():
        out = torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda")
        if wt:
            hip_backend.fp32_matmul_wt_dev(dev(torch, a), 0, dev(torch, b), 0, out, 0, m, n, k)
        else:
            hip_backend.fp32_matmul_dev(dev(torch, a), 0, k, dev(torch, b), 0, n, out, 0, n, m, n, k)
        return out.cpu().numpy()

    got = run()
    tiles, cus = -(-m // 64) * -(-n // 128), torch.cuda.get_device_properties(0).multi_processor_count
    few = tiles < cus and not (k <= 32 and tiles * (4 if k < 32 else 2) >= cus)          # a K of one step is not split
    assert hip_backend.last_kernel() == ("sgemm_mfma_skinny_kernel" if few else "sgemm_mfma_kernel")
    close(got, want, rel=1e-5, abs_=2e-6 * np.sqrt(k) * 16)
    try:
        hip_backend.set_tuning("dense_mfma", 0)
        tile = run()
        assert hip_backend.last_kernel() == "sgemm_kernel"
    finally:
        hip_backend.set_tuning("dense_mfma", 1)
    close(got, tile, rel=1e-5, abs_=2e-6 * np.sqrt(k) * 16)
    if not wt:
        # the same product out of a wider A at an offset of one float: not 16-byte aligned, the tile kernel's business
        wide = np.zeros((m, k + 4), np.float32)
        wide[:, 1:k + 1] = a
        out = torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda")
        hip_backend.fp32_matmul_dev(dev(torch, wide), 1, k + 4, dev(torch, b), 0, n, out, 0, n, m, n, k)
        assert hip_backend.last_kernel() == "sgemm_kernel"
        close(out.cpu().numpy(), want, rel=1e-5, abs_=2e-6 * np.sqrt(k) * 16)


@pytest.mark.parametrize("wt", [True, False])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (1, 17, 31), (3, 16, 32), (16, 33, 33), (17, 100, 2047), (33, 4100, 65), (64, 8200, 96),
                                   (65, 5, 8192), (130, 4097, 161)])
def test_dense_fp32_products_with_k_split_over_waves(hip_backend, torch_cuda, m, n, k, wt):
    """Few rows or few columns: K is split over the waves of a workgroup, at every tile size (1, 2, 4 row tiles, 1 or 2
    column tiles), with partial last steps of K, ragged edges and rows that are not 16-byte aligned. An fp32 sum of k
    products in any order is within k * 2^-24 of the sum of magnitudes (about 0.8^2 k for N(0, 1) operands); the written
    bound takes a quarter of that worst case."""
    torch = torch_cuda
    rng = np.random.default_rng(7 * m + n + k)
    a = rng.standard_normal((m, k)).astype(np.float32)
    b = rng.standard_normal((n, k) if wt else (k, n)).astype(np.float32)
    want = a.astype(np.float64) @ (b.astype(np.float64).T if wt else b.astype(np.float64))
    out = torch.full((m + 1, n), float("nan"), dtype=torch.float32, device="cuda")
    if wt:
        hip_backend.fp32_matmul_wt_dev(dev(torch, a), 0, dev(torch, b), 0, out, 0, m, n, k)
    else:
        hip_backend.fp32_matmul_dev(dev(torch, a), 0, k, dev(torch, b), 0, n, out, 0, n, m, n, k)
    if wt or m < 64:                                    # unaligned rows of B at 64 rows and more stay on the tile kernel
        assert hip_backend.last_kernel() == "sgemm_mfma_skinny_kernel"
    got = out.cpu().numpy()
    assert np.isnan(got[m]).all()                       # nothing past the last row
    assert np.abs(got[:m] - want).max() <= max(1, k / 4) * 2.0 ** -24 * 0.64 * k + 1e-6


@pytest.mark.parametrize("kind,codec", [("bf16", "BFloat16"), ("fp16", "Float16")])
def test_narrow_float_matmuls(hip_backend, torch_cuda, kind, codec):
    """Bf16MatmulKernel / Fp16MatmulKernel through the host entry: the oracle on the recorded inputs (with the formats'
    specials), then a ragged larger product with offsets, an odd byte offset and a padded byte row stride for B."""
    from test_oracle_golden import narrow_inputs, narrow_values
    prov = hip_backend.HipKernelProvider()
    kern = prov.matmul_bf16() if kind == "bf16" else prov.matmul_fp16()
    assert kern.codec == codec and prov.supports("matmul", ["Float32", codec])
    a, b, m, n, k = narrow_inputs(kind)
    c = np.full((m, n), np.nan, np.float32)
    kern.matmul(a, 0, k, b, 0, 2 * n, c, 0, n, m, n, k)
    want = L.narrow_matmul(kind, a, b, m, n, k)
    close(c, want.astype(np.float64), rel=1e-5, abs_=1e-6)
    recorded = np.load(os.path.join(HERE, "golden", "ref_vectors.npz"))[f"narrow/{kind}"]
    close(c, recorded.astype(np.float64), rel=1e-5, abs_=1e-6)
    # 70 x 83 x 150 out of wider buffers; B starts at an odd byte and its rows are 2 * 90 + 6 bytes apart
    rng = np.random.default_rng(12)
    m, n, k = 70, 83, 150
    a = rng.standard_normal((m + 2, k + 9)).astype(np.float32)
    bv = rng.standard_normal((k, n)).astype(np.float32)
    bits = (bv.view(np.uint32) >> 16).astype("<u2") if kind == "bf16" else bv.astype("<f2").view("<u2")
    stride = 2 * 90 + 6
    raw = np.full(3 + k * stride, 0xA5, np.uint8)
    rows = np.lib.stride_tricks.as_strided(raw[3:], (k, 2 * n), (stride, 1))
    rows[:] = np.ascontiguousarray(bits).view(np.uint8).reshape(k, 2 * n)
    c = np.full((m + 1, n + 5), 3.0, np.float32)
    kern.matmul(a, 2 * (k + 9) + 4, k + 9, raw, 3, stride, c, (n + 5) + 2, n + 5, m, n, k)
    want = a[2:, 4:4 + k].astype(np.float64) @ narrow_values(kind, np.ascontiguousarray(bits).view(np.uint8).reshape(-1), k, n).astype(np.float64)
    close(c[1:, 2:2 + n], want, rel=1e-5, abs_=1e-5)
    assert (c[0] == 3).all() and (c[:, :2] == 3).all() and (c[:, 2 + n:] == 3).all()
    ref = np.full_like(c, 3.0)
    getattr(L.oracle(), f"orc_{kind}_matmul")(L.fp(a), 2 * (k + 9) + 4, k + 9, L.u8(raw), 3, stride, L.fp(ref), (n + 5) + 2, n + 5, m, n, k)
    close(c, ref.astype(np.float64), rel=1e-5, abs_=1e-5)
    z = np.full((4, 6), 9.0, np.float32)
    kern.matmul(a, 0, k + 9, raw, 0, stride, z, 0, 6, 4, 6, 0)              # k == 0 zeroes C
    assert not z.any()
    with pytest.raises(ValueError):
        kern.matmul(a, 0, k + 9, raw, 0, stride, z, 0, 6, 4, 6, -1)


def test_thread_release_frees_and_regrows_scratch(hip_backend, torch_cuda):
    """A worker thread's scratch can be handed back (skainet_hip_thread_release); calls after it allocate afresh and
    give the same bits, and the memory the thread held is free again."""
    import threading
    from oracle import golden as G
    torch = torch_cuda
    provider = hip_backend.HipKernelProvider()
    n, nblocks = 96, 4
    k = nblocks * 256
    blocks = G.weight_blocks("Q4_K", n, nblocks, 0x5EED0700)
    x = G.floats(k, 0x5EED0701)
    want = L.gemv("Q4_K", x, G.row_major(blocks), n)
    b, h, hkv, skv, d = 2, 8, 2, 300, 64           # decode shape: split partials live in the thread's workspace
    q, kk, vv = sdpa_inputs(b, h, hkv, 1, skv, d, 31)
    results, errors = {}, []

    def worker():
        try:
            kernel = provider.matmul_q4k()
            att = provider.attention_fp32()
            for tag in ("before", "after"):
                y = np.zeros(n, np.float32)
                kernel.matmul_row_major(x, 0, G.row_major(blocks), 0, k, n, y, 0)
                o = np.zeros(b * h * d, np.float32)
                att.sdpa(q, kk, vv, o, b, h, hkv, 1, skv, d, 0.125, True, 0, 0)
                big = np.ones((4096, 4096), np.float32)              # 64 MiB staged on the device by the host-pointer entry
                provider.norm_fp32().rms_norm(big, 0, np.ones(4096, np.float32), np.empty_like(big), 0, 4096, 4096, 1e-5)
                results[tag] = (y, o)
                if tag == "before":
                    hip_backend.sync()
                    held = torch.cuda.mem_get_info()[0]
                    hip_backend.thread_release()
                    results["freed"] = torch.cuda.mem_get_info()[0] - held
            hip_backend.thread_release()
            hip_backend.thread_release()                              # idempotent
        except Exception as e:                                        # surfaced in the main thread below
            errors.append(e)

    t = threading.Thread(target=worker)
    t.start()
    t.join()
    assert not errors, errors
    assert normalized_err(results["before"][0], want) <= 1e-3
    assert np.array_equal(results["before"][0], results["after"][0])
    assert np.array_equal(results["before"][1], results["after"][1])
    assert results["freed"] >= 64 << 20, results["freed"]


@pytest.mark.parametrize("batch,heads,kv_heads,d,sq,skv,causal,window,rc,lengths,mask_dims", [
    (1, 8, 2, 128, 17, 700, True, 0, 0, None, None),                  # a chunk of a long prompt: one ragged query group
    (1, 2, 2, 64, 300, 300, True, 0, 0, None, None),                  # early groups have fewer blocks than there are splits
    (2, 6, 3, 64, 64, 513, False, 0, 0, [513, 70], None),             # one key in the last block; a sequence whose keys end in the first split
    (1, 4, 1, 128, 40, 640, True, 100, 3, None, None),                # a window inside two or three blocks
    (3, 4, 4, 64, 130, 130, True, 50, 0, [130, 40, 0], None),         # queries without a key: every key equally, over all splits
    (2, 4, 2, 128, 33, 260, True, 0, 0, [260, 0], (2, 4, 33, 260)),   # an additive mask, -1e30 + mask where no key is left
])
def test_attention_prefill_with_the_keys_split_over_workgroups(hip_backend, torch_cuda, batch, heads, kv_heads, d, sq, skv, causal, window,
                                                               rc, lengths, mask_dims):
    """Several workgroups share a query group's keys and a second launch merges their outputs: 2, 3 and as many splits as there
    are blocks, against the oracle at the bounds of the unsplit kernel, and as token rows against the same call unsplit (weights
    are rounded to bf16 against another running maximum: 2^-8 of a convex combination of values, at most the largest one)."""
    rng = np.random.default_rng(sq * skv + d)
    q = rng.standard_normal((batch, heads, sq, d)).astype(np.float32)
    k = rng.standard_normal((batch, kv_heads, skv, d)).astype(np.float32)
    v = rng.standard_normal((batch, kv_heads, skv, d)).astype(np.float32)
    scale = float(1 / np.sqrt(d))
    ln = None if lengths is None else np.asarray(lengths, np.int32)
    mask = None if mask_dims is None else (rng.standard_normal(mask_dims) * 2).astype(np.float32)
    want = L.sdpa(q, k, v, scale, causal, window, rc, ln, mask)
    try:
        hip_backend.set_tuning("sdpa_prefill_teams", 1)
        for splits in (1, 2, 3, 32):
            hip_backend.set_tuning("sdpa_prefill_splits", splits)
            got = gpu_sdpa(hip_backend, torch_cuda, q, k, v, scale, causal, window, rc, ln, mask)
            assert hip_backend.last_kernel() == "sdpa_prefill_kernel"
            assert np.isfinite(got).all()
            assert normalized_err(got, want, eps=1.0) <= 2e-2
            assert np.sqrt(np.mean((got - want) ** 2)) <= 5e-3 * np.abs(want).max()
            ones = gpu_sdpa(hip_backend, torch_cuda, q, k, np.ones_like(v), scale, causal, window, rc, ln, mask)
            assert np.abs(ones - 1.0).max() <= 1e-2
            if ln is None and mask is None and rc == 0 and batch == 1:
                t = [dev(torch_cuda, a) for a in (q, k, v)]
                rows = torch_cuda.full((sq, heads, d), float("nan"), device="cuda")
                hip_backend.sdpa_cache_rows_dev(*t, rows, 1, heads, kv_heads, sq, skv, skv, d, scale, causal, window)
                assert np.array_equal(rows.cpu().numpy(), got[0].transpose(1, 0, 2))
    finally:
        hip_backend.set_tuning("sdpa_prefill_teams", 0)
        hip_backend.set_tuning("sdpa_prefill_splits", 0)


@pytest.mark.parametrize("heads,kv_heads,d,sq,skv,slope,splits", [
    (4, 1, 128, 96, 96, 100.0, 1), (4, 1, 128, 96, 96, -100.0, 1), (2, 1, 64, 70, 90, 8.0, 1), (1, 1, 64, 70, 90, -100.0, 1), (4, 2, 128, 40, 90, 100.0, 2)])
def test_attention_prefill_reference_point_moves(hip_backend, torch_cuda, heads, kv_heads, d, sq, skv, slope, splits):
    """Scores that rise or fall by `slope` from key to key, into the thousands: the reference point of the exponentials moves in every
    half block (rising), is large (taken off behind the products, not inside them) or stays at the first key's (falling), and the two
    teams' states and the splits differ by thousands. A query's weight is all on its last (first) key but for e^-7.9 at the smallest
    slope (multiples of 8 up to 712 are bf16 values, the factor log2 e is rounded by at most 2^-8 for all keys alike; at 100 the keys'
    rounding, 2^-9 of 9600, leaves a gap of more than 60), so the output is that key's V: bound 2^-8 for bf16's rounding of V and P,
    plus e^-7.9 / (1 - e^-7.9) of the largest difference of two values."""
    rng = np.random.default_rng(skv)
    q = np.zeros((1, heads, sq, d), np.float32)
    q[..., 0] = 1.0
    k = np.zeros((1, kv_heads, skv, d), np.float32)
    k[..., 0] = slope * np.arange(skv)
    v = rng.standard_normal((1, kv_heads, skv, d)).astype(np.float32)
    try:
        hip_backend.set_tuning("sdpa_prefill_teams", 1)
        hip_backend.set_tuning("sdpa_prefill_splits", splits)
        got = gpu_sdpa(hip_backend, torch_cuda, q, k, v, 1.0, True)
        assert hip_backend.last_kernel() == "sdpa_prefill_kernel"
    finally:
        hip_backend.set_tuning("sdpa_prefill_teams", 0)
        hip_backend.set_tuning("sdpa_prefill_splits", 0)
    at = np.arange(sq) + skv - sq if slope > 0 else np.zeros(sq, np.int64)
    want = np.repeat(v[:, :, at], heads // kv_heads, axis=1)
    bound = 2.0 ** -8 + (0.0 if abs(slope) > 50 else 2 * np.exp(-7.9) / (1 - np.exp(-7.9)))
    assert np.abs(got - want).max() <= bound * np.abs(v).max()


@pytest.mark.parametrize("d,sq,skv,causal,window,mask_dims,splits", [
    (64, 200, 456, True, 100, (1, 1, 200, 456), 1), (128, 96, 520, True, 0, (1, 4, 1, 520), 1), (128, 130, 388, False, 64, (1, 2, 130, 1), 1),
    (64, 40, 324, True, 0, (1, 1, 40, 324), 3), (128, 33, 68, True, 0, (1, 1, 33, 68), 1), (64, 20, 1030, True, 0, (1, 1, 1, 1), 2)])
def test_attention_prefill_mask_over_blocks_of_every_kind(hip_backend, torch_cuda, d, sq, skv, causal, window, mask_dims, splits):
    """Blocks of keys that every query of a wave attends, that some do and that none does, one to six of them per team, the last one
    part empty: the mask is added in each, whose values a wave requests a block ahead. Against the oracle, bounds as above."""
    rng = np.random.default_rng(sq + skv)
    q = rng.standard_normal((1, 4, sq, d)).astype(np.float32)
    k, v = (rng.standard_normal((1, 2, skv, d)).astype(np.float32) for _ in range(2))
    mask = (rng.standard_normal(mask_dims) * 2).astype(np.float32)
    try:
        hip_backend.set_tuning("sdpa_prefill_teams", 1)
        hip_backend.set_tuning("sdpa_prefill_splits", splits)
        got = gpu_sdpa(hip_backend, torch_cuda, q, k, v, d ** -0.5, causal, window, 0, None, mask)
        assert hip_backend.last_kernel() == "sdpa_prefill_kernel"
    finally:
        hip_backend.set_tuning("sdpa_prefill_teams", 0)
        hip_backend.set_tuning("sdpa_prefill_splits", 0)
    want = L.sdpa(q, k, v, d ** -0.5, causal, window, 0, None, mask)
    assert normalized_err(got, want, eps=1.0) <= 2e-2
    assert np.sqrt(np.mean((got - want) ** 2)) <= 5e-3 * np.abs(want).max()


@pytest.mark.parametrize("d,heads,kv_heads,sq,skv,causal,window", [(128, 1, 1, 64, 2048, True, 128), (64, 4, 1, 96, 752, True, 0)])
def test_attention_prefill_splits_the_keys_that_a_masked_call_walks(hip_backend, torch_cuda, d, heads, kv_heads, sq, skv, causal, window):
    """A mask is added to excluded keys' scores too, so every key is walked: many workgroups share them where few query groups leave CUs
    idle, also under a window that without a mask would leave a fraction of the keys."""
    torch = torch_cuda
    g = torch.Generator(device="cuda").manual_seed(skv)
    q, k, v, mask = (torch.randn(s, generator=g, device="cuda") for s in ((1, heads, sq, d), (1, kv_heads, skv, d), (1, kv_heads, skv, d), (1, 1, sq, skv)))
    out = torch.full_like(q, float("nan"))
    ran = launches(torch, lambda: hip_backend.sdpa_dev(q, k, v, out, 1, heads, kv_heads, sq, skv, d, d ** -0.5, causal, window, 0, None, mask, (1, 1, sq, skv)))
    assert ["kv_to_fragments_kernel" in ran[0][0], f"sdpa_prefill_kernel<{d}, true, true>" in ran[1][0], "sdpa_prefill_merge_kernel" in ran[2][0]] == [True] * 3, ran
    blocks = -(-skv // 64)
    assert ran[1][1][2] >= blocks // 6                                     # at most six blocks each
    want = L.sdpa(*(t.cpu().numpy() for t in (q, k, v)), d ** -0.5, causal, window, 0, None, mask.cpu().numpy())
    assert normalized_err(out.cpu().numpy(), want, eps=1.0) <= 2e-2


def test_attention_prefill_workgroup_with_three_query_groups(hip_backend, torch_cuda):
    """As many workgroups as CUs, each with its share of the query groups one after the other: three turns at the most, the last
    of them for one workgroup of two only, rows past the end in the last group."""
    rng = np.random.default_rng(3)
    b, h, sq, d = 16, 8, 520, 64
    q, k, v = (rng.standard_normal((b, h, sq, d)).astype(np.float32) for _ in range(3))
    got = gpu_sdpa(hip_backend, torch_cuda, q, k, v, 0.125, True)
    assert hip_backend.last_kernel() == "sdpa_prefill_kernel"
    want = L.sdpa(q, k, v, 0.125, True)
    assert normalized_err(got, want, eps=1.0) <= 2e-2
    assert np.sqrt(np.mean((got - want) ** 2)) <= 5e-3 * np.abs(want).max()


@pytest.mark.parametrize("m,n,k,offset", [
    (1, 20, 512, 0), (3, 33, 545, 0), (16, 16, 8192, 0), (5, 1000, 1500, 3),            # sixteen waves: one step each, a tail, many, an odd base
    (20, 4100, 1028, 0), (18, 4099, 2053, 0), (2, 4200, 1028, 0), (2, 4200, 2049, 0),   # eight waves, two row tiles and one
    (2, 4200, 2047, 0),                                                                 # an element short of eight unaligned steps: the straight kernel
    (1, 8200, 516, 0), (33, 4160, 2052, 0), (64, 8200, 2080, 0), (70, 8210, 2051, 0)])  # four waves; four row tiles, one and two column tiles
def test_dense_fp32_products_staged_through_lds(hip_backend, torch_cuda, m, n, k, offset):
    """Few rows with enough K per wave: operands come in through LDS, 16 or 4 bytes a lane by their alignment, in two to four stages,
    with partial last steps, rows and columns past the end and a row of another buffer behind the last. `last_kernel` names both
    forms alike: the tracer tells which ran."""
    torch = torch_cuda
    rng = np.random.default_rng(m + n + k)
    a = rng.standard_normal((m, k)).astype(np.float32)
    b = rng.standard_normal((n, k)).astype(np.float32)
    want = a.astype(np.float64) @ b.astype(np.float64).T
    flat = np.full(offset + n * k + k, np.nan, np.float32)
    flat[offset:offset + n * k] = b.reshape(-1)
    out = torch.full((m + 1, n), float("nan"), dtype=torch.float32, device="cuda")
    da, db = dev(torch, a), dev(torch, flat)
    ran = launches(torch, lambda: hip_backend.fp32_matmul_wt_dev(da, 0, db, offset, out, 0, m, n, k))
    assert hip_backend.last_kernel() == "sgemm_mfma_skinny_kernel" and len(ran) == 1, ran
    assert ("sgemm_mfma_skinny_lds_kernel<" if k != 2047 else "sgemm_mfma_skinny_kernel<true, 1, 1, 8>") in ran[0][0], ran
    got = out.cpu().numpy()
    assert np.isnan(got[m]).all()
    # an fp32 chain of K / shares products and then the shares, each step rounding by at most 2^-24 of the sum of magnitudes
    shares = ran[0][2][0] // 64 * (2 if "<4, 2, 4, 3, 4, 2>" in ran[0][0] else 1)
    magnitude = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64).T
    assert (np.abs(got[:m] - want) <= (-(-k // shares) + 32 + shares) * 2.0 ** -24 * magnitude).all()


@pytest.mark.parametrize("m,n,k", [(48, 8200, 2080), (33, 16300, 4260), (64, 8208, 4128), (48, 9000, 4491)])
def test_dense_fp32_products_of_eight_tiles_keep_their_eight_shares_of_k(hip_backend, torch_cuda, m, n, k):
    """Four by two tiles on 256 to 511 workgroups: K in eight shares whether the operands come through LDS (W^T) or straight from memory
    (the same values as a [k, n] operand), the last, partial step in a share of the first four or the last four: the same bits."""
    torch = torch_cuda
    rng = np.random.default_rng(m + n + k)
    a = dev(torch, rng.standard_normal((m, k)).astype(np.float32))
    b = dev(torch, rng.standard_normal((n, k)).astype(np.float32))
    bt = b.t().contiguous()
    out, straight = (torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda") for _ in range(2))
    hip_backend.fp32_matmul_wt_dev(a, 0, b, 0, out, 0, m, n, k)
    hip_backend.fp32_matmul_dev(a, 0, k, bt, 0, n, straight, 0, n, m, n, k)
    assert torch.equal(out.view(torch.int32), straight.view(torch.int32))


@pytest.mark.parametrize("m,n,k,staged", [
    (129, 8301, 1199, False), (129, 8300, 1200, True), (129, 8301, 1789, False), (129, 8301, 1793, True),      # four waves: from 14 steps, 16-byte rows from 8
    (48, 9000, 4491, False), (48, 9000, 4492, True)])                                                          # eight waves: 16-byte rows alone
def test_dense_fp32_products_of_eight_tiles_go_through_lds_where_that_is_faster(hip_backend, torch_cuda, m, n, k, staged):
    """Rows that are not 16-byte aligned take four times the loads: on both sides of the rule's lines, against float64 (an fp32 chain of at most
    k / 4 products and the partial sums, each rounding 2^-24 of the sum of magnitudes so far; a quarter of that worst case)."""
    torch = torch_cuda
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, b = torch.randn(m, k, generator=g, device="cuda"), torch.randn(n, k, generator=g, device="cuda")
    out = torch.full((m, n), float("nan"), device="cuda")
    ran = launches(torch, lambda: hip_backend.fp32_matmul_wt_dev(a, 0, b, 0, out, 0, m, n, k))
    assert len(ran) == 1 and ("sgemm_mfma_skinny_lds_kernel<4, 2, 4," if staged else "sgemm_mfma_skinny_kernel<true, 4, 2,") in ran[0][0], ran
    magnitude = a.double().abs() @ b.double().abs().T
    assert bool(((out.double() - a.double() @ b.double().T).abs() <= k / 16 * 2.0 ** -24 * magnitude).all())


@pytest.mark.parametrize("rows,cols", [(3, 1), (2, 3), (5, 4), (1, 1023), (2, 1024), (1, 1025), (3, 4095), (2, 4096), (1, 8191), (2, 8192), (1, 8193)])
def test_layer_norm_and_softmax_row_shapes(hip_backend, torch_cuda, rows, cols):
    """Every form of the kernels that keep a row in registers (4, 16 and 32 elements per thread, float4s and single floats) and the looping
    ones behind them, at the edges of their ranges, with and without gamma and beta, a row of -inf but for one element, log form:
    against float64 (a sum of cols fp32 terms in a tree: within 16 * 2^-24 of the magnitudes that enter it)."""
    torch, kx = torch_cuda, hip_backend
    rng = np.random.default_rng(cols)
    x = (rng.standard_normal((rows, cols)) * 2 + 0.5).astype(np.float32)
    g, b = (rng.standard_normal(cols).astype(np.float32) for _ in range(2))
    xd = x.astype(np.float64)
    mu, var = xd.mean(1, keepdims=True), xd.var(1, keepdims=True)
    norm = (xd - mu) / np.sqrt(var + 1e-5)
    out = torch.full((rows + 1, cols), float("nan"), device="cuda")
    for gamma, beta in ((g, b), (None, b), (g, None), (None, None)):
        kx.layer_norm_dev(dev(torch, x), None if gamma is None else dev(torch, gamma), None if beta is None else dev(torch, beta), out, rows, cols, 1e-5)
        want = norm * (1 if gamma is None else gamma) + (0 if beta is None else beta)
        got = out.cpu().numpy()
        # the difference x - mean carries 2^-24 of |x| and of the mean, scaled up where a row's values lie close together
        assert np.abs(got[:rows] - want).max() <= 16 * 2.0 ** -24 * (np.abs(x).max() / np.sqrt(var.min() + 1e-5) + 1) * 8
        assert np.isnan(got[rows]).all()
    x[0, :] = -np.inf
    x[0, cols // 2] = 3.0
    xd = x.astype(np.float64)
    e = np.exp(xd - xd.max(1, keepdims=True))
    for log in (False, True):
        out.fill_(float("nan"))
        kx.softmax_rows_dev(dev(torch, x), out, rows, cols, log)
        got = out.cpu().numpy()
        assert np.isnan(got[rows]).all()
        if log:
            want = xd - (np.log(e.sum(1, keepdims=True)) + xd.max(1, keepdims=True))
            assert np.array_equal(np.isneginf(got[:rows]), np.isneginf(want))
            fin = np.isfinite(want)
            close(got[:rows][fin], want[fin], rel=1e-5, abs_=1e-5)
        else:
            close(got[:rows], e / e.sum(1, keepdims=True), rel=1e-5, abs_=1e-7)


@pytest.mark.parametrize("batch,heads,kv_heads,sq,skv,dim,window", [(3, 8, 2, 8, 3815, 128, 0), (7, 8, 1, 1, 2600, 128, 0), (6, 16, 2, 1, 4556, 64, 0), (7, 12, 3, 1, 1500, 256, 0),
                                                                    (4, 10, 2, 3, 3591, 128, 0), (12, 64, 8, 1, 4775, 128, 360)])
def test_attention_groups_of_one_die_give_the_same_bits(hip_backend, torch_cuda, batch, heads, kv_heads, sq, skv, dim, window):
    """Where the workgroups that share keys are placed on one die each (enough traffic, several groups of rows per KV head): the
    same splits by the same workgroups, so the outputs of the plain grid bit for bit, with a count of workgroups that eight does not
    divide and with key counts on the device, one of them zero."""
    torch, kx = torch_cuda, hip_backend
    gen = torch.Generator(device="cuda").manual_seed(skv)
    q, k, v = (torch.randn(s, generator=gen, device="cuda") for s in ((batch, heads, sq, dim), (batch, kv_heads, skv, dim), (batch, kv_heads, skv, dim)))
    lengths = torch.tensor([skv - 7 * i if i != 2 else 0 for i in range(batch)], dtype=torch.int32, device="cuda")
    got = {}
    try:
        for dies in (0, 1):
            kx.set_tuning("sdpa_decode_dies", dies)
            for keys in (None, lengths):
                out = torch.full((batch, heads, sq, dim), float("nan"), device="cuda")
                ran = launches(torch, lambda: kx.sdpa_cache_dev(q, k, v, out, batch, heads, kv_heads, sq, skv, skv, dim, dim ** -0.5, True, window, 0, keys))
                grid = [g for name, g, _ in ran if "sdpa_decode_kernel" in name]
                assert len(grid) == 1 and (grid[0][1] == 1 and grid[0][2] == 1) == (dies == 1), ran
                got[dies, keys is None] = out
    finally:
        kx.set_tuning("sdpa_decode_dies", 1)
    for keys in (False, True):
        assert not torch.isnan(got[0, keys]).any() and torch.equal(got[0, keys], got[1, keys])


def test_attention_of_more_workgroups_than_one_grid_dimension_holds(hip_backend, torch_cuda):
    """65 535 sequences of one key, 86 KV heads, three query heads each: 16.9 million workgroups of 256, more than 2^32 work-items, so the grid has
    to keep its three dimensions. One key: the output is its V."""
    torch, kx = torch_cuda, hip_backend
    b, hkv, d = 65535, 86, 64
    v = torch.randn((b, hkv, 1, d), device="cuda")
    q = torch.zeros((b, 3 * hkv, 1, d), device="cuda")
    out = torch.full_like(q, float("nan"))
    kx.sdpa_cache_dev(q, v, v, out, b, 3 * hkv, hkv, 1, 1, 1, d, 1.0, True)
    assert kx.last_kernel() == "sdpa_decode_kernel"
    assert torch.equal(out.reshape(b, hkv, 3, d), v.expand(b, hkv, 3, d))


@pytest.mark.parametrize("cols", [1, 255, 257, 4095, 4096, 4097, 15454, 16384, 65537])
def test_argmax_at_the_edges_of_a_thread_s_walk(hip_backend, torch_cuda, cols):
    """The maximum at the first and the last column, ties between a thread's own elements and between threads, rows of -inf."""
    torch, kx = torch_cuda, hip_backend
    lg = np.random.default_rng(cols).standard_normal((5, cols)).astype(np.float32)
    lg[0, 0] = lg[1, cols - 1] = 9.0
    lg[2, cols // 3] = lg[2, min(cols // 3 + 256, cols - 1)] = 9.0
    lg[3, cols // 2:] = 9.0
    lg[4, :] = -np.inf
    idx = torch.full((5,), -1, dtype=torch.int32, device="cuda")
    kx.argmax_rows_dev(dev(torch, lg), 5, cols, idx)
    assert idx.cpu().tolist() == [int(r.argmax()) for r in lg]


@pytest.mark.parametrize("cols", [2 ** 31 - 1, 2 ** 31 - 64, 2 ** 31 - 500])
def test_argmax_of_a_row_up_to_the_last_int(hip_backend, torch_cuda, cols):
    """Where the share of a workgroup, rounded up, and a thread's step past the row's end are beyond the int range."""
    torch = torch_cuda
    row = torch.zeros(cols, device="cuda")
    idx = torch.full((1,), -1, dtype=torch.int32, device="cuda")
    for at in (cols - 1, cols - 300, 0):
        row[at] = 1.0
        hip_backend.argmax_rows_dev(row, 1, cols, idx)
        assert int(idx.cpu()[0]) == at
