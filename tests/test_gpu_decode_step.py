"""GPU: the C5 decode step over the real polar_cache (small model, 4096-token
context, sparse selection on, one flush inside the run)."""
import pytest
import torch

from zoomkv_revision_amd import decode_step as ds

pytestmark = pytest.mark.gpu


def test_decode_steps_through_polar_cache_with_a_flush(monkeypatch):
    for k, v in ds.PRODUCTION_ENV.items():
        monkeypatch.setenv(k, v)
    monkeypatch.delenv("POLAR_FORCE_CAND_TOKENS", raising=False)
    geo = ds.Qwen3Geometry(layers=2, hidden=256, heads=32, kv_heads=8, head_dim=128, ffn=512, vocab=1000)
    dev = torch.device("cuda:0")
    batch, context, interval, steps = 2, 4096, 64, 70
    model = ds.RandomQwen3(geo, dev, seed=42, max_position=8192)
    cache = ds.build_cache(geo, batch, context, steps + 8, interval, 2048, dev)
    ds.fill_cache(cache, geo, batch, context, 43, dev)
    retrieval0 = int(cache.cpu_valid_end[0])
    gen = torch.Generator(device=dev).manual_seed(42)
    tok = torch.randint(0, geo.vocab, (batch,), generator=gen, device=dev)
    seen = []
    for _ in range(steps):
        logits = model.decode_step(tok, cache)
        tok = ds.sample_next_token(logits, 0.6, 0.95, 20, generator=gen)
        seen.append(tok)
    torch.cuda.synchronize()
    assert cache.context == context + steps
    assert int(cache.cpu_valid_end[0]) == retrieval0 + interval          # one flush of 64 tokens
    assert cache._last_topk_indices is not None                          # the sparse path ran
    assert torch.isfinite(logits).all()
    toks = torch.stack(seen)
    assert ((toks >= 0) & (toks < geo.vocab)).all()
    b = ds.attention_path_bytes(cache, 0)
    assert b["total"] > b["quest_gqa"] > 0


def test_windowed_sampling_matches_full_vocabulary_on_device():
    """On the device generator: the windowed sampler and the op-for-op
    restatement of LLM.py:63-139 draw the same tokens over a Qwen3-size
    vocabulary (both consume one Exp(1) row per draw, so the streams stay
    aligned across calls)."""
    g = torch.Generator(device="cuda").manual_seed(3)
    ga = torch.Generator(device="cuda").manual_seed(11)
    gb = torch.Generator(device="cuda").manual_seed(11)
    for trial in range(40):
        logits = torch.randn(4, 151936, generator=g, device="cuda") * (0.5, 4.0, 16.0, 40.0)[trial % 4]
        a = ds.sample_next_token(logits, 0.6, 0.95, 20, generator=ga)
        b = ds.sample_next_token_full(logits, 0.6, 0.95, 20, generator=gb)
        assert torch.equal(a, b), (trial, a, b)


@pytest.mark.parametrize("bs,vocab", [(4, 151936), (1, 8192 + 10), (3, 100), (8, 3000), (2, 16384)])
@pytest.mark.parametrize("temperature,top_p,top_k", [(0.6, 0.95, 20), (1.0, 0.5, 5), (0.8, 0.0, 48),
                                                     (1.3, 0.99, 1)])
def test_hip_sampler_matches_full_vocabulary(bs, vocab, temperature, top_p, top_k):
    """The one-launch sampler (zkv_sample_window) against the op-for-op
    restatement of LLM.py:63-139 from the same device generator state: vocab
    sizes with a slice shorter than the window (8202), single slices (100,
    3000) and exact multiples; peaked and flat rows."""
    if top_k + 16 >= vocab:
        pytest.skip("the window covers the vocabulary: the full path runs")
    g = torch.Generator(device="cuda").manual_seed(vocab + top_k)
    ga = torch.Generator(device="cuda").manual_seed(5)
    gb = torch.Generator(device="cuda").manual_seed(5)
    for trial in range(12):
        logits = torch.randn(bs, vocab, generator=g, device="cuda") * (0.5, 4.0, 16.0)[trial % 3]
        a = ds.sample_next_token(logits, temperature, top_p, top_k, generator=ga)
        b = ds.sample_next_token_full(logits, temperature, top_p, top_k, generator=gb)
        assert a.dtype == torch.int64 and a.shape == (bs,)
        assert torch.equal(a, b), (trial, a, b)
        # the launch itself (no tie overflow on these rows, so no full-vocabulary draw)
        expo = torch.empty_like(logits).exponential_(1, generator=g)
        tok, flags = ds.sample_window_launch(logits, temperature, top_p, top_k, expo)
        assert int(flags.abs().sum()) == 0
        assert torch.equal(tok, ds.draw_full_vocabulary(logits, temperature, top_p, top_k, expo)), trial


def test_hip_sampler_ties_at_kth_value():
    """Ties at the k-th value: a group inside the window is drawn like any
    kept token; one wider than the window sets the row's overflow flag and the
    draw runs over the whole vocabulary with the same Exp(1) row."""
    for n_ties in (3, 40):
        logits = torch.full((2, 20000), -5.0, device="cuda")
        logits[:, 7:11] = torch.tensor([4.0, 3.0, 2.5, 2.0], device="cuda")
        logits[:, 9000:9000 + n_ties] = 1.0           # k = 6: the 6th value is a tie
        expo = torch.empty_like(logits).exponential_(1)
        _, flags = ds.sample_window_launch(logits, 1.0, 0.999, 6, expo)
        assert flags.tolist() == [int(n_ties > 16)] * 2
        ga = torch.Generator(device="cuda").manual_seed(1)
        gb = torch.Generator(device="cuda").manual_seed(1)
        seen = set()
        for _ in range(200):
            a = ds.sample_next_token(logits, 1.0, 0.999, 6, generator=ga)
            b = ds.sample_next_token_full(logits, 1.0, 0.999, 6, generator=gb)
            assert torch.equal(a, b)
            seen.update(a.tolist())
        assert seen <= set(range(7, 11)) | set(range(9000, 9000 + n_ties))
        assert len(seen & set(range(9000, 9000 + n_ties))) > 1


def test_hip_sampler_rejects_bad_arguments():
    from zoomkv_revision_amd._lib import ZkvError, check, lib, ptr
    L = lib()
    x = torch.randn(2, 1000, device="cuda")
    e = torch.ones_like(x)
    tok = torch.empty(2, dtype=torch.int64, device="cuda")
    fl = torch.empty(2, dtype=torch.int32, device="cuda")
    ws = torch.zeros(1 << 16, dtype=torch.uint8, device="cuda")
    args = lambda k, w, nbytes: (ptr(x), 1000, 2, 1000, 1.0, k, w, 0.9, ptr(e), 1000, ptr(tok), ptr(fl),
                                 ptr(ws), nbytes, 0)
    with pytest.raises(ZkvError):
        check(L.zkv_sample_window(*args(20, 65, ws.numel())))        # window over one wave
    with pytest.raises(ZkvError):
        check(L.zkv_sample_window(*args(20, 20, ws.numel())))        # window not past k
    with pytest.raises(ZkvError):
        check(L.zkv_sample_window(*args(20, 36, 16)))                # workspace too small
    check(L.zkv_sample_window(*args(20, 36, ws.numel())))
    torch.cuda.synchronize()
    assert ((tok >= 0) & (tok < 1000)).all() and (fl == 0).all()


def _bf16_close(got, ref, ulps=1.0):
    """Within `ulps` bf16 units at the tensor's largest magnitude (the fp32
    accumulation order differs from the library GEMM's)."""
    got, ref = got.float(), ref.float()
    scale = ref.abs().max().item()
    tol = ulps * scale * 2.0 ** -7 + 1e-6
    err = (got - ref).abs().max().item()
    assert err <= tol, (err, tol)


@pytest.mark.parametrize("M,K,N", [(4, 2560, 6144), (1, 512, 1000), (16, 256, 48), (4, 9728, 2560),
                                   (2, 4096, 2560), (8, 2560, 1000), (5, 256, 13), (3, 9728, 24),
                                   (8, 8192, 64), (12, 384, 40)])
def test_decode_linear_plain_and_norm(M, K, N):
    g = torch.Generator(device="cuda").manual_seed(M * 7 + N)
    x = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn(N, K, generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    nw = (torch.rand(K, generator=g, device="cuda") + 0.5).to(torch.bfloat16)
    out = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    ds.decode_linear(x, w, out)
    _bf16_close(out, (x.float() @ w.float().T).to(torch.bfloat16))
    xn = ds.rms_norm(x, nw, 1e-6)
    ds.decode_linear(x, w, out, norm_w=nw, eps=1e-6)
    _bf16_close(out, (xn.float() @ w.float().T).to(torch.bfloat16), ulps=2.0)
    out32 = torch.empty(M, N, dtype=torch.float32, device="cuda")
    ds.decode_linear(x, w, out32, norm_w=nw, eps=1e-6)
    assert torch.equal(out32, out32.to(torch.bfloat16).float())        # bf16 values held in fp32
    assert torch.equal(out32.to(torch.bfloat16), out)


@pytest.mark.parametrize("M,K,F_", [(4, 2560, 9728), (7, 512, 37), (12, 256, 24), (6, 256, 384)])
def test_decode_linear_residual_and_silu_mul(M, K, F_):
    g = torch.Generator(device="cuda").manual_seed(5 + M)
    x = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn(2 * F_, K, generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    act = torch.empty(M, F_, dtype=torch.bfloat16, device="cuda")
    ds.decode_linear(x, w, act, silu_mul=True)
    y = (x.float() @ w.float().T).to(torch.bfloat16)
    ref = torch.nn.functional.silu(y[:, :F_]) * y[:, F_:]
    _bf16_close(act, ref, ulps=2.0)
    if F_ % 128:
        return                                           # the down projection needs K = F_ % 128 == 0
    wo = (torch.randn(K, F_, generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    res = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    h = torch.empty(M, K, dtype=torch.bfloat16, device="cuda")
    ds.decode_linear(act, wo, h, residual=res)
    _bf16_close(h, res + (act.float() @ wo.float().T).to(torch.bfloat16), ulps=2.0)


@pytest.mark.parametrize("M,K,N", [
    (1, 128, 16), (4, 384, 4099), (3, 640, 33000),        # the stream: a lone unit, a row tail, several units per wave
    (2, 2688, 130), (4, 4352, 90),                        # x rows past the first request, a chunk that K ends inside
    (5, 2560, 6144), (9, 2560, 4896),                     # 4 KiB blocks at and under the wide kernel's 6144
    (6, 384, 33000), (16, 256, 98304), (12, 2688, 9000),  # its units passed over twice; 1, 2 and more chains
    (8, 7680, 1700), (16, 4352, 2890),                    # x rows of 123 and 139 KB
    (5, 2048, 2570), (16, 128, 4100), (6, 9728, 514),     # units of 11 rows, 9 and 3 (the last short); 5 K blocks or 4
    (5, 14720, 34), (7, 1152, 1), (8, 3072, 18),          # 8 K blocks per wave or 7; one row; half of the waves with one
])
def test_decode_linear_units_and_k_ranges(M, K, N):
    """The row, unit and K counts where the kernel or its split changes, with
    strided rows, the residual over several units and Inf in a row that only
    its own output sees.  fp32 sums of K products: within one bf16 unit of the
    fp32 product at the tensor's scale (two after a norm)."""
    g = torch.Generator(device="cuda").manual_seed(M + K + N)
    x = torch.randn(M, K + 8, generator=g, device="cuda").to(torch.bfloat16)[:, :K]
    w = (torch.randn(N, K, generator=g, device="cuda") * 0.05).to(torch.bfloat16)
    res = torch.randn(M, N, generator=g, device="cuda").to(torch.bfloat16)
    nw = (torch.rand(K, generator=g, device="cuda") + 0.5).to(torch.bfloat16)
    y = (x.float() @ w.float().T).to(torch.bfloat16)
    out = torch.full((M, N + 3), 7.0, dtype=torch.bfloat16, device="cuda")
    ds.decode_linear(x, w, out[:, :N], residual=res)
    _bf16_close(out[:, :N], res + y, ulps=2.0)
    assert (out[:, N:] == 7.0).all()
    xn = ds.rms_norm(x, nw, 1e-6)
    yn = (xn.float() @ w.float().T).to(torch.bfloat16)
    normed = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    ds.decode_linear(x, w, normed, norm_w=nw, eps=1e-6)
    _bf16_close(normed, yn, ulps=2.0)
    if N % 2 == 0:
        for source, norm_w in ((y, None), (yn, nw)):
            act = torch.empty(M, N // 2, dtype=torch.bfloat16, device="cuda")
            ds.decode_linear(x, w, act, norm_w=norm_w, eps=1e-6, silu_mul=True)
            _bf16_close(act, torch.nn.functional.silu(source[:, :N // 2]) * source[:, N // 2:], ulps=2.0)
    w[N // 2, K - 1] = float("inf")
    ds.decode_linear(x, w, normed)
    bad = torch.arange(N, device="cuda") == N // 2
    assert torch.isfinite(normed[:, ~bad]).all() and not torch.isfinite(normed[:, bad]).any()


@pytest.mark.parametrize("M,K,N", [
    (6, 3072, 4096), (5, 4096, 4096),                     # eight waves per unit, two chains each
    (7, 2560, 8192), (13, 3328, 8200),                    # four waves; two long rows per wave, a last unit of 8 rows
    (5, 3328, 17602), (9, 2688, 17602),                   # more units than the resident groups: two or three each
    (16, 4352, 2890), (6, 9728, 1090), (5, 2560, 4896),   # LDS nearly full; rows past the first requests; a workgroup per tile
])
def test_decode_linear_normed_splits(M, K, N):
    """The waves per unit, units per group and row lengths of the normed linear
    at 5 rows and more, without and with silu * up, the latter over both halves
    of the same weights.  Two bf16 units, as above."""
    g = torch.Generator(device="cuda").manual_seed(M + K + N)
    x = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn(N, K, generator=g, device="cuda") * 0.05).to(torch.bfloat16)
    nw = (torch.rand(K, generator=g, device="cuda") + 0.5).to(torch.bfloat16)
    y = (ds.rms_norm(x, nw, 1e-6).float() @ w.float().T).to(torch.bfloat16)
    out = torch.full((M + 1, N), 7.0, dtype=torch.bfloat16, device="cuda")
    ds.decode_linear(x, w, out[:M], norm_w=nw, eps=1e-6)
    _bf16_close(out[:M], y, ulps=2.0)
    act = torch.full((M + 1, N // 2), 7.0, dtype=torch.bfloat16, device="cuda")
    ds.decode_linear(x, w, act[:M], norm_w=nw, eps=1e-6, silu_mul=True)
    _bf16_close(act[:M], torch.nn.functional.silu(y[:, :N // 2]) * y[:, N // 2:], ulps=2.0)
    assert (out[M] == 7.0).all() and (act[M] == 7.0).all()


@pytest.mark.parametrize("M,K,N", [
    (1, 512, 12288), (2, 512, 12289), (3, 384, 5),        # a lane per 16 bytes of a row: one unit per wave, some two, a lone one
    (4, 2048, 3072), (1, 2048, 3073), (2, 1664, 2050),    # split K, one chunk per wave: 768 units, 769, a short last chunk
    (4, 2176, 2050),                                      # a wave with two chunks
    (3, 1152, 40002), (4, 1152, 39998), (2, 4096, 40000),  # units of 8 rows, the last of 2 (silu * up: of 1); of 4; of 4 (8)
])
def test_decode_linear_stream_units(M, K, N):
    """Where the waves of the stream kernel (4 rows and fewer, no norm) have
    one item or more and where its units change, plain, with the residual and as silu * up."""
    g = torch.Generator(device="cuda").manual_seed(M + K + N)
    x = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn(N, K, generator=g, device="cuda") * 0.05).to(torch.bfloat16)
    res = torch.randn(M, N, generator=g, device="cuda").to(torch.bfloat16)
    y = (x.float() @ w.float().T).to(torch.bfloat16)
    out = torch.full((M + 1, N), 7.0, dtype=torch.bfloat16, device="cuda")
    ds.decode_linear(x, w, out[:M])
    _bf16_close(out[:M], y)
    ds.decode_linear(x, w, out[:M], residual=res)
    _bf16_close(out[:M], res + y, ulps=2.0)
    assert (out[M] == 7.0).all()
    if N % 2 == 0:
        act = torch.full((M + 1, N // 2), 7.0, dtype=torch.bfloat16, device="cuda")
        ds.decode_linear(x, w, act[:M], silu_mul=True)
        _bf16_close(act[:M], torch.nn.functional.silu(y[:, :N // 2]) * y[:, N // 2:], ulps=2.0)
        assert (act[M] == 7.0).all()


@pytest.mark.parametrize("K,N", [(512, 1030), (2560, 4896), (2560, 6144), (3328, 17602), (4352, 2890), (256, 98304)])
@pytest.mark.parametrize("M", [2, 6, 16])
def test_decode_linear_norm_with_residual(M, K, N):
    """Norm and residual in one call, under and over 6144 blocks of 4 KiB, with
    one unit and with several per group of waves, out of place and in place.
    Two bf16 units, as above."""
    if M * K * 2 + 16384 > 160 * 1024:
        pytest.skip("x rows past the LDS")
    g = torch.Generator(device="cuda").manual_seed(M + K + N)
    x = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn(N, K, generator=g, device="cuda") * 0.05).to(torch.bfloat16)
    nw = (torch.rand(K, generator=g, device="cuda") + 0.5).to(torch.bfloat16)
    res = 4 * torch.randn(M, N, generator=g, device="cuda").to(torch.bfloat16)
    ref = res + (ds.rms_norm(x, nw, 1e-6).float() @ w.float().T).to(torch.bfloat16)
    out = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    ds.decode_linear(x, w, out, norm_w=nw, eps=1e-6, residual=res)
    _bf16_close(out, ref, ulps=2.0)
    ds.decode_linear(x, w, res, norm_w=nw, eps=1e-6, residual=res)
    assert torch.equal(res, out)


def test_decode_linear_rejects_bad_shapes():
    from zoomkv_revision_amd._lib import ZkvError
    x = torch.zeros(4, 200, dtype=torch.bfloat16, device="cuda")
    w = torch.zeros(16, 200, dtype=torch.bfloat16, device="cuda")
    with pytest.raises(ZkvError):                                        # K not a multiple of 128
        ds.decode_linear(x, w, torch.empty(4, 16, dtype=torch.bfloat16, device="cuda"))


def test_qk_norm_rope_and_append_match_torch():
    geo = ds.Qwen3Geometry(layers=1, hidden=256, heads=32, kv_heads=8, head_dim=128, ffn=512, vocab=1000)
    m = ds.RandomQwen3(geo, "cuda", seed=3, max_position=4096)
    L = m.layers[0]
    L["q_norm"] = (torch.rand(128, device="cuda") + 0.5).to(torch.bfloat16)
    L["k_norm"] = (torch.rand(128, device="cuda") + 0.5).to(torch.bfloat16)
    bs, pos = 3, 3001
    qkv = torch.randn(bs, (32 + 16) * 128, device="cuda").to(torch.bfloat16)
    q = torch.empty(bs, 1, 32, 128, dtype=torch.bfloat16, device="cuda")
    K = torch.zeros(bs, 8, 40, 128, dtype=torch.bfloat16, device="cuda")
    V = torch.zeros_like(K)
    ds.qk_norm_rope(qkv, 32, 8, L["q_norm"], L["k_norm"], geo.eps, m.cos[pos], m.sin[pos], q,
                    K[:, :, 17], V[:, :, 17])
    qr, kr, vr = qkv.split([32 * 128, 8 * 128, 8 * 128], dim=-1)
    q_ref = m._rope(ds.rms_norm(qr.reshape(bs, 1, 32, 128), L["q_norm"], geo.eps), pos)
    k_ref = m._rope(ds.rms_norm(kr.reshape(bs, 1, 8, 128), L["k_norm"], geo.eps), pos)
    _bf16_close(q, q_ref, ulps=2.0)
    _bf16_close(K[:, :, 17], k_ref[:, 0], ulps=2.0)
    assert torch.equal(V[:, :, 17], vr.reshape(bs, 8, 128))
    assert not K[:, :, 16].any() and not K[:, :, 18].any()              # only the reserved row


def test_fused_decode_step_matches_torch_layers(monkeypatch):
    for k, v in ds.PRODUCTION_ENV.items():
        monkeypatch.setenv(k, v)
    monkeypatch.delenv("POLAR_FORCE_CAND_TOKENS", raising=False)
    geo = ds.Qwen3Geometry(layers=2, hidden=256, heads=32, kv_heads=8, head_dim=128, ffn=512, vocab=1000)
    dev = torch.device("cuda:0")
    batch, context = 2, 4096
    outs = []
    for fused in (True, False):
        model = ds.RandomQwen3(geo, dev, seed=42, max_position=8192, fused=fused)
        cache = ds.build_cache(geo, batch, context, 8, 64, 2048, dev)
        ds.fill_cache(cache, geo, batch, context, 43, dev)
        tok = torch.tensor([5, 77], device=dev)
        logits = [model.decode_step(tok, cache) for _ in range(3)]
        outs.append((logits, cache))
    (lf, cf), (lt, ct) = outs
    assert cf.context == ct.context == context + 3
    for a, b in zip(lf, lt):
        _bf16_close(a, b, ulps=8.0)
    row = ct._near0 + (ct.current_seq_len[0] - 1 - int(ct.cpu_valid_end[0]))
    _bf16_close(cf.unified_keys[1][:, :, row], ct.unified_keys[1][:, :, row], ulps=8.0)
