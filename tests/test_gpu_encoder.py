"""The audio encoder (qwen_hip_encoder_*) against the reference's encoder
(qwen_encoder_forward, qwen_asr_encoder.c:171-372): the committed fixtures
tests/golden/enc_*.npz hold the compiled reference's output on seeded
weights and mel (tests/golden/make_enc_golden.py; test_encoder_oracle.py
re-derives one of them on the CPU).

Both compute in fp32 (the products of the fp32 matrix cores are exact fp32
products); sums run in another order, tanhf / expf of two libms differ by
ulps, and 2 layers of LayerNorm / attention / GELU amplify that: the bar is
|gpu - ref| <= 1e-4 + 1e-3 |ref| elementwise.
"""
import ctypes as C
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")
ATOL, RTOL = 1e-4, 1e-3


def fixture(name):
    return np.load(os.path.join(GOLD, name + ".npz"))


def build(qa, P, g):
    cfg = qa.EncConfig(*[int(v) for v in g["cfg"]])
    m = P.SynthEncoder(cfg, seed=int(g["seed"]))
    from golden.make_enc_golden import weight_checksum
    assert abs(weight_checksum(m) - float(g["weight_sum"])) <= 1e-9 * abs(float(g["weight_sum"]))
    mel = P.synth_mel(int(g["frames"]), int(g["seed"]), int(g["mel_set"]))
    assert float(np.float64(mel).sum()) == float(g["mel_sum"])
    return cfg, m, mel


def load(qa, cfg, m):
    e = qa.Encoder(cfg, 0)
    for l, arrs in enumerate(m.layers):
        e.load_layer(l, arrs)
    e.load_stem(m.stem)
    return e


@pytest.mark.parametrize("name", ["enc_tiny", "enc_06b2"])
def test_encoder_matches_reference(P, qa, gpu, name):
    g = fixture(name)
    cfg, m, mel = build(qa, P, g)
    e = load(qa, cfg, m)
    assert qa.lib().qk_enc_ring_ok(C.c_void_p(e.h))
    out = e.forward(mel)
    ref = g["out"]
    assert out.shape == ref.shape
    err = np.abs(out - ref)
    print(f"{name}: {out.shape[0]} tokens, max |d| {err.max():.2e}, max rel {float((err / (np.abs(ref) + 1e-6)).max()):.2e}")
    assert np.all(err <= ATOL + RTOL * np.abs(ref)), float((err - RTOL * np.abs(ref)).max())
    e.close()


def d2h(ptr, shape):
    """copy a device buffer (raw pointer) to a new host array"""
    hip = C.CDLL("libamdhip64.so")
    hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    out = np.empty(shape, np.float32)
    assert hip.hipMemcpy(out.ctypes.data, C.c_void_p(ptr), out.nbytes, 2) == 0   # hipMemcpyDeviceToHost
    return out


def test_encoder_synthetic_loader_and_device_path(P, qa, gpu):
    """load_synthetic (C recipe) == the same weights through load_layer/load_stem,
    bit for bit; forward_device == forward; repeated calls with other lengths
    (buffers regrown, partial chunks of every size class)"""
    cfg = qa.EncConfig(128, 2, 2, 64, 256, 96, 100, 200)
    m = P.SynthEncoder(cfg, seed=5)
    a = load(qa, cfg, m)
    b = qa.Encoder(cfg, 0)
    b.load_synthetic(5, 0.02)
    for frames in (320, 99, 1, 400):
        mel = P.synth_mel(frames, 5, 3)
        oa = a.forward(mel)
        ob = b.forward(mel)
        assert oa.shape[0] == a.tokens(frames)
        assert np.array_equal(oa, ob), frames
        dm = gpu.from_numpy(np.ascontiguousarray(mel)).to("cuda")
        gpu.cuda.synchronize()
        T, p = b.forward_device(dm.data_ptr(), frames)
        assert np.array_equal(d2h(p, (T, cfg.output_dim)), ob), frames
    a.close()
    b.close()


def test_encoder_rows_feed_the_decoder(P, qa, gpu):
    """encoder output (0.6B widths: 1024 = the decoder's hidden) straight into
    the decoder's device prefill gives what the host path gives"""
    cfg = qa.enc_preset(0)
    cfg.layers = 2
    e = qa.Encoder(cfg, 0)
    e.load_synthetic(0, 0.02)
    mel = P.synth_mel(300, 0, 4)
    rows = e.forward(mel)
    dm = gpu.from_numpy(np.ascontiguousarray(mel)).to("cuda")
    gpu.cuda.synchronize()
    T, p = e.forward_device(dm.data_ptr(), 300)
    dcfg = qa.preset(0)
    d = qa.Decoder(dcfg, 0, 512)
    d.load_synthetic(0, 0.02, 0.0)
    d.set_engine(0)
    d.prefill(rows[:-1])
    t_host = d.forward(rows[-1])
    d.set_kv_len(0)
    d.prefill_device(p, T - 1)
    t_dev = d.forward(rows[-1])
    assert T == rows.shape[0] and t_dev == t_host
    d.close()
    e.close()


def test_encoder_from_checkpoint(P, qa, gpu, tmp_path):
    """thinker.audio_tower.* read from a safetensors checkpoint (BF16 matrices,
    F32 vectors, two shards): shape taken from the tensors, chunk 100 and
    attention window 800 frames as the reference fixes them (qwen_asr.c:182-184),
    output bit-identical to the same weights loaded by hand with that config"""
    import ckpt_util
    from safetensors.torch import save_file
    g = fixture("enc_tiny")
    cfg, m, mel = build(qa, P, g)
    t = ckpt_util.enc_tensors(m)
    names = sorted(t)
    half = len(names) // 2
    save_file({n: t[n] for n in names[:half]}, str(tmp_path / "model-00001-of-00002.safetensors"))
    save_file({n: t[n] for n in names[half:]}, str(tmp_path / "model-00002-of-00002.safetensors"))
    e = qa.Encoder.from_checkpoint(str(tmp_path), 0)
    cfg.n_window_infer = 800
    for f, _ in qa.EncConfig._fields_:
        assert getattr(e.cfg, f) == getattr(cfg, f), f
    out = e.forward(mel)
    ref_h = load(qa, cfg, m)
    np.testing.assert_array_equal(out, ref_h.forward(mel))
    e.close()
    ref_h.close()


def test_encoder_error_conventions(P, qa, gpu):
    """Invalid shapes, calls before the weights are in, empty input and a
    layer index out of range fail with a code and a message; the encoder
    stays usable afterwards."""
    bad = qa.EncConfig(128, 2, 3, 64, 256, 96, 100, 200)          # heads * 64 != d_model
    assert not qa.lib().qwen_hip_encoder_create(C.byref(bad), 0)
    assert "encoder configuration" in qa.last_error()
    cfg = qa.EncConfig(128, 2, 2, 64, 256, 96, 100, 200)
    e = qa.Encoder(cfg, 0)
    mel = P.synth_mel(120, 1, 0)
    with pytest.raises(RuntimeError, match="not loaded"):
        e.forward(mel)
    m = P.SynthEncoder(cfg, seed=1)
    e.load_stem(m.stem)
    with pytest.raises(RuntimeError, match="layer 0 not loaded"):
        e.forward(mel)
    with pytest.raises(RuntimeError):
        e.load_layer(cfg.layers, m.layers[0])
    assert "outside" in qa.last_error()
    for l, arrs in enumerate(m.layers):
        e.load_layer(l, arrs)
    with pytest.raises(RuntimeError, match="bad argument"):
        e.forward(np.zeros((128, 0), np.float32))
    ref = load(qa, cfg, m).forward(mel)
    np.testing.assert_array_equal(e.forward(mel), ref)
    e.close()


def test_encoder_fp32_weights_take_the_fp32_gemm(P, qa, gpu):
    """A weight matrix whose values are not all bf16 values (possible through
    the fp32 load API) keeps fp32 and runs on the fp32 GEMM, next to
    bf16-valued ones on the bf16 GEMM; the mix matches the reference encoder
    (oracle/_ref) on the same weights."""
    if not P.ref_available():
        pytest.skip("oracle/_ref not built")
    cfg = qa.EncConfig(128, 2, 2, 64, 256, 96, 100, 200)
    m = P.SynthEncoder(cfg, seed=9)
    rng = np.random.default_rng(9)
    wo = m.layers[1][6]
    m.layers[1][6] = (wo * (1.0 + 1e-3 * rng.standard_normal(wo.shape))).astype(np.float32)   # off the bf16 grid
    assert np.any(m.layers[1][6].view(np.uint32) & 0xFFFF)
    mel = P.synth_mel(250, 9, 1)
    e = load(qa, cfg, m)
    out = e.forward(mel)
    ref = P.RefEncoder(m).forward(mel, e.tokens(250))
    err = np.abs(out - ref)
    assert np.all(err <= ATOL + RTOL * np.abs(ref)), float(err.max())
    e.close()


class RingArgs(C.Structure):
    _fields_ = [(n, C.c_void_p) for n in ("A", "W", "zero")] + [(n, C.c_int) for n in (
        "M", "N", "K", "taps", "in_h", "in_w", "col_h", "col_w", "chunks", "valid")] + [
        ("bias", C.c_void_p), ("pe", C.c_void_p), ("pe_rows", C.c_int), ("gelu", C.c_int), ("add", C.c_int),
        ("C", C.c_void_p), ("out", C.c_void_p), ("ln_w", C.c_void_p), ("ln_b", C.c_void_p), ("ln_eps", C.c_float),
        ("ws", C.c_void_p), ("kc", C.c_int), ("split", C.c_int)]


def halves(gpu, x, pixel=False):
    """fp32 [M][K] -> rows [K hi | K lo], or pixels K / 32 x [32 hi | 32 lo], and the value they carry"""
    hi = x.bfloat16()
    lo = (x - hi.float()).bfloat16()
    M, K = x.shape
    t = gpu.stack([hi.view(M, K // 32, 32), lo.view(M, K // 32, 32)], 2) if pixel else gpu.cat([hi, lo], 1)
    return t.reshape(M, 2 * K).contiguous(), hi.double() + lo.double()


def unhalve(gpu, t, N, pixel=False):
    t = t.double()
    return (t.view(-1, N // 32, 2, 32).sum(2).reshape(-1, N) if pixel else t[:, :N] + t[:, N:])


def gelu64(gpu, v):
    return 0.5 * v * (1 + gpu.tanh(0.7978845608028654 * (v + 0.044715 * v ** 3)))


class RingPlan(C.Structure):
    _fields_ = [(n, C.c_int) for n in ("bm", "bn", "groups", "kc", "split")]


def ring_choice(lib, M, N, K, fused, ws, gather=0):
    """(tile rows, tile columns, k groups, splits) of the launch"""
    p = RingPlan()
    lib.qk_enc_ring_plan_for(M, N, K, int(fused), gather, C.c_long(ws), C.byref(p))
    return p.bm, p.bn, p.groups, p.split


# every kernel of the products: the tile, k groups and splits that a product with an
# own epilogue (fp32, GELU) and one that is split for the LayerNorm pass launch; ragged
# rows and columns, k walks shorter and longer than the ring, no whole 64-deep stages
@pytest.mark.parametrize("M,N,K,own,part", [
    (1, 128, 128, (32, 128, 2, 1), (32, 128, 2, 1)), (32, 96, 64, (32, 128, 2, 1), (32, 128, 2, 1)),
    (20, 1000, 1120, (32, 128, 1, 7), (32, 128, 1, 7)), (31, 960, 96, (32, 128, 1, 1), (32, 128, 1, 1)),
    (33, 192, 96, (64, 128, 1, 1), (64, 128, 1, 1)), (97, 1024, 1024, (32, 64, 2, 1), (64, 128, 2, 8)),
    (390, 896, 3584, (64, 128, 2, 5), (64, 128, 2, 5)), (390, 2688, 896, (64, 128, 2, 1), None),
    (390, 3584, 896, (64, 128, 2, 1), None), (300, 1000, 1120, (64, 128, 1, 6), (64, 128, 1, 6)),
    (1030, 2048, 96, (64, 128, 1, 1), None), (65, 4096, 896, (32, 64, 2, 1), None), (1600, 3072, 128, (128, 128, 1, 1), None),
    (4100, 1024, 64, (128, 128, 1, 1), (128, 128, 1, 1))])
@pytest.mark.parametrize("what", ["f32", "gelu", "ln"])
def test_ring_products(P, qa, gpu, M, N, K, own, part, what):
    """qk_enc_ring_launch on rows of halves against a float64 product of the
    same halves: fp32 accumulation leaves 4 K 2^-24 sum |x w|, halves of the
    result 2^-16 relative."""
    if part or what != "ln":
        got = ring_choice(qa.lib(), M, N, K, what != "ln", max(8 * 64 * 64 * 1024, M * N))
        assert got == (part if what == "ln" else own), got
    ring_product(qa, gpu, M, N, K, what)


def ring_product(qa, gpu, M, N, K, what):
    lib = qa.lib()
    lib.qk_enc_ring_launch.argtypes = [C.c_void_p, C.c_void_p, C.c_long, C.c_void_p]
    g = gpu.Generator(device="cuda").manual_seed(M + N)
    r = lambda *s: gpu.randn(*s, generator=g, device="cuda")
    x, W = r(M, K), (r(N, K) * 0.05).bfloat16()
    A, xv = halves(gpu, x)
    bias, x0 = r(N), r(M, N)
    ws = gpu.empty(max(8 * 64 * 64 * 1024, M * N), device="cuda")
    f, out = x0.clone(), gpu.zeros(M, 2 * N, dtype=gpu.bfloat16, device="cuda")
    a = RingArgs(A=A.data_ptr(), W=W.data_ptr(), M=M, N=N, K=K, bias=bias.data_ptr())
    if what == "f32":
        a.C = f.data_ptr()
    elif what == "gelu":
        a.out, a.gelu = out.data_ptr(), 1
    else:
        w, b = 1 + 0.1 * r(N), r(N)
        a.C, a.out, a.add, a.ln_w, a.ln_b, a.ln_eps = f.data_ptr(), out.data_ptr(), 1, w.data_ptr(), b.data_ptr(), 1e-5
    if what == "ln" and N > 1024:
        assert lib.qk_enc_ring_launch(C.byref(a), ws.data_ptr(), ws.numel(), None) == -1
        return
    qa.check(lib.qk_enc_ring_launch(C.byref(a), ws.data_ptr(), ws.numel(), None), "ring")
    gpu.cuda.synchronize()
    y = xv @ W.double().t().contiguous() + bias.double()
    bound = 4 * K * 2.0 ** -24 * (xv.abs() @ W.double().abs().t().contiguous()) + 1e-6
    if what == "f32":
        assert bool(((f.double() - y).abs() <= bound).all())
    elif what == "gelu":
        got = unhalve(gpu, out, N)
        ref = gelu64(gpu, y)
        assert bool(((got - ref).abs() <= 1.2 * bound + 2.0 ** -16 * ref.abs() + 2.0 ** -22 * y.abs()).all())
    else:
        y = y + x0.double()
        assert bool(((f.double() - y).abs() <= bound + 2.0 ** -22 * y.abs()).all())
        fd = f.double()
        ref = (fd - fd.mean(1, keepdim=True)) / gpu.sqrt(fd.var(1, unbiased=False, keepdim=True) + 1e-5) * w + b
        assert float((unhalve(gpu, out, N) - ref).abs().max()) < 2e-4      # 2^-16 of values up to ~8


# few rows with an own epilogue: 32 x 64 tiles on one block per CU, at the fewest
# blocks (32) and the most (256), ragged rows and columns, k walks shorter than the ring
@pytest.mark.parametrize("M,N,K", [(1, 2048, 128), (64, 1024, 64), (1, 8192, 64), (33, 3080, 128), (97, 2688, 896),
                                   (128, 4096, 1024), (160, 3068, 640)])
@pytest.mark.parametrize("what", ["f32", "gelu"])
def test_ring_products_narrow(P, qa, gpu, M, N, K, what):
    assert ring_choice(qa.lib(), M, N, K, 1, 1 << 30) == (32, 64, 2, 1)
    ring_product(qa, gpu, M, N, K, what)


# 64-row tiles, split and unsplit; 128-row tiles (the second layer of 11 chunks and
# more), with a ragged last one
@pytest.mark.parametrize("chunks,h,w,valid,bm,split", [(1, 8, 5, 3, 64, 8), (3, 32, 25, 1, 64, 6), (9, 32, 50, 25, 64, 1),
                                                       (2, 4, 1, 1, 64, 8), (10, 64, 50, 7, 64, 1), (11, 64, 50, 12, 128, 1)])
def test_ring_convolution(P, qa, gpu, chunks, h, w, valid, bm, split):
    """The gathered 3x3 / stride 2 / padding 1 convolution with GELU, weights
    through qk_enc_tile_weights_launch, and the last chunk's padding zeroed,
    against float64 on the same halves."""
    lib, CH = qa.lib(), 480
    lib.qk_enc_ring_launch.argtypes = [C.c_void_p, C.c_void_p, C.c_long, C.c_void_p]
    lib.qk_enc_tile_weights_launch.argtypes = [C.c_void_p, C.c_void_p, C.c_int, C.c_int, C.c_int, C.c_void_p]
    g = gpu.Generator(device="cuda").manual_seed(h * w)
    x = gpu.randn(chunks * h * w, CH, generator=g, device="cuda")
    W = (gpu.randn(CH, 9 * CH, generator=g, device="cuda") * 0.02).bfloat16()      # [n][tap][channel]
    Wt, zero = gpu.empty_like(W), gpu.zeros(64, dtype=gpu.bfloat16, device="cuda")
    qa.check(lib.qk_enc_tile_weights_launch(W.data_ptr(), Wt.data_ptr(), CH, 9 * CH, 1, None), "tile")
    A, xv = halves(gpu, x, pixel=True)
    ho, wo = (h + 1) // 2, (w + 1) // 2
    M = chunks * ho * wo
    got = ring_choice(lib, M, CH, 9 * CH, 1, 8 * M * CH, 1)
    assert got == (bm, 128, 1, split), got
    bias = gpu.randn(CH, generator=g, device="cuda")
    out = gpu.full((M, 2 * CH), 7.0, dtype=gpu.bfloat16, device="cuda")
    ws = gpu.empty(8 * M * CH, device="cuda")
    a = RingArgs(A=A.data_ptr(), W=Wt.data_ptr(), zero=zero.data_ptr(), M=M, N=CH, K=9 * CH, taps=9, in_h=h, in_w=w,
                 col_h=ho, col_w=wo, chunks=chunks, valid=valid, bias=bias.data_ptr(), gelu=1, out=out.data_ptr())
    qa.check(lib.qk_enc_ring_launch(C.byref(a), ws.data_ptr(), ws.numel(), None), "ring")
    gpu.cuda.synchronize()
    im = gpu.nn.functional.pad(xv.view(chunks, h, w, CH), (0, 0, 1, 2, 1, 2))
    cols = gpu.cat([im[:, i:i + 2 * ho - 1:2, j:j + 2 * wo - 1:2] for i in range(3) for j in range(3)], -1).reshape(M, -1)
    y = cols @ W.double().t().contiguous() + bias.double()
    bound = 4 * 9 * CH * 2.0 ** -24 * (cols.abs() @ W.double().abs().t().contiguous()) + 1e-6
    ref = gelu64(gpu, y).view(chunks, ho, wo, CH)
    ref[-1, :, valid:] = 0
    ref = ref.view(M, CH)
    got = unhalve(gpu, out, CH, pixel=True)
    assert bool(((got - ref).abs() <= 1.2 * bound + 2.0 ** -16 * ref.abs() + 2.0 ** -22 * y.abs()).all())


# a token's pixels, top to bottom, against the positions' table and the first LayerNorm:
# 64-row tiles in splits and 128-row tiles, ragged last ones
@pytest.mark.parametrize("T,w,N,bm,split", [(1, 1, 128, 64, 8), (39, 13, 896, 64, 8), (390, 13, 896, 64, 5),
                                            (4750, 13, 896, 128, 1), (4161, 13, 1024, 128, 1)])
def test_ring_token_rows(P, qa, gpu, T, w, N, bm, split):
    lib, CH, H = qa.lib(), 480, 16
    lib.qk_enc_ring_launch.argtypes = [C.c_void_p, C.c_void_p, C.c_long, C.c_void_p]
    lib.qk_enc_tile_weights_launch.argtypes = [C.c_void_p, C.c_void_p, C.c_int, C.c_int, C.c_int, C.c_void_p]
    g = gpu.Generator(device="cuda").manual_seed(T)
    chunks, K = -(-T // w), CH * H
    x = gpu.randn(chunks * H * w, CH, generator=g, device="cuda")
    W = (gpu.randn(N, K, generator=g, device="cuda") * 0.02).bfloat16()            # column channel * 16 + row
    Wt, zero = gpu.empty_like(W), gpu.zeros(64, dtype=gpu.bfloat16, device="cuda")
    qa.check(lib.qk_enc_tile_weights_launch(W.data_ptr(), Wt.data_ptr(), N, CH, H, None), "tile")
    A, xv = halves(gpu, x, pixel=True)
    pe, lw, lb = (gpu.randn(n, N, generator=g, device="cuda") for n in (w, 1, 1))
    f, out = gpu.empty(T, N, device="cuda"), gpu.empty(T, 2 * N, dtype=gpu.bfloat16, device="cuda")
    ws = gpu.empty(max(2048 * 64 * 64, T * N), device="cuda")
    got = ring_choice(lib, T, N, K, 0, ws.numel(), 1)
    assert got == (bm, 128, 1, split), got
    a = RingArgs(A=A.data_ptr(), W=Wt.data_ptr(), zero=zero.data_ptr(), M=T, N=N, K=K, taps=H, in_h=H, in_w=w,
                 pe=pe.data_ptr(), pe_rows=w, C=f.data_ptr(), out=out.data_ptr(), ln_w=lw.data_ptr(), ln_b=lb.data_ptr(),
                 ln_eps=1e-5)
    qa.check(lib.qk_enc_ring_launch(C.byref(a), ws.data_ptr(), ws.numel(), None), "ring")
    gpu.cuda.synchronize()
    cols = xv.view(chunks, H, w, CH).permute(0, 2, 3, 1).reshape(chunks * w, K)[:T].contiguous()
    rows = pe.double()[gpu.arange(T, device="cuda") % w]
    y = cols @ W.double().t().contiguous() + rows
    bound = 4 * K * 2.0 ** -24 * (cols.abs() @ W.double().abs().t().contiguous()) + 2.0 ** -22 * rows.abs() + 1e-6
    assert bool(((f.double() - y).abs() <= bound).all())
    fd = f.double()
    ref = (fd - fd.mean(1, keepdim=True)) / gpu.sqrt(fd.var(1, unbiased=False, keepdim=True) + 1e-5) * lw + lb
    assert bool(((unhalve(gpu, out, N) - ref).abs() <= 2.0 ** -16 * ref.abs() + 2e-5).all())   # fp32 sums of the row


# windows of one and several rounds of the four waves' 128 keys; ragged last
# windows of one key, and a window longer than the sequence
@pytest.mark.parametrize("T,win", [(1, 104), (97, 104), (209, 104), (33, 16), (300, 150), (401, 400), (130, 1000)])
def test_window_attention(P, qa, gpu, T, win):
    lib, H = qa.lib(), 3
    lib.qk_enc_attention_launch.argtypes = [C.c_void_p] * 3 + [C.c_int] * 4 + [C.c_float, C.c_void_p]
    g = gpu.Generator(device="cuda").manual_seed(T)
    qkv = gpu.randn(T, 3, H, 64, generator=g, device="cuda")
    out, out16 = gpu.empty(T, H * 64, device="cuda"), gpu.empty(T, 2 * H * 64, dtype=gpu.bfloat16, device="cuda")
    qa.check(lib.qk_enc_attention_launch(qkv.data_ptr(), out.data_ptr(), None, T, H, 64, win, 0.125, None), "attn")
    qa.check(lib.qk_enc_attention_launch(qkv.data_ptr(), None, out16.data_ptr(), T, H, 64, win, 0.125, None), "attn")
    gpu.cuda.synchronize()
    ref = gpu.empty(T, H, 64, dtype=gpu.float64, device="cuda")
    for t0 in range(0, T, win):
        q, k, v = (qkv[t0:t0 + win, i].double().transpose(0, 1).contiguous() for i in range(3))
        p = gpu.softmax(gpu.bmm(q, k.transpose(1, 2).contiguous()) * 0.125, -1)
        ref[t0:t0 + win] = gpu.bmm(p, v).transpose(0, 1)
    ref = ref.view(T, H * 64)
    assert float((out.double() - ref).abs().max()) < 1e-5                # fp32 products and sums
    assert bool(((unhalve(gpu, out16, H * 64) - out.double()).abs() <= 2.0 ** -16 * out.double().abs() + 1e-9).all())


# a window's rows stay in it: the rows of the next window that a wave's 32 keys reach
# over weigh nothing, whatever they hold
@pytest.mark.parametrize("T,win", [(260, 104), (100, 16), (97, 33), (301, 150)])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_window_attention_nonfinite_rows(P, qa, gpu, T, win, bad):
    lib, H = qa.lib(), 2
    lib.qk_enc_attention_launch.argtypes = [C.c_void_p] * 3 + [C.c_int] * 4 + [C.c_float, C.c_void_p]
    g = gpu.Generator(device="cuda").manual_seed(T)
    qkv = gpu.randn(T, 3, H, 64, generator=g, device="cuda")

    def run(x):
        out = gpu.empty(T, H * 64, device="cuda")
        qa.check(lib.qk_enc_attention_launch(x.data_ptr(), out.data_ptr(), None, T, H, 64, win, 0.125, None), "attn")
        gpu.cuda.synchronize()
        return out
    clean = run(qkv)
    for w0 in range(0, T, win):
        w1 = min(T, w0 + win)
        x = qkv.clone()
        x[w0:w1] = bad
        out = run(x)
        assert gpu.equal(out[:w0], clean[:w0]) and gpu.equal(out[w1:], clean[w1:]), w0
        # an infinite value of the window's last key weighs more than 0 in each of its rows
        x = qkv.clone()
        x[w1 - 1, 2] = float("inf")
        assert bool((run(x)[w0:w1] == float("inf")).all()), w0


class GemmArgs(C.Structure):
    _fields_ = [(n, C.c_void_p) for n in ("A", "B", "C")] + [(n, C.c_int) for n in ("M", "N", "K", "lda", "ldb", "ldc")] + [
        (n, C.c_void_p) for n in ("bias_m", "bias_n", "pe")] + [(n, C.c_int) for n in (
            "pe_rows", "gelu", "add", "col_w", "col_h", "col_chunks", "col_valid", "pad_rows", "conv_c", "conv_in_h",
            "conv_in_w")] + [("ws", C.c_void_p), ("ws_elems", C.c_long), ("kc", C.c_int), ("split", C.c_int)] + [
        (n, C.c_void_p) for n in ("A16", "B16", "ln_w", "ln_b", "ln_out")] + [("ln_eps", C.c_float)]


# The GELU against 64 bits, through a product that hands each value to it exactly: over
# each range no further off (root mean square of the relative error) than the
# reference's expression 0.5 v (1 + tanh(u)) is in fp32 with a correctly rounded tanh.
def test_gelu_precision(P, qa, gpu):
    lib, n = qa.lib(), 65536
    rng = np.random.default_rng(3)
    f32 = np.float32
    ranges = [(-6, -4), (-4, -2), (-2, -1), (-1, -.5), (-.5, -.1), (-.1, -.01), (.01, .1), (.1, .5), (.5, 1), (1, 2),
              (2, 3), (3, 4), (4, 6), (6, 9), (9, 40)]
    v = np.concatenate([rng.uniform(a, b, n).astype(f32) for a, b in ranges])
    edge = np.array([0.0, 9.0, 9.5, -9.0, -9.5, 1e30, -1e30, np.inf, -np.inf, np.nan, 1e-30, -1e-30], f32)
    W = np.zeros((v.size + 64, 4), f32)
    W[:v.size, 0], W[v.size:v.size + edge.size, 0] = v, edge
    A = np.array([[1, 0, 0, 0]], f32)
    got = np.empty(W.shape[0], f32)
    dA, dW, dC = gpu.from_numpy(A).cuda(), gpu.from_numpy(W).cuda(), gpu.empty(1, W.shape[0], device="cuda")
    a = GemmArgs(A=dA.data_ptr(), B=dW.data_ptr(), C=dC.data_ptr(), M=1, N=W.shape[0], K=4, lda=4, ldb=4, ldc=W.shape[0],
                 gelu=1)
    qa.check(lib.qk_enc_gemm_launch(C.byref(a), None), "gemm")
    got = dC.cpu().numpy()[0]
    w = v.astype(np.float64)
    u = 0.7978845608028654 * (w + 0.044715 * w ** 3)
    exact = w / (1.0 + np.exp(-2.0 * u))
    u32 = f32(0.7978845608028654) * (v + f32(0.044715) * (v * v * v))
    form = f32(0.5) * v * (f32(1) + np.tanh(u32.astype(np.float64)).astype(f32))
    for i, r in enumerate(ranges):
        s = slice(i * n, (i + 1) * n)
        rms = [float(np.sqrt((((y[s] - exact[s]) / exact[s]) ** 2).mean())) for y in (got, form)]
        # 1 %: 65536 samples of each
        assert rms[0] <= 1.01 * rms[1], (r, rms)
    e = got[v.size:v.size + edge.size]
    assert e[0] == 0 and e[1] == 9 and e[2] == f32(9.5) and e[5] == f32(1e30) and e[7] == np.inf
    assert np.all(np.abs(e[[3, 4, 6]]) < 1e-27) and np.isnan(e[8]) and np.isnan(e[9])     # -inf * 0 is the reference's
    assert np.allclose(e[10:], f32([5e-31, -5e-31]), rtol=1e-6, atol=0)


def test_encoder_stem_reload_that_fails(P, qa, gpu):
    """A stem reload that fails at conv2's bias leaves the new conv1, conv2 and
    conv3 matrices beside the old rest: both forms of a matrix, as loaded and as
    the products read it, are the same one."""
    cfg = qa.EncConfig(128, 2, 2, 64, 256, 96, 100, 200)
    a, b = P.SynthEncoder(cfg, seed=5), P.SynthEncoder(cfg, seed=6)
    mel = P.synth_mel(250, 5, 3)
    e = load(qa, cfg, a)
    arrs = [np.ascontiguousarray(x, np.float32) for x in b.stem]
    w = qa.EncStemWeights(*[x.ctypes.data for x in arrs])
    w.conv2_b = None
    assert qa.lib().qwen_hip_encoder_load_stem(e.h, C.byref(w)) < 0
    out = e.forward(mel)
    a.stem[0:3], a.stem[4] = b.stem[0:3], b.stem[4]
    m = load(qa, cfg, a)
    assert np.array_equal(out, m.forward(mel))
    e.close()
    m.close()


def test_encoder_mel_in_host_memory(P, qa, gpu):
    """a mel in pinned host memory: copied, with the same result"""
    cfg = qa.EncConfig(128, 2, 2, 64, 256, 96, 100, 200)
    e = qa.Encoder(cfg, 0)
    e.load_synthetic(5, 0.02)
    mel = P.synth_mel(250, 5, 3)
    want = e.forward(mel)
    h = gpu.empty(128, 250, pin_memory=True)
    h.copy_(gpu.from_numpy(mel))
    T, p = e.forward_device(h.data_ptr(), 250)
    assert np.array_equal(d2h(p, (T, cfg.output_dim)), want)
    e.close()


def test_encoder_activation_memory(P, qa, gpu):
    """A bf16-valued encoder allocates what its products use: the stem's pixels,
    the rows' activations and the split workspace, and no patch or row matrix of
    the general path (80 MB of token rows here)."""
    cfg = qa.EncConfig(128, 2, 2, 64, 256, 96, 100, 200)
    frames, chunks = 20000, 200
    e = qa.Encoder(cfg, 0)
    e.load_synthetic(1, 0.02)
    mel = P.synth_mel(frames, 1, 0)
    before = gpu.cuda.mem_get_info()[0]
    e.forward(mel)
    used = before - gpu.cuda.mem_get_info()[0]
    pixels = 480 * chunks * (64 * 50 + 32 * 25 + 16 * 13) * 4
    T = chunks * 13
    rows = T * 4 * (3 * 128 + 4 * 128 + 256 + 96)
    ws = 2048 * 64 * 64 * 4
    assert used <= 128 * frames * 4 + pixels + rows + ws + (40 << 20), used     # 12 buffers, rounded up each
    e.close()


def encoder64(gpu, m, mel):
    """qwen_encoder_forward (qwen_asr_encoder.c:171-372) in float64 on a SynthEncoder's arrays"""
    t = lambda a: gpu.from_numpy(np.ascontiguousarray(a, np.float32)).cuda().double()
    c, cw = m.cfg, m.cfg.chunk_size
    stem, F = [t(a) for a in m.stem], gpu.nn.functional
    x, n = t(mel), -(-mel.shape[1] // cw)

    def ln(v, w, b):
        d = v - v.mean(-1, keepdim=True)
        return d / gpu.sqrt((d * d).mean(-1, keepdim=True) + 1e-5) * w + b
    rows = []
    for i in range(n):                                       # every chunk is an image of its own
        y = x[None, None, :, i * cw:(i + 1) * cw]
        for k in range(0, 6, 2):
            co, ci, (h, w) = 480, y.shape[1], y.shape[2:]
            ho, wo = (h + 1) // 2, (w + 1) // 2
            im = F.pad(y, (1, 2, 1, 2))[0]
            cols = gpu.stack([im[:, a:a + 2 * ho - 1:2, b:b + 2 * wo - 1:2] for a in range(3) for b in range(3)], 1)
            y = gelu64(gpu, stem[k].view(co, ci * 9) @ cols.reshape(ci * 9, ho * wo) + stem[k + 1][:, None])
            y = y.view(1, co, ho, wo)
        y = y[0].permute(2, 0, 1).reshape(y.shape[3], -1) @ stem[6].t()
        half = c.d_model // 2
        inv = gpu.exp(-gpu.arange(half, device="cuda").double() * np.log(10000.0) / (half - 1))
        a = gpu.arange(y.shape[0], device="cuda").double()[:, None] * inv
        rows.append(y + gpu.cat([gpu.sin(a), gpu.cos(a)], 1))
    x = gpu.cat(rows)
    tpc = cw
    for _ in range(3):
        tpc = (tpc + 1) // 2
    win, H = tpc * (c.n_window_infer // cw), c.heads
    for arrs in m.layers:
        w = [t(a) for a in arrs]
        v = ln(x, w[8], w[9])
        q, k, u = (v @ w[2 * i].t() + w[2 * i + 1] for i in range(3))
        att = gpu.empty_like(q)
        for t0 in range(0, x.shape[0], win):
            s = slice(t0, t0 + win)
            qq, kk, uu = (z[s].view(-1, H, 64).transpose(0, 1) for z in (q, k, u))
            att[s] = (gpu.softmax(qq @ kk.transpose(1, 2) / 8.0, -1) @ uu).transpose(0, 1).reshape(-1, c.d_model)
        x = x + att @ w[6].t() + w[7]
        x = x + gelu64(gpu, ln(x, w[14], w[15]) @ w[10].t() + w[11]) @ w[12].t() + w[13]
    return gelu64(gpu, ln(x, stem[7], stem[8]) @ stem[9].t() + stem[10]) @ stem[11].t() + stem[12]


def test_encoder64_is_the_reference(P, qa, gpu):
    """the float64 encoder of this file against the compiled reference's output"""
    g = fixture("enc_tiny")
    cfg, m, mel = build(qa, P, g)
    err = np.abs(encoder64(gpu, m, mel).cpu().numpy() - g["out"])
    assert np.all(err <= ATOL + RTOL * np.abs(g["out"])), float(err.max())


# The general path: off-grid weights (fp32 products), bf16-valued ones of widths the ring
# products do not take (d above 1024; outputs that are no whole float4s), off-grid ones
# among bf16-valued ones (stem, a layer's fc2, the output projection), an ffn of no whole
# 32-wide tiles; a few rows (split products, LayerNorm in the reduce) and 12 chunks
# (128 x 128 tiles of the second convolution)
@pytest.mark.parametrize("frames", [41, 350, 1230])
@pytest.mark.parametrize("d,ffn,out,off", [(128, 256, 96, "all"), (1088, 256, 96, ""), (128, 256, 98, ""),
                                           (128, 256, 96, "mixed"), (128, 132, 96, "all"), (192, 1056, 1030, "")])
def test_encoder_general_path(P, qa, gpu, d, ffn, out, off, frames):
    cfg = qa.EncConfig(d, 2, d // 64, 64, ffn, out, 100, 200)
    m = P.SynthEncoder(cfg, seed=11)
    rng = np.random.default_rng(11)

    def nudge(arrs, ids):
        for i in ids:
            arrs[i] = (arrs[i] * (1.0 + 1e-3 * rng.standard_normal(arrs[i].shape))).astype(np.float32)
    if off == "all":
        for l in m.layers:
            nudge(l, (0, 2, 4, 6, 10, 12))
        nudge(m.stem, (2, 4, 6, 9, 11))
    elif off == "mixed":
        nudge(m.stem, (4, 11))
        nudge(m.layers[1], (12,))
    mel = P.synth_mel(frames, 11, 2)
    e = load(qa, cfg, m)
    assert not qa.lib().qk_enc_ring_ok(C.c_void_p(e.h))
    got, ref = e.forward(mel), encoder64(gpu, m, mel).cpu().numpy()
    err = np.abs(got - ref)
    assert got.shape == ref.shape and np.all(err <= ATOL + RTOL * np.abs(ref)), float(err.max())
    assert np.array_equal(e.forward(mel[:, :40]), load(qa, cfg, m).forward(mel[:, :40]))     # after a longer call
    e.close()


# the ring path at its narrowest and widest, products narrower than a tile, k walks of
# odd 32-deep tiles, one-frame and one-chunk inputs
@pytest.mark.parametrize("frames", [1, 100, 431])
@pytest.mark.parametrize("d,ffn,out", [(64, 32, 4), (192, 96, 100), (320, 1056, 36), (1024, 64, 2048)])
def test_encoder_ring_path_widths(P, qa, gpu, d, ffn, out, frames):
    cfg = qa.EncConfig(d, 2, d // 64, 64, ffn, out, 100, 200)
    m, mel = P.SynthEncoder(cfg, seed=13), P.synth_mel(frames, 13, 1)
    e = load(qa, cfg, m)
    assert qa.lib().qk_enc_ring_ok(C.c_void_p(e.h))
    got, ref = e.forward(mel), encoder64(gpu, m, mel).cpu().numpy()
    err = np.abs(got - ref)
    assert got.shape == ref.shape and np.all(err <= ATOL + RTOL * np.abs(ref)), float(err.max())
    e.close()
