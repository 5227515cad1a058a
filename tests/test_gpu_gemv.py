"""GPU parity of the activation quantizer, weight quantizers and block-quantized
GEMV entry points against the CPU oracle, through the C ABI.

Bar: Q8_1 bytes, weight bytes and int32 block dots bit-exact; fp32 GEMV
outputs bit-exact against the oracle run in the kernels' documented order
(L=16 lanes, G=1) -- stronger than the required max relative error of 1e-5
(Q8_0/Q4_0) / 1e-4 (IQ3_S) normalised by ||y||, which is asserted as well
against the order-free float64 result."""
import numpy as np
import pytest
import torch

import oracle as O
import npref
from chimere_amd import ggml_gpu as G

pytestmark = pytest.mark.gpu
TOL = {O.Q8_0: 1e-5, O.Q4_0: 1e-5, O.IQ3_S: 1e-4}


def dev_t(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


@pytest.mark.parametrize("ncols,pad,batch", [(2048, 2048, 1), (512, 512, 8), (2000, 2048, 3), (4096, 4096, 2)])
def test_quantize_q8_1_bit_exact(dev, ncols, pad, batch):
    rng = np.random.default_rng(ncols + batch)
    x = rng.standard_normal((batch, ncols)).astype(np.float32) * np.float32(3)
    x[0, :32] = 0                                   # all-zero block
    x[-1, 40:72] = np.float32(2.0 ** 20)            # large, uniform block
    out = torch.zeros(batch, pad // 32 * 36, dtype=torch.uint8, device=dev)
    G.lib().chimere_quantize_q8_1_batched(G._ptr(dev_t(x, dev)), G._ptr(out), ncols, pad, batch, G._stream())
    G.check()
    ref = O.quantize_q8_1(x, pad)
    assert (host(out) == ref).all()


@pytest.mark.parametrize("t", [O.Q8_0, O.Q4_0, O.IQ3_S])
def test_weight_quantizers_bit_exact(dev, t):
    rng = np.random.default_rng(50 + t)
    x = rng.normal(0, 0.02, (64, 2048)).astype(np.float32)
    x[3, :256] = 0                                   # zero super-block
    x[5, :256] *= 1e4
    out = torch.zeros(64 * O.row_bytes(t, 2048), dtype=torch.uint8, device=dev)
    G.quantize_weights(t, dev_t(x, dev), out)
    assert (host(out) == O.quantize(t, x).reshape(-1)).all()


def _case(t, nrows, ncols, seed):
    rng = np.random.default_rng(seed)
    w = O.quantize(t, rng.normal(0, 0.02, (nrows, ncols)).astype(np.float32))
    x = rng.standard_normal(ncols).astype(np.float32)
    return w, x, O.quantize_q8_1(x)


SHAPES = [(4096, 2048), (37, 2048), (512, 2048), (2048, 512), (300, 8192), (16, 256), (256, 4096)]


@pytest.mark.parametrize("t", [O.Q8_0, O.Q4_0, O.IQ3_S])
@pytest.mark.parametrize("nrows,ncols", SHAPES)
def test_gemv_bit_exact(dev, t, nrows, ncols):
    print(f"gemv type={t} {nrows}x{ncols}", flush=True)
    w, x, xq = _case(t, nrows, ncols, nrows * 7 + ncols + t)
    wd, xd, xqd = dev_t(w, dev), dev_t(x, dev), dev_t(xq, dev)
    y = torch.zeros(nrows, dtype=torch.float32, device=dev)
    {O.Q8_0: G.ggml_gpu_gemv_q8_0_q8, O.Q4_0: G.ggml_gpu_gemv_q4_0_q8, O.IQ3_S: G.ggml_gpu_gemv_iq3s_q8}[t](
        wd, xqd, y, nrows, ncols)
    yg = host(y)
    yo = O.gemv(t, w, xq, ncols, nrows, L=16, G=1)
    assert (yg.view(np.uint32) == yo.view(np.uint32)).all()
    y64 = npref.gemv_f64(t, w, xq, ncols)
    assert np.linalg.norm(yg - y64) / np.linalg.norm(y64) < TOL[t]
    # block dots (debug entry point): exact int32
    bd = torch.zeros(nrows, ncols // 32, dtype=torch.int32, device=dev)
    G.block_dots(t, wd, xqd, bd, nrows, ncols)
    assert (host(bd) == O.block_dots(t, w, xq, ncols, nrows)).all()
    # fused f32 -> Q8_1 -> GEMV entry point, scratch padded to 512
    scratch = torch.zeros(G.q8_1_row_bytes(ncols), dtype=torch.uint8, device=dev)
    y2 = torch.zeros(nrows, dtype=torch.float32, device=dev)
    {O.Q8_0: G.ggml_gpu_gemv_q8_0_f32, O.Q4_0: G.ggml_gpu_gemv_q4_0_f32, O.IQ3_S: G.ggml_gpu_gemv_iq3s_f32}[t](
        wd, xd, y2, scratch, nrows, ncols)
    assert (host(y2).view(np.uint32) == yo.view(np.uint32)).all()


@pytest.mark.parametrize("t", [O.Q8_0, O.Q4_0, O.IQ3_S])
@pytest.mark.parametrize("H", [1024, 2048])
def test_gemv_batched_by_expert_ids(dev, t, H):
    """ggml_gpu_cuda.cu:243-279 semantics: slot k uses expert ids[k] and input
    k*input_stride (0 = shared).  H=2048: whole 64-block chunks (the GEMV's
    compile-time chunk path); H=1024: a partial chunk."""
    rng = np.random.default_rng(70 + t)
    E, F, K = 12, 64, 5
    w = O.quantize(t, rng.normal(0, 0.02, (E * F, H)).astype(np.float32)).reshape(E, -1)
    xs = rng.standard_normal((K, H)).astype(np.float32)
    xq = O.quantize_q8_1(xs)                        # [K, row bytes]
    ids = np.array([7, 0, 11, 7, 3], np.int32)
    fn = {O.Q8_0: G.ggml_gpu_gemv_q8_0_batched, O.Q4_0: G.ggml_gpu_gemv_q4_0_batched,
          O.IQ3_S: G.ggml_gpu_gemv_iq3s_batched}[t]
    wd, xqd, idd = dev_t(w, dev), dev_t(xq, dev), dev_t(ids, dev)
    for stride in (0, xq.shape[1]):
        y = torch.zeros(K * F, dtype=torch.float32, device=dev)
        fn(wd, xqd, y, idd, F, H, w.shape[1], stride, K)
        yg = host(y).reshape(K, F)
        for k in range(K):
            xk = xq[k] if stride else xq[0]
            yo = O.gemv(t, w[ids[k]], xk, H, F)
            assert (yg[k].view(np.uint32) == yo.view(np.uint32)).all()


@pytest.mark.parametrize("t", [O.Q8_0, O.Q4_0, O.IQ3_S])
@pytest.mark.parametrize("ntok", [1, 2, 5, 8])
def test_gemv_multi_token(dev, t, ntok):
    rng = np.random.default_rng(90 + t * 10 + ntok)
    nrows, ncols = 200, 2048
    w = O.quantize(t, rng.normal(0, 0.02, (nrows, ncols)).astype(np.float32))
    xq = O.quantize_q8_1(rng.standard_normal((ntok, ncols)).astype(np.float32))
    y = torch.zeros(ntok, nrows, dtype=torch.float32, device=dev)
    G.gemv_multi(t, dev_t(w, dev), dev_t(xq, dev), y, nrows, ncols, ntok)
    yo = O.gemv(t, w, xq, ncols, nrows, ntok=ntok, xq_stride=xq.shape[1])
    assert (host(y).reshape(ntok, nrows).view(np.uint32) == np.asarray(yo).reshape(ntok, nrows).view(np.uint32)).all()
    # the per-type entry point gives the same bits
    import ctypes as C
    from chimere_amd._lib import check, lib
    fn = {O.Q4_0: "chimere_mmvq_q4_0_multi", O.Q8_0: "chimere_mmvq_q8_0_multi", O.IQ3_S: "chimere_mmvq_iq3s_multi"}[t]
    y2 = torch.zeros_like(y)
    wd, xd = dev_t(w, dev), dev_t(xq, dev)
    getattr(lib(), fn)(C.c_void_p(wd.data_ptr()), C.c_void_p(xd.data_ptr()), C.c_void_p(y2.data_ptr()), ncols, nrows,
                       xq.shape[1] // 36, ntok, G._stream())
    check()
    assert (host(y2).view(np.uint32) == host(y).view(np.uint32)).all()


def test_gemv_synth251_fixture(dev):
    """The reference's synthetic IQ3_S bytes (fused_gate_up.rs:386-412): block
    dots equal the committed golden file."""
    import os
    W = (np.arange(16 * 8 * 110) % 251).astype(np.uint8)
    xq = np.zeros(64 * 36, np.uint8)
    for b in range(64):
        xq[b * 36 + 1] = 0x10
        xq[b * 36 + 4:b * 36 + 36] = np.arange(32) % 5
    bd = torch.zeros(16, 64, dtype=torch.int32, device=dev)
    G.block_dots(O.IQ3_S, dev_t(W, dev), dev_t(xq, dev), bd, 16, 2048)
    gold = np.load(os.path.join(os.path.dirname(__file__), "golden", "iq3s_synth251_block_dots.npy"))
    assert (host(bd) == gold).all()


def test_q4_0_head_full_size(dev):
    """Config 2 at full size (151936 x 2048 Q4_0, 175 MB): weights drawn and
    quantized on the device, GEMV checked bit-exact against the oracle on the
    same bytes, plus the linearity property y(-x) = -y(x)."""
    V, H = 151936, 2048
    g = torch.Generator(device=dev).manual_seed(2)
    wf = torch.randn(V, H, generator=g, device=dev) * 0.02
    w = torch.empty(V * H // 32 * 18, dtype=torch.uint8, device=dev)
    G.quantize_weights(O.Q4_0, wf, w)
    del wf
    x = torch.randn(H, generator=g, device=dev)
    xq = torch.zeros(G.q8_1_row_bytes(H), dtype=torch.uint8, device=dev)
    G.ggml_gpu_quantize_q8_1(x, xq, H)
    y = torch.zeros(V, dtype=torch.float32, device=dev)
    G.ggml_gpu_gemv_q4_0_q8(w, xq, y, V, H)
    yo = O.gemv(O.Q4_0, host(w), host(xq), H, V)
    yg = host(y)
    assert (yg.view(np.uint32) == yo.view(np.uint32)).all()
    G.ggml_gpu_quantize_q8_1(-x, xq, H)
    G.ggml_gpu_gemv_q4_0_q8(w, xq, y, V, H)
    assert (host(y) == -yg).all()


# ---- ggml K-quants and MXFP4 (ffi/ggml_cuda_gemv.cu:118-175, 292-460)

KQ_FN = {O.Q4_K: ("chimere_mmvq_q4k", "chimere_mmvq_q4k_f32"), O.Q5_K: ("chimere_mmvq_q5k", "chimere_mmvq_q5k_f32"),
         O.Q6_K: ("chimere_mmvq_q6k", "chimere_mmvq_q6k_f32"), O.MXFP4: ("chimere_mmvq_mxfp4", None)}
KQ_SHAPES = [(4096, 2048), (37, 2304), (300, 4096), (16, 256), (512, 4096)]


@pytest.mark.parametrize("t,nrows,ncols", [(t, r, c) for r, c in KQ_SHAPES for t in (O.Q4_K, O.Q5_K, O.Q6_K, O.MXFP4)]
                         + [(O.MXFP4, 64, 2080), (O.MXFP4, 19, 96)])
def test_kquant_gemv_bit_exact(dev, t, nrows, ncols):
    """Bit-exact against the oracle's (L=16, G=1) order; within 1e-5 of the
    float64 result; int32 block dots exact; the fused f32 entry gives the same
    bits.  (64, 2080) and (19, 96) are MXFP4-only shapes (rows not 4-byte
    aligned)."""
    print(f"kquant gemv type={t} {nrows}x{ncols}", flush=True)
    rng = np.random.default_rng(nrows * 3 + ncols + t)
    w = npref.rand_kq(t, nrows, ncols, rng)
    x = rng.standard_normal(ncols).astype(np.float32)
    pad = G.pad(ncols, 512)
    xq = O.quantize_q8_1(x, pad)
    wd, xd, xqd = dev_t(w, dev), dev_t(x, dev), dev_t(xq, dev)
    import ctypes as C
    from chimere_amd._lib import check, lib
    y = torch.zeros(nrows, dtype=torch.float32, device=dev)
    q8, f32 = KQ_FN[t]
    getattr(lib(), q8)(C.c_void_p(wd.data_ptr()), C.c_void_p(xqd.data_ptr()), C.c_void_p(y.data_ptr()), ncols,
                       nrows, pad // 32, G._stream())
    check()
    yg = host(y)
    yo = O.gemv(t, w, xq, ncols, nrows, L=16, G=1)
    assert (yg.view(np.uint32) == yo.view(np.uint32)).all()
    y64 = npref.kq_gemv_f64(t, w, xq, ncols)
    assert np.linalg.norm(yg - y64) / np.linalg.norm(y64) < 1e-5
    bd = torch.zeros(nrows, ncols // 32, dtype=torch.int32, device=dev)
    G.block_dots(t, wd, xqd, bd, nrows, ncols)
    assert (host(bd) == O.block_dots(t, w, xq, ncols, nrows)).all()
    scratch = torch.zeros(pad // 32 * 36, dtype=torch.uint8, device=dev)
    y2 = torch.zeros(nrows, dtype=torch.float32, device=dev)
    {O.Q4_K: G.ggml_gpu_gemv_q4k_f32, O.Q5_K: G.ggml_gpu_gemv_q5k_f32, O.Q6_K: G.ggml_gpu_gemv_q6k_f32,
     O.MXFP4: G.ggml_gpu_gemv_mxfp4_f32}[t](wd, xd, y2, scratch, nrows, ncols)
    assert (host(y2).view(np.uint32) == yo.view(np.uint32)).all()


@pytest.mark.parametrize("t", [O.Q4_K, O.Q5_K, O.Q6_K, O.MXFP4])
def test_kquant_multi_token(dev, t):
    rng = np.random.default_rng(400 + t)
    nrows, ncols, ntok = 100, 2048, 3
    w = npref.rand_kq(t, nrows, ncols, rng)
    xq = O.quantize_q8_1(rng.standard_normal((ntok, ncols)).astype(np.float32))
    y = torch.zeros(ntok, nrows, dtype=torch.float32, device=dev)
    G.gemv_multi(t, dev_t(w, dev), dev_t(xq, dev), y, nrows, ncols, ntok)
    yo = O.gemv(t, w, xq, ncols, nrows, ntok=ntok, xq_stride=xq.shape[1])
    assert (host(y).view(np.uint32) == np.asarray(yo).view(np.uint32)).all()


def test_mxfp4_batched_device_ids(dev):
    """chimere_mmvq_mxfp4_batched reads the expert ids on the device (the
    reference's host-side dereference, ggml_cuda_gemv.cu:438-444, is not kept)."""
    rng = np.random.default_rng(39)
    E, F, H, K = 6, 48, 1024, 4
    w = npref.rand_kq(O.MXFP4, E * F, H, rng).reshape(E, -1)
    xq = O.quantize_q8_1(rng.standard_normal((K, H)).astype(np.float32))
    ids = np.array([5, 0, 5, 2], np.int32)
    wd, xqd, idd = dev_t(w, dev), dev_t(xq, dev), dev_t(ids, dev)
    for stride in (0, xq.shape[1]):
        y = torch.zeros(K * F, dtype=torch.float32, device=dev)
        G.ggml_gpu_gemv_mxfp4_batched(wd, xqd, y, idd, F, H, w.shape[1], stride, K)
        yg = host(y).reshape(K, F)
        for k in range(K):
            yo = O.gemv(O.MXFP4, w[ids[k]], xq[k] if stride else xq[0], H, F)
            assert (yg[k].view(np.uint32) == yo.view(np.uint32)).all()


@pytest.mark.parametrize("nrows,ncols", [(4096, 2048), (37, 2048), (2048, 512), (300, 8192)])
def test_gemv_q4_0_sform_bit_exact(dev, nrows, ncols):
    """ggml's s-form Q4_0 block term (chimere_mmvq_q4_0_sform) against the
    oracle's restatement, bit for bit; and within the bound of the exact form."""
    print(f"gemv q4_0 s-form {nrows}x{ncols}", flush=True)
    w, x, xq = _case(O.Q4_0, nrows, ncols, nrows * 11 + ncols)
    wd, xqd = dev_t(w, dev), dev_t(xq, dev)
    ys = torch.zeros(nrows, dtype=torch.float32, device=dev)
    ye = torch.zeros(nrows, dtype=torch.float32, device=dev)
    G.ggml_gpu_gemv_q4_0_sform_q8(wd, xqd, ys, nrows, ncols)
    G.ggml_gpu_gemv_q4_0_q8(wd, xqd, ye, nrows, ncols)
    gs, ge = host(ys), host(ye)
    assert (gs.view(np.uint32) == O.gemv(O.Q4_0_SFORM, w, xq, ncols, nrows).view(np.uint32)).all()
    assert (ge.view(np.uint32) == O.gemv(O.Q4_0, w, xq, ncols, nrows).view(np.uint32)).all()
    # the forms differ by at most sum_b 8 |d_w| |s_x - d_x * sum(q_x)| per row (+ fp32 rounding)
    nb = ncols // 32
    xb = xq[:nb * 36].reshape(nb, 36)
    f16 = lambda b: np.frombuffer(np.ascontiguousarray(b).tobytes(), np.float16).astype(np.float64)  # noqa: E731
    dx, sx = f16(xb[:, 0:2]), f16(xb[:, 2:4])
    sq = xb[:, 4:].view(np.int8).astype(np.int64).sum(axis=1)
    dw = f16(w.reshape(nrows, nb, 18)[:, :, :2]).reshape(nrows, nb)
    bound = (8 * np.abs(dw) * np.abs(sx - dx * sq)[None, :]).sum(axis=1)
    diff = np.abs(gs.astype(np.float64) - ge)
    assert (diff <= bound + 1e-5 * np.abs(ge).max()).all() and diff.max() > 0


@pytest.mark.parametrize("t", [O.Q8_0, O.Q4_0, O.IQ3_S, O.Q4_K, O.Q5_K, O.Q6_K, O.MXFP4])
@pytest.mark.parametrize("nrows,ncols", [
    (16, 256), (37, 2048), (64, 4096), (33, 2304), (48, 6144),   # one launch: whole and ragged chunks and tiles
    (16384, 2048), (16385, 2048), (8192, 4096), (8193, 4096),    # the last one-launch size and the next
])
def test_f32_gemv_is_quantizer_plus_gemv(dev, t, nrows, ncols):
    """The f32 entry points in one launch and in two: the output bits and the
    scratch bytes (zero blocks up to the padded length included) of the
    quantizer followed by the Q8_1 entry point; an input that is not 16-byte
    aligned gives the same."""
    rng = np.random.default_rng(nrows + ncols + t)
    w = torch.randint(0, 120, (nrows * O.row_bytes(t, ncols),), dtype=torch.uint8, device=dev,
                      generator=torch.Generator(device=dev).manual_seed(t))
    x = rng.standard_normal(ncols).astype(np.float32)
    x[:32] = 0
    x[40:50] *= np.float32(1e-44)
    pad = G.pad(ncols, 512)
    xq = dev_t(O.quantize_q8_1(x, pad), dev)
    want = torch.zeros(nrows, device=dev)
    G.gemv_multi(t, w, xq, want, nrows, ncols, 1)
    fn = {O.Q8_0: G.ggml_gpu_gemv_q8_0_f32, O.Q4_0: G.ggml_gpu_gemv_q4_0_f32, O.IQ3_S: G.ggml_gpu_gemv_iq3s_f32,
          O.Q4_K: G.ggml_gpu_gemv_q4k_f32, O.Q5_K: G.ggml_gpu_gemv_q5k_f32, O.Q6_K: G.ggml_gpu_gemv_q6k_f32,
          O.MXFP4: G.ggml_gpu_gemv_mxfp4_f32}[t]
    buf = torch.empty(ncols + 4, device=dev)
    for off in (0, 1):
        xd = buf[off:off + ncols]
        xd.copy_(dev_t(x, dev))
        scratch = torch.full((pad // 32 * 36,), 255, dtype=torch.uint8, device=dev)
        y = torch.zeros(nrows, device=dev)
        fn(w, xd, y, scratch, nrows, ncols)
        assert (host(scratch) == host(xq).reshape(-1)).all()
        assert (host(y).view(np.uint32) == host(want).view(np.uint32)).all()


@pytest.mark.parametrize("t", [O.Q8_0, O.Q4_0, O.IQ3_S, O.Q4_K, O.Q5_K, O.Q6_K, O.MXFP4])
@pytest.mark.parametrize("nrows,ncols,ntok,off", [
    (16, 256, 4, 0), (35, 2048, 4, 0), (50, 2304, 8, 0),      # fewer than 16 blocks; short tiles; a ragged chunk
    (33, 4096, 6, 0), (64, 2048, 7, 0), (20, 1280, 8, 4),     # short token groups; inputs only 4-byte aligned
])
def test_multi_token_on_matrix_cores(dev, t, nrows, ncols, ntok, off):
    """Four and six to eight tokens (the 16-slot matrix products): bit-exact
    against the oracle's (L=16, G=1) order."""
    print(f"multi type={t} {nrows}x{ncols} ntok={ntok} off={off}", flush=True)
    rng = np.random.default_rng(nrows + ncols + ntok + t)
    if t in (O.Q8_0, O.Q4_0, O.IQ3_S):
        w = O.quantize(t, rng.normal(0, 0.02, (nrows, ncols)).astype(np.float32))
    else:
        w = npref.rand_kq(t, nrows, ncols, rng)
    x = rng.standard_normal((ntok, ncols)).astype(np.float32)
    x[0, :32] = 0
    xq = O.quantize_q8_1(x)
    buf = torch.zeros(xq.size + 16, dtype=torch.uint8, device=dev)
    buf[off:off + xq.size] = dev_t(xq, dev).reshape(-1)
    y = torch.zeros(ntok, nrows, dtype=torch.float32, device=dev)
    G.gemv_multi(t, dev_t(w, dev), buf[off:], y, nrows, ncols, ntok)
    yo = O.gemv(t, w, xq, ncols, nrows, ntok=ntok, xq_stride=xq.shape[1])
    assert (host(y).view(np.uint32) == np.asarray(yo).reshape(ntok, nrows).view(np.uint32)).all()


SUPER = [(37, 256, 1), (16, 1280, 1), (50, 4352, 1), (33, 2816, 2), (35, 768, 4), (20, 4352, 8)]
BLOCKS = [(37, 96, 1), (35, 96, 4), (20, 2080, 4), (33, 2080, 7), (17, 4192, 8), (50, 4192, 1)]


@pytest.mark.parametrize("t,nrows,ncols,ntok,off", [
    (t, *s, off) for t in (O.IQ3_S, O.Q6_K, O.MXFP4) for s in SUPER for off in (0, 2, 6)
] + [(O.MXFP4, *s, off) for s in BLOCKS for off in (0, 1, 7)     # 17-byte blocks: rows at odd bytes too
] + [(t, *s, off) for t in (O.Q4_0, O.Q8_0) for s in BLOCKS for off in (0, 2)])
def test_gemv_unaligned_rows(dev, t, nrows, ncols, ntok, off):
    """Rows that start anywhere in a 16-byte granule (an odd number of
    superblocks, or of 32-element blocks), whole and ragged chunks, matrices at
    any even address (MXFP4: any): bit-exact against the oracle's (L=16, G=1)
    order."""
    print(f"unaligned type={t} {nrows}x{ncols} ntok={ntok} off={off}", flush=True)
    rng = np.random.default_rng(nrows + ncols + ntok + t + off)
    w = (O.quantize(t, rng.normal(0, 0.02, (nrows, ncols)).astype(np.float32)) if t in (O.IQ3_S, O.Q4_0, O.Q8_0)
         else npref.rand_kq(t, nrows, ncols, rng))
    xq = O.quantize_q8_1(rng.standard_normal((ntok, ncols)).astype(np.float32))
    buf = torch.zeros(w.size + 32, dtype=torch.uint8, device=dev)
    buf[off:off + w.size] = dev_t(w, dev).reshape(-1)
    y = torch.zeros(ntok, nrows, dtype=torch.float32, device=dev)
    G.gemv_multi(t, buf[off:], dev_t(xq, dev), y, nrows, ncols, ntok)
    yo = O.gemv(t, w, xq, ncols, nrows, ntok=ntok, xq_stride=xq.shape[1])
    assert (host(y).view(np.uint32) == np.asarray(yo).reshape(ntok, nrows).view(np.uint32)).all()


@pytest.mark.parametrize("t", [O.Q8_0, O.Q4_0, O.Q5_K])
@pytest.mark.parametrize("n,shift", [(2048, 0), (2048, 1024), (2048, -1024), (2304, 0), (4096, 0), (8192, 0)])
def test_f32_gemv_output_over_input(dev, t, n, shift):
    """A square projection whose output is its input's buffer (shift 0) or a
    view that overlaps half of it: the bits of the call with its own output.
    Disjoint buffers of all sizes but the last take a single launch, in which
    later work-groups would read outputs that earlier ones stored."""
    print(f"f32 output over input type={t} n={n} shift={shift}", flush=True)
    rng = np.random.default_rng(n + t)
    # random blocks, f16 scales below 1
    w = torch.randint(0, 60, (n * O.row_bytes(t, n),), dtype=torch.uint8, device=dev,
                      generator=torch.Generator(device=dev).manual_seed(t))
    x = dev_t(rng.standard_normal(n).astype(np.float32), dev)
    fn = {O.Q8_0: G.ggml_gpu_gemv_q8_0_f32, O.Q4_0: G.ggml_gpu_gemv_q4_0_f32, O.Q5_K: G.ggml_gpu_gemv_q5k_f32}[t]
    scratch = torch.empty(G.q8_1_row_bytes(n), dtype=torch.uint8, device=dev)
    want = torch.zeros(n, device=dev)
    fn(w, x, want, scratch, n, n)
    want = host(want).view(np.uint32)
    buf = torch.zeros(n + 2 * abs(shift), device=dev)
    xv = buf[abs(shift):abs(shift) + n]
    yv = buf[abs(shift) + shift:abs(shift) + shift + n]
    for _ in range(3):
        xv.copy_(x)
        fn(w, xv, yv, scratch, n, n)
        assert (host(yv).view(np.uint32) == want).all()


@pytest.mark.parametrize("where", ["row", "output"])
def test_f32_gemv_scratch_over_row_or_output(dev, where):
    """One 32-element block: a scratch that starts where the row does (the
    quantizer's wave reads the block before it writes), and an output over the
    scratch's zero blocks past the row's own (which no GEMV reads): the bits of
    the call with buffers of its own."""
    import ctypes as C
    from chimere_amd._lib import check, lib
    n, nrows, pad = 32, 2048, 32 if where == "row" else 512
    rng = np.random.default_rng(7)
    w = dev_t(O.quantize(O.Q8_0, rng.normal(0, 0.02, (nrows, n)).astype(np.float32)), dev)
    x = rng.standard_normal(n).astype(np.float32)
    want = np.asarray(O.gemv(O.Q8_0, host(w), O.quantize_q8_1(x), n, nrows)).reshape(-1)
    buf = torch.zeros(nrows + 1024, device=dev)
    # floats: row, scratch, output
    xo, so, yo = (0, 0, 256) if where == "row" else (nrows + 512, 0, 9)
    for _ in range(3):
        buf.zero_()
        buf[xo:xo + n] = dev_t(x, dev)
        p = [C.c_void_p(buf.data_ptr() + 4 * o) for o in (xo, yo, so)]
        lib().chimere_mmvq_q8_0_f32(C.c_void_p(w.data_ptr()), p[0], p[1], n, nrows, pad, p[2], G._stream())
        check()
        assert (host(buf[yo:yo + nrows]).view(np.uint32) == want.view(np.uint32)).all()


@pytest.mark.parametrize("t", [O.Q8_0, O.Q6_K, O.IQ3_S])
@pytest.mark.parametrize("ncols", [4096, 6144, 7168, 8192])
def test_f32_gemv_many_chunks(dev, t, ncols):
    """Rows on both sides of the f32 entry points' lines (one launch up to two or
    three chunks, any number for rows off the 16-byte grid): the bits of
    the quantizer launch and the GEMV."""
    print(f"f32 many chunks type={t} ncols={ncols}", flush=True)
    rng = np.random.default_rng(ncols + t)
    nrows = 100
    w = dev_t(O.quantize(t, rng.normal(0, 0.02, (nrows, ncols)).astype(np.float32)) if t != O.Q6_K
              else npref.rand_kq(t, nrows, ncols, rng), dev)
    x = dev_t(rng.standard_normal(ncols).astype(np.float32), dev)
    fn = {O.Q8_0: G.ggml_gpu_gemv_q8_0_f32, O.Q6_K: G.ggml_gpu_gemv_q6k_f32, O.IQ3_S: G.ggml_gpu_gemv_iq3s_f32}[t]
    scratch, xq = (torch.full((G.q8_1_row_bytes(ncols),), 7, dtype=torch.uint8, device=dev) for _ in range(2))
    y, y2 = torch.zeros(nrows, device=dev), torch.zeros(1, nrows, device=dev)
    fn(w, x, y, scratch, nrows, ncols)
    G.ggml_gpu_quantize_q8_1_batched(x, xq, ncols, 1)
    G.gemv_multi(t, w, xq, y2, nrows, ncols, 1)
    assert (host(y).view(np.uint32) == host(y2)[0].view(np.uint32)).all()
    assert (host(scratch) == host(xq)).all()


@pytest.mark.parametrize("t", [O.Q4_K, O.Q5_K])
@pytest.mark.parametrize("nrows", [4096, 4099])
def test_seven_tokens_both_kernels(dev, t, nrows):
    """Seven tokens of the types with a min term, with one work-group per CU and
    with one more (Q5_K: the matrix-core kernel, the other one): bit-exact
    against the oracle."""
    print(f"seven tokens type={t} nrows={nrows}", flush=True)
    rng = np.random.default_rng(nrows + t)
    w = npref.rand_kq(t, nrows, 512, rng)
    xq = O.quantize_q8_1(rng.standard_normal((7, 512)).astype(np.float32))
    y = torch.zeros(7, nrows, device=dev)
    G.gemv_multi(t, dev_t(w, dev), dev_t(xq, dev), y, nrows, 512, 7)
    yo = O.gemv(t, w, xq, 512, nrows, ntok=7, xq_stride=xq.shape[1])
    assert (host(y).view(np.uint32) == np.asarray(yo).reshape(7, nrows).view(np.uint32)).all()
