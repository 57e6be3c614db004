"""The one-call products and layers in both of their forms: built for a
caller's buffers (the default, which test_gpu_ops.py checks) and the model's
(SURGE_ONESHOT=model: weights repacked into planes, a position ring for the
conv, attention rows prepared in place). The model's forms pass the same
per-op tests; where both run the same arithmetic they give the same bits."""
import ctypes as C

import numpy as np
import pytest

import surge_amd as S
import test_gpu_ops as T

pytestmark = pytest.mark.gpu


@pytest.fixture
def model_forms(monkeypatch):
    monkeypatch.setenv("SURGE_ONESHOT", "model")


# ---------------------------------------------------------------- the per-op tests on the model's forms

def test_gemv_planes_scale_decode(gpu, model_forms):
    T.test_gemv_q8_scale_decode_exact_all_f16_patterns(gpu)


def test_gemv_planes_4096(gpu, model_forms):
    T.test_gemv_q8_baseline_config_4096(gpu)


@pytest.mark.parametrize("rows,cols", [(1, 32), (37, 64), (3, 17408), (5120, 6144), (16480, 5120), (40000, 2048), (7, 96)])
def test_gemv_planes_shapes(gpu, model_forms, rows, cols):
    """k_gemv_q8, and k_gemv_bal at 5120, 6144 and 17408 columns."""
    T.test_gemv_q8_shapes(gpu, rows, cols)


@pytest.mark.parametrize("N,M,K", [(70, 130, 256), (300, 260, 96), (1, 32, 32), (129, 384, 1056)])
def test_gemm_planes(gpu, model_forms, N, M, K):
    T.test_matmul_q8_prefill_gemm(gpu, N, M, K)


@pytest.mark.parametrize("N,M,K", [(2, 5, 32), (17, 129, 96), (33, 260, 1120), (48, 31, 6144), (49, 128, 2080), (80, 257, 544),
                                   (81, 130, 288)])
def test_gemm_planes_few_tokens(gpu, model_forms, N, M, K):
    T.test_matmul_q8_few_tokens(gpu, N, M, K)


def test_gemm_planes_round_split(gpu, model_forms, monkeypatch):
    T.test_matmul_q8_prefill_gemm_round_split(gpu, monkeypatch, "wide", "14")


@pytest.mark.parametrize("nv,nk,dk,dv,ks,tiled", T.GDN_CASES)
def test_gdn_step_ring(gpu, model_forms, nv, nk, dk, dv, ks, tiled):
    T.test_gdn_decode_step_vs_oracle(gpu, nv, nk, dk, dv, ks, tiled)


@pytest.mark.parametrize("nv,nk,dk,dv,ks,tiled,n1,n2", T.GDN_CHUNK_CASES + [(48, 16, 128, 128, 4, True, 215, 1)])
def test_gdn_chunk_ring(gpu, model_forms, nv, nk, dk, dv, ks, tiled, n1, n2):
    """k_conv_chunk on the ring, four and sixteen tokens per thread, the ring
    written by k_dm_prep and by k_conv_window, from ring slots 1 and 2."""
    T.test_gdn_prefill_chunk_vs_oracle(gpu, nv, nk, dk, dv, ks, tiled, n1, n2)


@pytest.mark.parametrize("nh,nkv,hd,rd,base,n", T.ATTN_CHUNK_CASES + [(8, 2, 256, 64, 1024, 77)])
def test_attn_chunk_in_place(gpu, model_forms, nh, nkv, hd, rd, base, n):
    T.test_attn_prefill_chunk_vs_oracle(gpu, nh, nkv, hd, rd, base, n)


# ---------------------------------------------------------------- the same bits in both forms

def _forms(monkeypatch, call):
    """call()'s arrays in the caller's form, then in the model's."""
    got = [call()]
    monkeypatch.setenv("SURGE_ONESHOT", "model")
    got.append(call())
    return got


@pytest.mark.parametrize("N,M,K", [(1, 40, 64), (40, 300, 2080), (80, 257, 5120), (81, 130, 288), (300, 1100, 544),
                                   (640, 33, 64)])
def test_matmul_forms_agree(gpu, monkeypatch, N, M, K):
    rng = np.random.default_rng(N)
    X, raw = rng.standard_normal(N * K).astype(np.float32), T.q8_matrix(rng, M, K, sigma=1.0)

    def call():
        yb = gpu.buf(np.zeros(N * M, np.float32))
        gpu.run_op("k_matmul_q8", gpu.buf(X), gpu.buf(raw), yb, [N, M, K])
        return yb.array.copy()
    a, b = _forms(monkeypatch, call)
    assert np.array_equal(a, b)


@pytest.mark.parametrize("nv,nk,dk,dv,ks,n", [(48, 16, 128, 128, 4, 45), (4, 2, 64, 64, 2, 1), (4, 4, 256, 32, 3, 18),
                                              (3, 3, 32, 5, 1, 9)])
def test_gdn_chunk_forms_agree(gpu, monkeypatch, nv, nk, dk, dv, ks, n):
    rng = np.random.default_rng(n)
    cd, vd = 2 * nk * dk + nv * dv, nv * dv
    w = np.concatenate([rng.standard_normal(cd * ks) * 0.5, -np.exp(rng.uniform(-1, 1, nv)), rng.uniform(-0.5, 0.5, nv),
                        1.0 + 0.1 * rng.standard_normal(dv)]).astype(np.float32)
    state = rng.standard_normal((ks - 1) * cd + vd * dk).astype(np.float32)
    inp = rng.standard_normal(n * (cd + vd + 2 * nv)).astype(np.float32)

    def call():
        sb, ob = gpu.buf(state.copy()), gpu.buf(np.zeros(n * vd, np.float32))
        gpu.gdn_chunk(gpu.buf(inp), gpu.buf(w), sb, ob, [dk, dv, nv, nk, ks, 3 | 3 << 2, n, S.fbits(1e-6)])
        return np.concatenate([ob.array, sb.array])
    a, b = _forms(monkeypatch, call)
    assert np.array_equal(a, b)


@pytest.mark.parametrize("nh,nkv,hd,rd,base,n", [(24, 4, 256, 64, 700, 90), (6, 6, 64, 62, 0, 3), (12, 4, 128, 128, 1500, 130)])
def test_attn_chunk_forms_agree(gpu, monkeypatch, nh, nkv, hd, rd, base, n):
    rng = np.random.default_rng(base + n)
    inp = rng.standard_normal(n * (2 * nh + 2 * nkv) * hd).astype(np.float32)
    w = (1.0 + 0.1 * rng.standard_normal(2 * hd)).astype(np.float32)
    kv = rng.standard_normal(2 * (base + n) * nkv * hd).astype(np.float16).view(np.uint16)

    def call():
        kvb, ob = gpu.buf(kv.copy()), gpu.buf(np.zeros(n * nh * hd, np.float32))
        gpu.attn_chunk(gpu.buf(inp), gpu.buf(w), kvb, ob, [nh, nkv, hd, rd, base, n, S.fbits(1e7), S.fbits(1e-6)])
        return np.concatenate([ob.array.view(np.uint16), kvb.array])
    a, b = _forms(monkeypatch, call)
    assert np.array_equal(a, b)


def test_oneshot_value_is_checked(gpu, monkeypatch):
    monkeypatch.setenv("SURGE_ONESHOT", "planes")
    with pytest.raises(S.SurgeError):
        gpu.run_op("k_scale", gpu.buf(np.ones(4, np.float32)), None, gpu.buf(np.ones(4, np.float32)), [4, S.fbits(2.0)])


# ---------------------------------------------------------------- blocks off their natural alignment

@pytest.mark.parametrize("off", [1, 2, 6])
@pytest.mark.parametrize("N", [2, 40, 80, 81, 300])
def test_matmul_on_blocks_anywhere(gpu, N, off):
    """The products on a caller's blocks at addresses that no load is aligned
    to, the last row's last block ending where the buffer ends: the bits of the
    aligned call."""
    M, K = 131, 544
    rng = np.random.default_rng(N)
    X, raw = rng.standard_normal(N * K).astype(np.float32), T.q8_matrix(rng, M, K, sigma=1.0)
    xb, wb, ya, yb = (gpu.buf(a) for a in (X, raw, np.zeros(N * M, np.float32), np.zeros(N * M, np.float32)))
    gpu.run_op("k_matmul_q8", xb, wb, ya, [N, M, K])
    held = gpu.buf(np.concatenate([np.zeros(off, np.uint8), raw]))
    S.check(S.lib().sg_gpu_buf_upload(held.handle))
    h = C.c_void_p()
    S.check(S.lib().sg_gpu_wrap_device(gpu.handle, S.lib().sg_gpu_buf_device(held.handle) + off, raw.size, C.byref(h)))
    S.check(S.lib().sg_gpu_run_op(gpu.handle, b"k_matmul_q8", xb.handle, h, yb.handle, S.params([N, M, K])))
    S.lib().sg_gpu_buf_free(h)
    held.free()
    assert np.array_equal(yb.array, ya.array)
