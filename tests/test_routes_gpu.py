"""Which kernel a call launches, where a rule on sizes chooses between forms: the
launches of one call as torch's profiler records them."""
import json

import pytest
import torch
from torch.profiler import ProfilerActivity, profile

from helm_amd import kernels as hk
from helm_amd.kernels import attention as ka
from helm_amd.kernels import fused

pytestmark = pytest.mark.gpu


def launches(fn, tmp_path):
    """(kernel name, workgroups) of each launch of the second of two calls, in order."""
    fn()
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA], acc_events=True) as p:
        fn()
        torch.cuda.synchronize()
    path = tmp_path / "trace.json"
    p.export_chrome_trace(str(path))
    events = [e for e in json.loads(path.read_text())["traceEvents"] if e.get("cat") == "kernel"]
    out = []
    for e in sorted(events, key=lambda e: e["ts"]):
        gx, gy, gz = e["args"]["grid"]
        out.append((e["name"].replace("(anonymous namespace)::", "").removeprefix("void "), gx * gy * gz))
    assert out, "no launch was recorded"
    return out


def int8_weights(N, K):
    return (torch.randint(-127, 128, (N, K), dtype=torch.int8, device="cuda"),
            torch.rand(N, device="cuda").half())


@pytest.mark.parametrize("tn", [2, 4, 5])
@pytest.mark.parametrize("M,N,K", [(130, 200, 320), (300, 1000, 1024), (257, 700, 2048), (17, 64, 64)])
def test_gemm_tile_width_override(M, N, K, tn, monkeypatch, tmp_path):
    """HELM_GEMM_TN takes the prompt form of that width for every shape, also one the
    few-row form would take."""
    x = torch.randn(M, K, device="cuda").half()
    q, s = int8_weights(N, K)
    monkeypatch.setenv("HELM_GEMM_TN", str(tn))
    (name, _), = launches(lambda: hk.int8_linear(x, q, s), tmp_path)
    assert name.startswith(f"int8_gemm_kernel<{tn}, {'true' if tn >= 4 else 'false'}, 4, 3, false"), name


@pytest.mark.parametrize("M,N,K,split", [(100, 9728, 2560, False), (97, 9728, 2560, False), (96, 9728, 2560, True),
                                         (100, 12288, 4096, True), (100, 6144, 2560, True), (64, 4096, 4096, True)])
def test_gemm_slices_by_price(M, N, K, split, tmp_path):
    """The few-row form cuts K where that pays (its second pass adds the slices)."""
    x = torch.randn(M, K, device="cuda").half()
    q, s = int8_weights(N, K)
    seen = launches(lambda: hk.int8_linear(x, q, s), tmp_path)
    assert seen[0][0].startswith("int8_gemm_kernel<"), seen
    assert [n.startswith("gemm_split_reduce_kernel") for n, _ in seen[1:]] == [True] * split, seen


LDS, REGS, STREAM = "fp16_small_m_kernel<", "xreg_gemv_kernel<false", "gemv_stream_kernel<"


@pytest.mark.parametrize("M,N,K,norm,kernel", [
    (8, 14336, 2560, True, REGS), (8, 14337, 2560, True, LDS), (4, 14337, 3072, False, LDS),
    (4, 20480, 3584, True, REGS), (13, 20481, 3584, False, LDS), (5, 20481, 4608, True, LDS),
    (16, 20481, 4608, True, REGS),          # its x rows exceed LDS
    (8, 32000, 4096, True, REGS), (8, 32000, 2048, False, REGS),
    (5, 65536, 5120, False, REGS), (12, 65537, 5120, True, LDS), (16, 65537, 5120, True, REGS),
    (4, 5000, 1920, True, LDS), (3, 5000, 1920, True, REGS),
    (3, 4096, 2560, True, STREAM), (3, 4097, 2560, True, REGS), (3, 4096, 2560, False, REGS),
    (3, 4096, 4096, True, STREAM), (3, 4096, 5120, True, REGS)])
def test_fp16_form_by_size(M, N, K, norm, kernel, tmp_path):
    """Either side of each line of the rule for fp16 weights, and the result there
    (fp32 accumulation and one rounding; with the norm one step of an fp16 operand
    more)."""
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device="cuda").half()
    w = (torch.randn(N, K, generator=g, device="cuda") * 0.02).half()
    nw = (1 + 0.1 * torch.randn(K, generator=g, device="cuda")).half()
    run = (lambda: fused.fp16_gemv_rmsnorm(x, nw, 1e-6, w)) if norm else (lambda: hk.fp16_linear(x, w))
    (name, _), = launches(run, tmp_path)
    assert name.startswith(kernel), name
    rows = torch.randperm(N, generator=g, device="cuda")[:4000]
    rows[0], rows[1] = N - 1, 0
    xn = x.float()
    if norm:
        xn = (nw.float() * (xn * torch.rsqrt(xn.square().mean(-1, keepdim=True) + 1e-6)).half().float()).half()
    ws = w[rows].double().t().contiguous()
    exact = torch.mm(xn.double(), ws)
    mag = torch.mm(xn.double().abs(), ws.abs())
    bound = mag * 2.0 ** -22 + exact.abs() * 2.0 ** -11 + 2.0 ** -24
    if norm:      # x * rsqrt may round to the neighbouring fp16 value
        bound += mag * 2.0 ** -10
    assert ((run()[:, rows].double() - exact).abs() <= bound).all()


RES, RING, REG8 = "int8_small_m_resident_kernel<", "int8_small_m_kernel<", "xreg_gemv_kernel<true"


@pytest.mark.parametrize("M,N,K,kernel", [
    (3, 1000, 4096, RES), (16, 4097, 4096, RES),
    (11, 2048, 2048, REG8), (12, 4096, 2048, RING), (12, 4097, 2048, REG8),
    (7, 4096, 6144, RING), (8, 4096, 6144, REG8), (7, 3328, 6144, REG8), (7, 4097, 6144, REG8),
    (12, 8192, 6144, RES), (11, 8192, 6144, REG8), (12, 8128, 6144, REG8),
    # k slices of 3072 in one round of workgroups, the other form walking 10 units or more
    (8, 4096, 9216, RES), (8, 4000, 9216, REG8), (12, 4096, 12288, RES), (12, 4092, 12288, RES),
    (16, 3844, 12288, RES), (9, 3072, 12288, REG8), (9, 4100, 12288, REG8), (8, 2048, 24576, RES),
    (12, 3072, 15360, RES), (12, 4092, 15360, REG8), (8, 4098, 12288, REG8),
    # all of x^T in LDS
    (4, 1040, 12288, RES), (4, 1024, 12288, REG8), (3, 5120, 12288, REG8), (4, 8192, 12288, RES),
    # ring
    (16, 4096, 8192, RING), (16, 4097, 8192, REG8), (16, 3344, 7168, RING), (9, 3328, 8192, REG8),
    (8, 3328, 8192, RING), (6, 2048, 8192, RING), (7, 2048, 8192, REG8), (10, 8192, 7168, RING),
    (10, 4096, 14336, RING), (11, 4096, 14336, REG8), (4, 3072, 16384, RING), (5, 3072, 16384, REG8),
    (4, 3072, 15360, REG8), (7, 4096, 17408, RING), (8, 4096, 17408, REG8), (8, 5120, 17408, REG8)])
def test_int8_form_by_size(M, N, K, kernel, tmp_path):
    """Either side of each line of the rule for int8 weights at 3-16 tokens, and the
    result there (exact products, fp32 accumulation, one rounding)."""
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device="cuda").half()
    q = torch.randint(-127, 128, (N, K), dtype=torch.int8, generator=g, device="cuda")
    s = (torch.rand(N, generator=g, device="cuda") * 1e-2).half()
    seen = launches(lambda: hk.int8_linear(x, q, s), tmp_path)
    assert seen[0][0].startswith(kernel), seen
    if kernel == RES and K != 4096 and M >= 8:
        assert seen[1][0].startswith("small_m_split_reduce_kernel"), seen
    qs = q.double().t().contiguous()
    exact = torch.mm(x.double(), qs) * s.double()
    mag = torch.mm(x.double().abs(), qs.abs()) * s.double()
    bound = mag * 2.0 ** -22 + exact.abs() * 2.0 ** -11 + 2.0 ** -24
    y = hk.int8_linear(x, q, s)
    assert ((y.double() - exact).abs() <= bound).all()
    assert torch.equal(hk.int8_linear(x, q, s), y)


@pytest.mark.parametrize("T,Hq,Hkv,D,prompt", [
    (204, 32, 8, 128, False), (214, 32, 8, 128, True), (191, 64, 8, 128, False), (192, 64, 8, 128, True),
    (1000, 8, 1, 128, False), (1024, 8, 1, 128, True), (300, 16, 8, 128, False),
    (227, 14, 2, 64, False), (228, 14, 2, 64, True), (341, 8, 2, 64, False), (342, 8, 2, 64, True)])
def test_kv_write_form_by_rows(T, Hq, Hkv, D, prompt, tmp_path):
    """A prompt's q / k norm, RoPE and page write takes its prompt form from 192
    tokens and 10240 (D = 64: 4096) rows on (the bits are the same in either)."""
    dev = torch.device("cuda")
    P, n = 16, -(-T // 16)
    pool = ka.PoolView.of_pool(torch.zeros(n, Hkv, P, D, dtype=torch.float16, device=dev),
                               ka.alloc_v((n, Hkv, P, D), torch.float16, dev, zero=True))
    qkv = torch.randn(T, (Hq + 2 * Hkv) * D, device=dev).half()
    w = torch.ones(D, dtype=torch.float16, device=dev)
    pos = torch.arange(T, dtype=torch.int32, device=dev)
    q = torch.empty(T, Hq, D, dtype=torch.float16, device=dev)
    args = (qkv, w, w, 1e-6, pos, fused.rope_inv_freq(D, 1e6, dev), q, pool, pos // P, pos % P, Hq, Hkv, D, P)
    (name, _), = launches(lambda: fused.qk_norm_rope_append(*args), tmp_path)
    assert name.startswith("qk_norm_rope_append_prompt_kernel" if prompt else "qk_norm_rope_append_kernel"), name


@pytest.mark.parametrize("T,past,Hq,Hkv,D,workgroups", [
    (96, 0, 40, 8, 128, 40), (97, 0, 40, 8, 128, 8 * 4), (17, 0, 28, 4, 64, 28), (1, 0, 8, 1, 128, 8),
    (130, 0, 8, 8, 64, 16)])
@pytest.mark.parametrize("masked", [False, True])
def test_prefill_blocks_by_queries(T, past, Hq, Hkv, D, workgroups, masked, tmp_path):
    """One pass over few queries keeps one head per 128-row block (up to 96 of them),
    longer prompts pack the heads of a group."""
    dev = torch.device("cuda")
    P, n = 16, -(-(past + T) // 16)
    pool = ka.PoolView.of_pool(torch.zeros(n, Hkv, P, D, dtype=torch.float16, device=dev),
                               ka.alloc_v((n, Hkv, P, D), torch.float16, dev, zero=True))
    q = torch.randn(T, Hq, D, device=dev).half()
    table = torch.arange(n, dtype=torch.int32, device=dev)
    mask = torch.ones(1, T, T, dtype=torch.bool, device=dev) if masked else None
    seen = launches(lambda: ka.prefill_attention(q, pool, table, P, past, mask=mask), tmp_path)
    attn = [n for name, n in seen if name.startswith("prefill_attn_kernel")]
    assert attn == [workgroups], seen
