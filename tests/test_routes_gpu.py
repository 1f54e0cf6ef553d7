"""Which kernel a call launches, where a rule on sizes chooses between forms: the
launches of one call as torch's profiler records them."""
import json

import pytest
import torch
from torch.profiler import ProfilerActivity, profile

from helm_amd import kernels as hk

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
