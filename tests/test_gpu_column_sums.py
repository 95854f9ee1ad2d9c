"""The sums of per-workgroup partials over the workgroups, bit for bit."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("needs a HIP device")
    from delta_feedback_experiment_amd import _lib

    _lib.lib()
    return torch.device("cuda:0")


# columns H * K of each width of the kernel (8, 16 and 32 a workgroup; dA_log,
# which shares the launch, has H of them), and partials fewer than the classes,
# one round of them and a little, several rounds
@pytest.mark.parametrize("H,K", [(3, 32), (17, 128), (65, 128)])
@pytest.mark.parametrize("docs", [1, 200, 260, 1300])
def test_column_sums_order(dev, docs, H, K):
    """The gate's bias gradient over documents of one token, whose per-chunk
    partials are the gate gradient's own rows: 256 classes in turn, then the
    halving tree over the classes."""
    from delta_feedback_experiment_amd import _lib
    from delta_feedback_experiment_amd.chunk import ChunkPlan, gate_backward

    print(f"[gpu] column sums docs={docs} H={H} K={K}", flush=True)
    gen = torch.Generator(device=dev).manual_seed(docs + H)
    g, dgcum = (torch.randn(docs, H, K, generator=gen, device=dev) for _ in range(2))
    A_log, dt_bias = torch.rand(H, generator=gen, device=dev), torch.randn(H * K, generator=gen, device=dev)
    plan = ChunkPlan.make(g.reshape(1, docs, H, K), torch.arange(docs + 1, device=dev, dtype=torch.int32))
    dg, _, ddt_bias = gate_backward(plan, g, _lib.GATE_RAW_CHANNEL, A_log, dt_bias, dgcum)
    torch.cuda.synchronize()
    acc = torch.zeros(256, H * K)
    rows = dg.reshape(docs, H * K).cpu()
    for q in range(0, docs, 256):
        acc[:len(rows[q:q + 256])] += rows[q:q + 256]
    while len(acc) > 1:
        acc = acc[:len(acc) // 2] + acc[len(acc) // 2:]
    assert torch.equal(ddt_bias.reshape(-1).cpu(), acc[0])
