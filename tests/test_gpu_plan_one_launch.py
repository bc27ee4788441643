"""The permutation plan in one launch, one block per 1024 slots: ends of blocks and of the launch's range, assignments off the
16 bytes that its vector loads need, ids outside the experts (clamped), all rows to few experts.  Exact against a stable sort."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [(1, 1, 1), (3, 16, 16), (341, 3, 7), (1024, 1, 512), (1025, 1, 512), (257, 4, 64), (509, 8, 128), (2049, 5, 33), (65536, 1, 32),
         (8192, 8, 500), (65537, 1, 32)]


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("few", [False, True])
@pytest.mark.parametrize("T,K,E", CASES)
def test_plan(gpu_device, T, K, E, few, off):
    from arctictraining_amd import ops

    print("plan", T, K, E, few, off, flush=True)
    g = torch.Generator().manual_seed(T + K)
    ids = torch.randint(0, 2, (T, K), generator=g) * (E - 1) if few else torch.randint(-1, E + 1, (T, K), generator=g)
    scores = torch.rand(T, K, generator=g)
    buf = torch.zeros(T * K + off, dtype=torch.int32)
    buf[off:] = ids.flatten()
    assign = buf.to(gpu_device)[off:].view(T, K)
    ws = ops.gemm_workspace(T * K, E, gpu_device)
    counts, offsets, token_of, slot_of, row_of, perm = ops.permute_plan(assign, E, scores.to(gpu_device), gemm_workspace=ws,
                                                                        gemm_dtype=torch.bfloat16)
    flat = ids.clamp(0, E - 1).t().reshape(-1)                 # slot f = k T + t
    order = torch.sort(flat, stable=True).indices
    want = torch.bincount(flat, minlength=E)
    assert torch.equal(counts.cpu().long(), want)
    assert torch.equal(offsets.cpu().long(), torch.cat([torch.zeros(1, dtype=torch.long), want.cumsum(0)]))
    assert torch.equal(slot_of.cpu().long(), order) and torch.equal(token_of.cpu().long(), order % T)
    place = (order % T) * K + order // T
    rows = torch.empty(T * K, dtype=torch.long)
    rows[place] = torch.arange(T * K)
    assert torch.equal(row_of.cpu().long().flatten(), rows)
    assert torch.equal(perm.cpu(), scores.flatten()[place])
