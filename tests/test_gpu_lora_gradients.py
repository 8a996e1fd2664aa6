"""LoRA gradients at the edges of their chunks: adapters with 1 to 513 rows (a chunk is 512 rows, staged 256 and read 32 at a
time), adapters without rows, columns that end inside a wave's 64, both rank widths.  Small whole numbers, so every
float32 sum is exact and the gradients are the reference's bit for bit."""

import pytest

from __graft_entry__ import load_package

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts", [(1,), (31, 33), (64, 0, 65), (255, 257), (512, 1), (513, 224, 225), (0,) * 62 + (97, 3)])
@pytest.mark.parametrize("k,n,rank", [(8, 264, 5), (328, 72, 32), (584, 520, 64)])
def test_edges_of_chunks(counts, k, n, rank):
    import torch

    pkg = load_package()
    n_ad, m = len(counts), sum(counts)
    print(f"[case] LoRA gradients {m}x{k}x{n} adapters={n_ad} rank={rank}", flush=True)
    g = torch.Generator(device="cuda:0").manual_seed(m + n + k)
    whole = lambda *s: torch.randint(-2, 3, s, generator=g, device="cuda:0").bfloat16()
    x, dy, a, b = whole(m, k), whole(m, n), whole(n_ad, k, rank), whole(n_ad, rank, n)
    s = torch.tensor([0.5, 2.0], device="cuda:0").repeat(n_ad)[:n_ad].contiguous()
    idx = torch.repeat_interleave(torch.arange(n_ad, device="cuda:0"), torch.tensor(counts, device="cuda:0"))
    idx = idx[torch.randperm(m, generator=g, device="cuda:0")].to(torch.int32)
    # what is not finite stays with its adapter and, in dA, with the 32 columns that are turned together
    first = int(idx[0])
    x[0, 0] = float("inf")
    codes = torch.randint(-127, 128, (k, n), generator=g, device="cuda:0", dtype=torch.int8)
    w = pkg.quantized_lora.GroupQuantizedWeight(codes, torch.full((1, n), 0.01, device="cuda:0"), k, k, 8, k)
    _, da, db = pkg.w8a8_lora.backward(x, dy, w, a, b, s, adapter_indices=idx)[:3]
    torch.cuda.synchronize()
    for ad in range(n_ad):
        rows = (idx == ad).nonzero().flatten()
        xd, dd = x[rows].double(), dy[rows].double()
        k0 = 32 if ad == first else 0
        want = xd[:, k0:].T @ (dd @ b[ad].double().T * s[ad])
        assert torch.equal(da[ad, k0:], want.float().bfloat16())
        if ad != first:
            assert torch.equal(db[ad], ((xd @ a[ad].double()).T @ dd * s[ad]).float().bfloat16())
