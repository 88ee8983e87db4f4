"""GPU: qblock_schedule, the work order by windows of whole heads, against its definition on the host, entry for
entry, at the edges: fewer entries than XCDs, shares that end inside a head, one window per share (a list longer
than a third of a slot's work), shares of very different work (the sort over everything), empty lists, the longest list
behind the shares."""
import numpy as np
import pytest
import torch

from fgattn_tk_cuda_amd import capi

pytestmark = pytest.mark.gpu


def _classes(counts):
    """Eighths of an octave over the seven octaves below the longest list, shorter lists, empty lists."""
    top, out = max(1, int(counts.max())).bit_length() - 1, []
    for c in counts.tolist():
        lg = c.bit_length() - 1
        below = (c >> (lg - 3)) & 7 if lg >= 3 else (c << (3 - lg)) & 7 if c > 0 else 0
        out.append(min(((top - lg) << 3) + 7 - below, (7 << 3) + 2) if c > 0 else (7 << 3) + 3)
    return np.array(out)


def _schedule(counts, per_head):
    n, per = len(counts), len(counts) // 8
    cls = _classes(counts)
    order = np.arange(n)
    shares = [float(counts[x * per:(x + 1) * per].sum()) for x in range(8)]
    if max(shares) * 8 > 1.1 * sum(shares):
        return np.argsort(cls, kind="stable")
    for x in range(8):
        a, end, seq = x * per, (x + 1) * per, []
        one = int(counts[:per * 8].max(initial=0)) * 64 > 0.3 * shares[x]
        while a < end:
            b = end
            if not one:
                b = (a // per_head + 1) * per_head
                while b - a < 192:
                    b += per_head
                b = min(b, end)
            seq.append(a + np.argsort(cls[a:b], kind="stable"))
            a = b
        if seq:
            order[np.arange(per) * 8 + x] = np.concatenate(seq)
    return order


@pytest.mark.parametrize("n,per_head,kind", [(5, 5, "even"), (8, 3, "even"), (3072, 256, "near"), (3072, 256, "zipf"), (10240, 256, "near"),
                                              (4728, 591, "near"), (2000, 64, "near"), (4096, 512, "skewed"), (70007, 9001, "near"), (1000, 7, "zeros"),
                                              (1003, 59, "last"), (1007, 53, "skewed_last")])
def test_schedule_equals_its_definition(dev, n, per_head, kind):
    print("case schedule", n, per_head, kind, flush=True)
    rng = np.random.default_rng(n)
    counts = {"even": np.full(n, 26), "near": rng.integers(1700, 3600, size=n), "zipf": np.minimum(rng.zipf(1.2, size=n), 1024),
              "skewed": np.where(np.arange(n) < n // 8, 5000, 300) + rng.integers(0, 200, size=n), "zeros": rng.integers(0, 2, size=n) * 9,
              "last": np.where(np.arange(n) == n - 1, 60000, 300),
              "skewed_last": np.where(np.arange(n) == n - 1, 60000, np.where(np.arange(n) < n // 8, 5000, 300))}[kind]
    counts = counts.astype(np.int32)
    c = torch.from_numpy(counts).to(dev)
    order = torch.full((n,), -1, dtype=torch.int32, device=dev)
    capi.qblock_schedule(order, c, per_head)
    got = order.cpu().numpy()
    assert np.array_equal(np.sort(got), np.arange(n))
    assert np.array_equal(got, _schedule(counts, per_head))


@pytest.mark.parametrize("n,per_head,densest", [(520, 65, 1.6), (3072, 256, 1.9), (23640, 591, 1.4), (3001, 250, 3.0), (8191, 256, 6.0),
                                                (8192, 256, 2.5), (23640, 591, 4.0), (23643, 591, 300.0)])
def test_schedule_of_heads_of_different_density(dev, n, per_head, densest):
    """Heads of rising density, so that the XCDs' shares differ: sorted over everything by all four waves, from 8192
    q-blocks on in quarters of an octave."""
    print("case schedule of uneven heads", n, per_head, densest, flush=True)
    rng = np.random.default_rng(n)
    head = np.arange(n) // per_head
    counts = (500 * (1 + (densest - 1) * head / head.max()) * rng.uniform(1.0, 1.02, size=n)).astype(np.int32)
    shares = [int(counts[x * (n // 8):(x + 1) * (n // 8)].sum()) for x in range(8)]
    assert max(shares) * 8 > 1.1 * sum(shares)
    cls = _classes(counts)
    if n >= 8192:
        cls = np.where(cls < (7 << 3) + 2, cls >> 1, cls)
    want = np.argsort(cls, kind="stable")
    c = torch.from_numpy(counts).to(dev)
    order = torch.full((n,), -1, dtype=torch.int32, device=dev)
    capi.qblock_schedule(order, c, per_head)
    assert np.array_equal(order.cpu().numpy(), want)
