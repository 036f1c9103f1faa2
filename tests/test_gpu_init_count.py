"""
The selection of k-means|| candidates with its count in pinned memory: a host that watches the count uses it again as soon
as it has changed, while the kernel that writes the rows may still be to come.
"""
import numpy as np
import pytest
import torch

from heat_amd import _native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 1024, 1025, 2095105, 4194305, 5000000])  # one block .. every slot of the block counts taken
def test_count_used_again_before_the_rows_are_written(cuda, n):
    g = torch.Generator(device=cuda).manual_seed(n)
    d2 = torch.rand(n, generator=g, device=cuda)
    u = torch.rand(n, generator=g, device=cuda)
    d2[-1], u[-1] = 1.0, 0.0  # the last block holds a row
    cost = torch.ones((), dtype=torch.float32, device=cuda)
    ws = _native.Workspace(cuda)
    count = torch.zeros((), dtype=torch.int64, pin_memory=True)
    seen = count.numpy()
    rounds = [0.25, 0.5, 1.0]  # `probability` of a row at distance 1
    got = []
    for os_ in rounds:
        idx = torch.full((n,), -1, dtype=torch.int64, device=cuda)
        seen[...] = -1
        _native.sample_select(d2, u, cost, os_, idx, count, ws)
        spins = 0
        while int(seen) < 0 and spins < 50_000_000:
            spins += 1
        got.append((int(seen), idx))
    for os_, (c, idx) in zip(rounds, got):
        ref = torch.where(u <= torch.tensor(os_, device=cuda) * d2.sqrt())[0]
        rows = idx[:c]
        assert bool((idx[c:] == -1).all()) and int(rows[-1]) == n - 1
        assert bool((rows[1:] > rows[:-1]).all())
        # only rows whose draw sits on the threshold may differ
        diff = np.setxor1d(rows.cpu().numpy(), ref.cpu().numpy())
        assert all(abs(float(u[i]) - os_ * float(d2[i]) ** 0.5) <= 1e-6 for i in diff), diff


class _Interrupt(BaseException):
    pass


@pytest.mark.parametrize("at", ["selection", "draw"])
def test_an_interrupt_leaves_no_selection_behind(cuda, monkeypatch, at):
    # the count's memory goes back to its pool with the exception: nothing may still be about to write it
    import heat_amd as ht
    from oracle import heat_oracle as orc

    x = torch.rand((50000, 6), generator=torch.Generator(device=cuda).manual_seed(3), device=cuda)
    select = _native.sample_select

    class Sampler(orc.CpuSampler):
        def uniform(self, n):
            if at == "draw" and selections:
                raise _Interrupt
            return super().uniform(n)

    selections = []

    def interrupted(*args):
        torch.cuda._sleep(20_000_000)  # (some milliseconds of other work before it)
        select(*args)
        selections.append(None)
        if at == "selection":
            raise _Interrupt

    monkeypatch.setattr(_native, "sample_select", interrupted)
    km = ht.cluster.KMeans(n_clusters=12, init="probability_based")
    ws = _native.Workspace(cuda)
    with pytest.raises(_Interrupt):
        km._centroid_sampling_helper(x, x[5:6].clone(), 24.0, 6, Sampler(17, cuda), ws)
    assert selections and torch.cuda.current_stream(cuda).query()
