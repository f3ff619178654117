"""Row geometry of prefill calls on the host: what the key assembly's launches would read or write out of range is
refused before any launch, as the gathers refused it."""
from ctypes import c_void_p

import pytest
import torch

CPU = torch.device("cpu")


@pytest.mark.parametrize("qsl,ksl", [([0, 5, 3], [0, 5, 8]), ([0, 3, 5], [0, 8, 5]), ([1, 3, 5], [0, 3, 5]),
                                     ([0, 3, 5], [2, 5, 7]), ([0, 3], [0, 3, 5])])
def test_starts_that_are_no_prefix_sums(qsl, ksl):
    from lfm3_kv800_amd import kv800_hip
    with pytest.raises(ValueError):
        kv800_hip.PrefillRows(qsl, ksl, [0, 0], CPU)


@pytest.mark.parametrize("call", ["prefill_quant_rows", "prefill_window_rows"])
@pytest.mark.parametrize("qsl,prev", [([0, 5, 3], [2, 0]), ([0, 3, 5], [4, -1])])
def test_calls_refuse_bad_rows(call, qsl, prev):
    from lfm3_kv800_amd import vllm_cache
    import lfm3_kv800_amd.kv800 as kv
    x = torch.zeros(5, 4, 128, dtype=torch.bfloat16)
    t = torch.zeros(8, 32, dtype=torch.bfloat16)
    with pytest.raises(ValueError):
        getattr(vllm_cache, call)(kv.Paged(), x.repeat(1, 4, 1), x, x, qsl, prev, t, t)


def test_counts_match_the_rows():
    from lfm3_kv800_amd import kv800_hip
    prev = [0, 255, 256, 300]
    assert kv800_hip.window_counts(prev, 256, 4) == [0, 255, 256, 259]
    assert kv800_hip.window_counts(prev, 256, 0) == [0, 255, 255, 255]
    rows = kv800_hip.PrefillRows([0, 2, 2, 5, 6], [0, 2, 257, 516, 776], prev, CPU)
    rows.need_counts(kv800_hip.window_counts(prev, 256, 4))
    with pytest.raises(ValueError):
        rows.need_counts(kv800_hip.window_counts(prev, 256, 0))


class Calls:
    """A library whose entry points only note that they were called."""
    def __init__(self):
        self.made = []

    def __getattr__(self, name):
        return lambda *a: self.made.append(name) or 0


@pytest.mark.parametrize("call", ["prefill_quant_rows", "prefill_window_rows"])
def test_calls_refuse_queries_of_another_device(monkeypatch, call):
    """The row geometry is made on the queries' device and the assembly reads it on the cache's."""
    from lfm3_kv800_amd import kv800_hip, vllm_cache
    import lfm3_kv800_amd.kv800 as kv
    lib = Calls()
    monkeypatch.setattr(kv800_hip, "ops", lambda: lib)
    monkeypatch.setattr(kv800_hip, "_stream", lambda dev: c_void_p(0))
    bf = dict(dtype=torch.bfloat16)
    P = kv.Paged(epool=torch.zeros(1, 4, 64, 256, **bf), eoff=torch.zeros(1, 1, dtype=torch.int64), ebs=64, e_hs=64 * 256,
                 e_ts=256, e_v=128, NQ=torch.zeros(1, dtype=torch.int32))
    x, t = torch.zeros(5, 4, 128, **bf), torch.zeros(16, 32, **bf)
    with pytest.raises(ValueError):
        getattr(vllm_cache, call)(P, torch.empty(5, 16, 128, device="meta", **bf), x, x, [0, 5], [7], t, t)
    assert lib.made == []
    getattr(vllm_cache, call)(P, x.repeat(1, 4, 1), x, x, [0, 5], [7], t, t)
    assert len(lib.made) == 2   # the assembly and the attention


def test_one_upload_per_stream():
    from lfm3_kv800_amd import kv800_hip
    rows = kv800_hip.PrefillRows([0, 5], [0, 12], [7], CPU)
    at = lambda stream: [p.value for p in rows.ptrs(c_void_p(stream))]
    first, second = at(0), at(64)
    assert set(first).isdisjoint(second) and at(64) == second and at(0) == first
