"""Key-split prefill on an MI355X on either side of the merge's switch from one wave per (query, head) to four, with
splits that hold no keys, against the unsplit launch: both round fp32 sums to bf16 once, so outputs of size up to 1
differ by at most one rounding step (2^-8) of values that the reassociated sum moves across a tie."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 3, 64, 65])
@pytest.mark.parametrize("splits", [16, 17, 63, 65, 256])
def test_merge_waves(hip, T, splits):
    g = torch.Generator(device="cuda").manual_seed(T)
    S = 64 * 40 + 5
    bf = lambda *s: (torch.rand(*s, generator=g, device="cuda") * 2 - 1).to(torch.bfloat16)
    q, K, V = 3 * bf(T, 16, 128), bf(S, 4, 128), bf(S, 4, 128)
    rows = hip.PrefillRows([0, T], [0, S], [S - T], q.device)
    print("prefill merge", T, splits, flush=True)
    want = hip.prefill_rows(q, rows, K, V, None, splits=1).float()
    got = hip.prefill_rows(q, rows, K, V, None, splits=splits).float()
    assert torch.isfinite(got).all() and (got - want).abs().max() <= 2 ** -8
    assert want.abs().max() > 0.05
