"""Key-split prefill on an MI355X on either side of the merge's switch from one wave per (query, head) to four, with
splits that hold no keys, against float64: with keys of one size, and with keys that grow over the row, so that the splits'
running maxima and the weights of their partials differ by orders of magnitude."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grow", [False, True])
@pytest.mark.parametrize("T", [1, 3, 64, 65])
@pytest.mark.parametrize("splits", [1, 16, 17, 63, 65, 256])
def test_merge_waves(hip, T, splits, grow):
    """The outputs are rounded to bf16 (relative rms of 2^-8 / sqrt(3) / 1.39 = 1.6e-3 over a binade of values), and so is
    every probability: their independent roundings give at most the same 1.6e-3 of the result's 2-norm, for values of one
    size and zero mean. Together 2.3e-3; a weight that is off by a fifth moves 2e-2 and more."""
    g = torch.Generator(device="cuda").manual_seed(T)
    S = 64 * 40 + 5
    bf = lambda *s: (torch.rand(*s, generator=g, device="cuda") * 2 - 1).to(torch.bfloat16)
    q, K, V = 3 * bf(T, 16, 128), bf(S, 4, 128), bf(S, 4, 128)
    if grow:
        K = (K.float() * (0.5 + 3 * torch.arange(S, device="cuda") / S)[:, None, None]).to(torch.bfloat16)
    rows = hip.PrefillRows([0, T], [0, S], [S - T], q.device)
    print("prefill merge", T, splits, grow, flush=True)
    got = hip.prefill_rows(q, rows, K, V, None, splits=splits).double()
    late = torch.arange(S, device="cuda")[None] > torch.arange(S - T, S, device="cuda")[:, None]
    want = torch.empty_like(got)
    for h in range(16):
        x = q[:, h].double() @ K[:, h // 4].double().T.contiguous() * 128 ** -0.5
        want[:, h] = torch.softmax(x.masked_fill(late, -torch.inf), -1) @ V[:, h // 4].double()
    assert ((got - want).norm() / want.norm()).item() <= 2.6e-3
