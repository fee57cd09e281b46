"""The matrix memory by chunks of 64 tokens against 64-bit arithmetic token by token: runs that end at, before and behind a
chunk's edge, go on from a state, and stand beside runs of one token."""
import pytest
import torch

from test_sunatar_gpu import _ctx

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
F64 = torch.float64


def _walk(x, heads, n, v, cap, eps, weight, state):
    """A run's outputs and the state it leaves, token by token; `state`: memory [H, n, v], normalizer [H, n], peak [H]."""
    mem, nrm, peak = state
    hn, hv = heads * n, heads * v
    out = []
    for row in x:
        q, k = row[:hn].view(heads, n) * n ** -0.5, row[hn:2 * hn].view(heads, n)
        val, gate = row[2 * hn:2 * hn + hv].view(heads, v), row[2 * hn + hv:2 * hn + 2 * hv]
        gi = cap * torch.tanh(row[-2 * heads:-heads] / cap)
        gf = torch.nn.functional.logsigmoid(cap * torch.tanh(row[-heads:] / cap))
        new = torch.maximum(gf + peak, gi)
        keep, take = torch.exp(gf + peak - new), torch.exp(gi - new)
        mem = keep[:, None, None] * mem + take[:, None, None] * k[:, :, None] * val[:, None, :]
        nrm, peak = keep[:, None] * nrm + take[:, None] * k, new
        o = (mem * q[:, :, None]).sum(1) / (torch.maximum((nrm * q).sum(-1).abs(), torch.exp(-peak)) + 1e-6)[:, None]
        o = o * torch.rsqrt((o * o).mean(-1, keepdim=True) + eps)
        out.append(o.reshape(-1) * weight * torch.sigmoid(gate))
    return torch.stack(out), (mem, nrm, peak)


@pytest.mark.parametrize("sizes", [(3, 64, 128), (2, 10, 7), (1, 128, 40), (2, 100, 24), (2, 66, 16), (4, 16, 16)])
@pytest.mark.parametrize("steps", [[[64], [1]], [[65, 1], [63, 130]], [[24, 1, 200], [127, 128, 1]], [[700], [64]]])
@pytest.mark.parametrize("gates,line", [(1.0, 1), (6.0, 24)])
def test_memory_by_chunks(sizes, steps, gates, line):
    from transformers_neuronx_amd.kernels import make_ops
    heads, n, v = sizes
    ops = make_ops("hip", torch.float32, DEV)
    ops.memory_chunk_run = ops.memory_chunk_run_beside = line
    g = torch.Generator().manual_seed(n + v + sum(steps[0]))
    cap, eps = 9.0, 1e-5
    total = 2 * heads * n + 2 * heads * v + 2 * heads
    weight = torch.rand(heads * v, generator=g) + 0.5
    rows = [len(s) for s in steps]
    slots = [2, 0, 3][:max(rows)]
    state = [torch.full((5, 2, heads, v, n), 3.0, device=DEV), torch.full((5, 2, heads, n), -2.0, device=DEV),
             torch.full((5, 2, heads), 5.0, device=DEV)]
    plain = [(torch.zeros(heads, n, v, dtype=F64), torch.zeros(heads, n, dtype=F64), torch.zeros(heads, dtype=F64))
             for _ in slots]
    have = [0] * len(slots)
    for lens in steps:
        proj = torch.randn(sum(lens), total, generator=g)
        proj[:, -2 * heads:] *= gates
        ctx = _ctx(lens, have[:len(lens)], slots[:len(lens)])
        got = ops.matrix_memory(proj.to(DEV), heads, n, v, cap, eps, weight.to(DEV), ctx, *state).double().cpu()
        at = 0
        for r, count in enumerate(lens):
            want, plain[r] = _walk(proj[at:at + count].double(), heads, n, v, cap, eps, weight.double(), plain[r])
            # a token's sums go over up to 700 tokens and 128 elements, each product rounded a few times: the roundings of
            # 2^-24 add up to 2e-5 of the result only where all of them point one way
            assert float((got[at:at + count] - want).norm() / want.norm()) < 2e-5
            have[r], at = have[r] + count, at + count
            place = (have[r] - 1) & 1
            scale = torch.exp(state[2][slots[r], place].double().cpu() - plain[r][2])[:, None]
            mem = state[0][slots[r], place].double().cpu().transpose(1, 2) * scale[:, :, None]
            nrm = state[1][slots[r], place].double().cpu() * scale
            assert float((mem - plain[r][0]).norm() / plain[r][0].norm()) < 2e-5
            assert float((nrm - plain[r][1]).norm() / plain[r][1].norm()) < 2e-5
    assert float(state[0][1].min()) == 3.0 and float(state[0][4].min()) == 3.0       # slots of no one are not touched


@pytest.mark.parametrize("column", ["query", "key", "value", "input gate", "forget gate"])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("at", [70, 129])
def test_a_token_that_is_no_number_leaves_the_ones_before_it(column, bad, at):
    """One projection of token 70 or of the last one of 130 is no number: the tokens before it are what they are without it, to
    the bit, and the head's tokens from it on (of a query: the token alone) are no numbers. A gate's cap makes a number of an
    infinite one. Token by token the same elements are no numbers, and the same of the state are none or infinite."""
    from transformers_neuronx_amd.kernels import make_ops
    heads, n, v = 2, 64, 32
    hn, hv = heads * n, heads * v
    ops = make_ops("hip", torch.float32, DEV)
    g = torch.Generator().manual_seed(8)
    proj = torch.randn(130, 2 * hn + 2 * hv + 2 * heads, generator=g)
    weight = torch.rand(hv, generator=g) + 0.5
    made, states = [], []
    for spoil, by_chunks in ((False, True), (True, True), (True, False)):
        ops.memory_chunk_run = ops.memory_chunk_run_beside = 1 if by_chunks else 131
        x = proj.clone()
        if spoil:
            x[at, {"query": n, "key": hn + n, "value": 2 * hn + v, "input gate": -heads + -heads + 1, "forget gate": -1}[column]] = bad
        state = [torch.zeros(1, 2, heads, v, n, device=DEV), torch.zeros(1, 2, heads, n, device=DEV), torch.zeros(1, 2, heads, device=DEV)]
        made.append(ops.matrix_memory(x.to(DEV), heads, n, v, 9.0, 1e-5, weight.to(DEV), _ctx([130], [0], [0]), *state).cpu())
        states.append([x[:, 1].cpu() for x in state])
    clean, spoilt, walked = made
    assert torch.equal(torch.isnan(spoilt), torch.isnan(walked))
    for mine, theirs in zip(states[1], states[2]):
        assert torch.equal(torch.isnan(mine), torch.isnan(theirs)) and torch.equal(torch.isposinf(mine), torch.isposinf(theirs))
        assert torch.equal(torch.isneginf(mine), torch.isneginf(theirs))
    assert torch.isfinite(clean).all()
    assert torch.equal(clean[:at], spoilt[:at]) and torch.equal(clean[:, :v], spoilt[:, :v])      # (the head before: untouched)
    if not ("gate" in column and bad == float("inf")):
        last = at + 1 if column == "query" else 130
        assert torch.isnan(spoilt[at:last, v:]).any(dim=1).all()
        assert torch.equal(clean[last:, v:], spoilt[last:, v:])
