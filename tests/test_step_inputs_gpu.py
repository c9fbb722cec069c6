"""The two ends of a captured decode step: rows of the embedding table into
fragment layout, and the picked tokens as the next step's inputs."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _hip():
    from ollamamq_amd.ops import hip
    hip.require()
    return hip


def _inputs(hip, B):
    def i32(v):
        return torch.tensor(v, dtype=torch.int32, device="cuda")
    return hip.StepInputs(
        tok=i32([-1] * B), out=torch.full((B,), -1, device="cuda"),
        pos=i32(list(range(B))), lens=i32(list(range(1, B + 1))),
        adv=i32([b % 3 != 1 for b in range(B)]))


@pytest.mark.parametrize("B", [1, 3, 32, 45, 128, 800])
@pytest.mark.parametrize("V", [8, 320, 2048, 2056, 32000])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_greedy(B, V, dtype):
    hip = _hip()
    g = torch.Generator(device="cuda").manual_seed(B * V)
    # few distinct values: the first of equal ones wins
    logits = torch.randint(-9, 9, (B, V), generator=g,
                           device="cuda").to(dtype)
    want = logits.double().argmax(1)
    step = _inputs(hip, B)
    pos, lens = step.pos.clone(), step.lens.clone()
    for n in (1, 2):
        assert hip.pick_and_advance(logits, step)
        first = (logits == logits.max(1, keepdim=True)[0]).int().argmax(1)
        assert torch.equal(step.out, first)
        assert torch.equal(step.tok.long(), first)
        assert torch.equal(step.pos, pos + n * step.adv)
        assert torch.equal(step.lens, lens + n * step.adv)
    assert torch.equal(logits.gather(1, step.out[:, None]),
                       logits.gather(1, want[:, None]))


def test_sampled():
    """The draw belongs to the length before the step."""
    hip = _hip()
    B, V = 37, 4096
    logits = torch.randn(B, V, device="cuda").bfloat16()
    temps = torch.tensor([0.0, 0.7, 1.3] * 12 + [0.0], device="cuda")
    seeds = torch.arange(B, device="cuda") * 977
    step = _inputs(hip, B)
    for _ in range(3):
        want = hip.sample_gumbel(logits, temps, seeds, step.lens)
        assert hip.pick_and_advance(logits, step, temps, seeds)
        assert torch.equal(step.tok, want)
        assert torch.equal(step.out, want.long())


def test_rows_that_are_not_aligned():
    hip = _hip()
    step = _inputs(hip, 2)
    before = [t.clone() for t in step]
    assert not hip.pick_and_advance(
        torch.randn(2, 321, device="cuda").bfloat16(), step)
    assert not hip.pick_and_advance(
        torch.randn(2, 640, device="cuda").bfloat16()[:, ::2], step)
    assert all(torch.equal(a, b) for a, b in zip(before, step))


@pytest.mark.parametrize("M", [1, 31, 32, 33, 64])
@pytest.mark.parametrize("H", [64, 512, 4096])
def test_embedding_rows(M, H):
    hip = _hip()
    table = torch.randn(50, H, device="cuda").bfloat16()
    tokens = torch.randint(0, 50, (M,), device="cuda")
    got, sq = hip.fragify_sumsq(table, tokens=tokens)
    want, sq2 = hip.fragify_sumsq(table[tokens])
    rows = torch.zeros(-(-M // 32) * 32, dtype=torch.bool, device="cuda")
    rows[:M] = True
    live = rows.view(-1, 1, 1, 32, 1).expand(-1, H // 16, 2, 32, 8).flatten()
    assert torch.equal(got[live], want[live]) and torch.equal(sq, sq2)
    torch.testing.assert_close(sq.double(),
                               table[tokens].double().square().sum(1),
                               rtol=1e-5, atol=0)
