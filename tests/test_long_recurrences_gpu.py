"""The recurrences over long portions of a prompt (`ops.ssm_scan`, `ops.memory_scan`: 16 tokens at a time on the matrix
cores) against the same kernels' walk token by token, which a prompt cut into portions of fewer than 64 tokens takes."""
import pytest
import torch

from wllm_amd.kernels import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
SHORT = 40                  # a portion of so many tokens is walked token by token


@pytest.fixture(autouse=True)
def _chunks_from_64_tokens(monkeypatch):
    """Whatever the sizes: where the chunks pay is not what is tested."""
    monkeypatch.setattr(ops, "ssm_chunk_from", lambda heads, groups: 64)
    monkeypatch.setattr(ops, "memory_chunk_from", lambda heads, value_dim, row_decays: 64)


def _ints(values):
    return torch.tensor(values, dtype=torch.int32, device=DEV)


class StateSpace:
    """Random operands of `ops.ssm_scan` for a sequence, and the recurrence over it in portions."""
    parts = ("x", "B", "C", "dt")

    def __init__(self, dtype, tokens, heads=4, groups=2, n_state=24, p=20, seed=1):
        g = torch.Generator().manual_seed(seed)
        self.heads, self.groups, self.n_state, self.p, self.tokens = heads, groups, n_state, p, tokens
        self.inner = heads * p
        self.xbc = (torch.randn(tokens, self.inner + 2 * groups * n_state, generator=g) * 0.7).to(dtype).to(DEV)
        self.dt = torch.randn(tokens, heads, generator=g).to(dtype).to(DEV)
        self.vectors = [(m + torch.randn(heads, generator=g)).to(DEV) for m in (-1.0, -0.5, 1.0)]
        self.state0 = torch.randn(3, heads * n_state * p + 4, generator=g).to(DEV)

    def put(self, part, token, value):
        at = {"x": 7, "B": self.inner + 5, "C": self.inner + self.groups * self.n_state + 5}
        if part == "dt":
            self.dt[token, 1] = value
        else:
            self.xbc[token, at[part]] = value

    def launch(self, rows, q_start, q_len, slots, state, y):
        ops.ssm_scan(self.xbc[rows].contiguous(), self.dt[rows].contiguous(), *self.vectors, state, _ints(q_start), _ints(q_len),
                     _ints(slots), y, heads=self.heads, groups=self.groups, state_size=self.n_state, head_dim=self.p)

    def run(self, cuts):
        state, out, at = self.state0.clone(), [], 0
        for n in cuts:
            y = torch.full((n, self.inner), 7.0, device=DEV)
            self.launch(slice(at, at + n), [0], [n], [1], state, y)
            out.append(y)
            at += n
        return torch.cat(out), state

    def exact(self):
        """Results and the state left behind in 64 bits."""
        h, g, n, p = self.heads, self.groups, self.n_state, self.p
        bias, a_log, skip = (v.double() for v in self.vectors)
        x = self.xbc.double()
        state, out = self.state0[1, :h * n * p].double().view(h, n, p), []
        for t in range(self.tokens):
            step = torch.nn.functional.softplus(self.dt[t].double() + bias)
            b, c = (x[t, self.inner + i * g * n:self.inner + (i + 1) * g * n].view(g, n).repeat_interleave(h // g, 0) for i in (0, 1))
            v = x[t, :self.inner].view(h, p)
            state = torch.exp(-torch.exp(a_log) * step)[:, None, None] * state + (step[:, None] * b)[:, :, None] * v[:, None]
            out.append(((state * c[:, :, None]).sum(1) + skip[:, None] * v).reshape(-1))
        return torch.stack(out), state


class Memory:
    """The same of `ops.memory_scan`, for each kind of decay (`own`: steps of its own, with the normaliser)."""
    parts = ("q", "k", "v", "decay")

    def __init__(self, dtype, tokens, kind, heads=3, d=24, dv=20, seed=2):
        g = torch.Generator().manual_seed(seed)
        self.kind, self.heads, self.d, self.dv, self.tokens = kind, heads, d, dv, tokens
        self.memory = heads * d * dv
        self.qk = torch.randn(3 if kind == "rows" else 2, tokens, heads * d, generator=g).to(DEV) * d ** -0.5
        if kind == "rows":
            self.qk[2] = torch.rand(tokens, heads * d, generator=g).to(DEV)
        self.v = torch.randn(tokens, heads * dv, generator=g).to(dtype).to(DEV)
        self.decays = (1.0 - torch.logspace(0, -4, heads)).to(DEV)
        self.steps = torch.rand(3, tokens, heads, generator=g).to(DEV)
        self.state0 = torch.randn(3, self.memory + heads * d, generator=g).to(DEV)

    def put(self, part, token, value):
        if part == "v":
            self.v[token, 7] = value
        elif part != "decay":
            self.qk[0 if part == "q" else 1, token, 9] = value
        elif self.kind == "rows":
            self.qk[2, token, 9] = value
        elif self.kind == "own":
            self.steps[0, token, 1] = value

    def launch(self, rows, q_start, q_len, slots, state, y):
        own, n = self.kind == "own", y.shape[0]
        width = self.heads * self.dv
        out, nq = torch.full((n, width), 7.0, device=DEV), torch.full((n, self.heads), 7.0, device=DEV)
        ops.memory_scan(self.qk[:, rows].contiguous(), self.v[rows].contiguous(), self.steps[:, rows].contiguous() if own else None,
                        self.decays if self.kind == "head" else None, state, _ints(q_start), _ints(q_len), _ints(slots), out,
                        heads=self.heads, head_dim=self.d, value_dim=self.dv, nq=nq if own else None,
                        n_offset=self.memory if own else 0, row_decays=self.kind == "rows")
        y.copy_(torch.cat([out, nq], dim=1))

    def run(self, cuts):
        state, out, at = self.state0.clone(), [], 0
        for n in cuts:
            y = torch.zeros(n, self.heads * self.dv + self.heads, device=DEV)
            self.launch(slice(at, at + n), [0], [n], [1], state, y)
            out.append(y)
            at += n
        return torch.cat(out), state

    def exact(self):
        """Results and the memory left behind in 64 bits."""
        h, d, dv = self.heads, self.d, self.dv
        state, out = self.state0[1, :self.memory].double().view(h, d, dv), []
        for t in range(self.tokens):
            q, k, v = self.qk[0, t].double().view(h, d), self.qk[1, t].double().view(h, d), self.v[t].double().view(h, dv)
            if self.kind == "rows":
                f = self.qk[2, t].double().view(h, d)
            else:
                f = (self.steps[0, t] if self.kind == "own" else self.decays).double()[:, None].expand(h, d)
            if self.kind == "own":
                k = k * self.steps[1, t].double()[:, None]
            state = f[:, :, None] * state + k[:, :, None] * v[:, None]
            out.append((state * q[:, :, None]).sum(1).reshape(-1))
        return torch.stack(out), state


KINDS = ["space", "head", "rows", "own"]


def _problem(kind, dtype, tokens, **sizes):
    return StateSpace(dtype, tokens, **sizes) if kind == "space" else Memory(dtype, tokens, kind, **sizes)


def _portions(tokens, most=SHORT):
    return [most] * (tokens // most) + ([tokens % most] if tokens % most else [])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kind", KINDS)
def test_a_value_that_is_not_finite_leaves_the_tokens_before_it_alone(dtype, kind):
    """An infinity or NaN in any operand of a token, at either end of a chunk of 16, inside one and in a prompt's last
    tokens: what comes before has the bits it has without it, and from there on it reaches what the walk token by token
    says it reaches, in the results and in the state left behind."""
    tokens = 101
    clean = _problem(kind, dtype, tokens).run([tokens])[0]
    parts = StateSpace.parts if kind == "space" else Memory.parts[:3] if kind == "head" else Memory.parts
    for part in parts:
        for at in (0, 15, 32, 40, 95, 99):
            for value in (float("inf"), float("-inf"), float("nan")):
                if part in ("dt", "decay") and value == float("-inf"):
                    continue                                  # (a step size of zero; decays are not negative)
                hit = _problem(kind, dtype, tokens)
                hit.put(part, at, value)
                (y, state), (ref, ref_state) = hit.run([tokens]), hit.run(_portions(tokens))
                case = f"{part} of token {at}: {value}"
                assert torch.equal(y[:at], clean[:at]), f"{case}: a token before it changed"
                assert torch.equal(torch.isfinite(y), torch.isfinite(ref)), f"{case}: results"
                assert not bool(torch.isfinite(y[at]).all()), case
                assert torch.equal(torch.isfinite(state), torch.isfinite(ref_state)), f"{case}: the state"


def test_a_key_that_overflows_is_infinite_and_not_nan():
    """A key of 3e38 that its step takes out of float32: infinite in the memory, as the walk token by token leaves it."""
    tokens = 96
    hit = _problem("own", torch.bfloat16, tokens)
    for t in (hit.qk, hit.v, hit.state0):
        t.abs_()
    hit.steps[0].clamp_(min=0.5)
    hit.qk[1, 94, 9], hit.steps[1, 94] = 3e38, 40.0            # (one of the last four tokens of a chunk)
    (y, state), (ref, ref_state) = hit.run([tokens]), hit.run(_portions(tokens))
    assert not bool(torch.isnan(ref).any() or torch.isnan(ref_state).any()) and bool(torch.isinf(ref_state).any())
    assert not bool(torch.isnan(y).any() or torch.isnan(state).any())
    assert torch.equal(torch.isinf(state), torch.isinf(ref_state))


@pytest.mark.parametrize("kind", KINDS)
def test_float32_has_the_same_bits_however_a_prompt_is_cut(kind):
    """In the true 32-bit path a token's results do not depend on the portion it came in."""
    tokens = 150
    problem = _problem(kind, torch.float32, tokens)
    whole, state = problem.run([tokens])
    for cuts in ([64, 1, 85], _portions(tokens), [1] * tokens):
        y, left = problem.run(cuts)
        assert torch.equal(y, whole) and torch.equal(left, state), f"{cuts[:3]}"


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("length", [0, 1, 15, 40, 63, 64, 70])
def test_one_segment_of_fewer_tokens_than_rows(kind, length):
    """A step's only segment holds fewer tokens than the operands have rows: its tokens are walked, whether there are
    enough for chunks or not, and the rows behind them are left alone."""
    problem = _problem(kind, torch.bfloat16, 80)
    state = problem.state0.clone()
    width = problem.inner if kind == "space" else problem.heads * (problem.dv + 1)
    y = torch.full((80, width), 7.0, device=DEV)
    problem.launch(slice(0, 80), [0], [length], [1], state, y)
    assert bool((y[length:] == 7.0).all())
    if length:
        want, left = problem.run(_portions(length))
        scale = float(want.abs().max())
        # float32 sums of some hundred products in two orders: some 2^-24 each, of the largest
        assert float((y[:length] - want).abs().max()) <= 2e-6 * scale
        assert float((state - left).abs().max()) <= 2e-6 * float(left.abs().max())
    else:
        assert torch.equal(state, problem.state0)


@pytest.mark.parametrize("kind", KINDS)
def test_segments_in_any_order_of_their_rows(kind):
    """The segments of a step need not come in the order of their rows: each has the bits that it has in that order, with
    short ones and rows of no segment between them."""
    places = [(0, 100), (100, 64), (167, 3), (170, 70), (245, 97), (342, 1)]           # (first row, tokens), rows left out
    problem = _problem(kind, torch.bfloat16, 350)
    width = problem.inner if kind == "space" else problem.heads * (problem.dv + 1)
    problem.state0 = problem.state0.repeat(2, 1)

    def run(order):
        state, y = problem.state0.clone(), torch.full((350, width), 7.0, device=DEV)
        problem.launch(slice(0, 350), [places[i][0] for i in order], [places[i][1] for i in order], list(order), state, y)
        return y, state
    want, left = run(range(6))
    for order in ((5, 4, 3, 2, 1, 0), (1, 0, 4, 5, 3, 2), (3, 1, 2, 0, 5, 4)):
        y, state = run(order)
        assert torch.equal(y, want) and torch.equal(state, left), f"{order}"
    assert bool((want[164:167] == 7.0).all()) and bool((want[240:245] == 7.0).all())
    for i, (at, n) in enumerate(places):
        alone = problem.state0.clone()
        y = torch.full((n, width), 7.0, device=DEV)
        problem.launch(slice(at, at + n), [0], [n], [i], alone, y)
        assert torch.equal(y, want[at:at + n]) and torch.equal(alone[i], left[i]), f"segment {i}"


@pytest.mark.parametrize("kind", ["space", "head"])
def test_more_heads_than_a_grid_has_rows_are_walked_token_by_token(kind):
    """Beyond 65,535 heads (groups) a long segment is not walked in chunks; it has the bits that its portions have."""
    heads = 65537
    sizes = dict(heads=heads, groups=heads, n_state=1, p=1) if kind == "space" else dict(heads=heads, d=1, dv=1)
    problem = _problem(kind, torch.bfloat16, 70, **sizes)
    (y, state), (want, left) = problem.run([70]), problem.run(_portions(70))
    assert torch.equal(y, want) and torch.equal(state, left)


@pytest.mark.parametrize("kind", ["rows", "own"])
def test_what_the_newest_keys_lose_in_rounding_is_carried_along(kind):
    """Of a chunk's last four keys, which weigh most, the memory takes what 32 bits lose of the decayed key too: a value of 3
    at one of these tokens alone, from an empty memory, leaves the nearest float32 number (half a unit, 2^-24; of the
    rounded key it would be up to two units)."""
    for token in range(60, 64):
        problem = _problem(kind, torch.bfloat16, 64, d=72)
        problem.state0.zero_()
        problem.v.zero_()
        problem.v[token] = 3.0
        if kind == "own":
            problem.steps[0] = 0.5 + 0.5 * problem.steps[0]
        else:
            problem.qk[2] = 0.5 + 0.5 * problem.qk[2]
        _, state = problem.run([64])
        key = problem.qk[1, token].double().view(problem.heads, problem.d)
        for t in range(token + 1, 64):
            key = key * (problem.steps[0, t].double()[:, None] if kind == "own" else problem.qk[2, t].double().view(problem.heads, problem.d))
        if kind == "own":
            key = key * problem.steps[1, token].double()[:, None]
        want = 3.0 * key[:, :, None].expand(-1, -1, problem.dv)
        got = state[1, :problem.memory].double().view(problem.heads, problem.d, problem.dv)
        assert float(((got - want) / want).abs().max()) <= 2.0 ** -24 * 1.001, f"token {token}"


@pytest.mark.parametrize("kind", KINDS)
def test_chunks_are_as_near_the_result_in_64_bits_as_the_walk(kind):
    """The relative error (2-norm) of results and state over 320 tokens, in chunks against token by token: no larger, up to
    a tenth for what a draw of the inputs does to both."""
    tokens = 320
    sizes = dict(heads=8, groups=2, n_state=128, p=32) if kind == "space" else dict(heads=4, d=128, dv=32)
    problem = _problem(kind, torch.bfloat16, tokens, **sizes)
    if kind != "space":
        problem.decays = (1.0 - torch.logspace(-1, -3, problem.heads)).to(DEV)
    outputs, states = zip(problem.run([tokens]), problem.run(_portions(tokens)))
    want, left = problem.exact()
    size = left.numel()
    for what, (chunks, walk), exact in (("results", outputs, want), ("state", [s[1, :size] for s in states], left.reshape(-1))):
        chunks, walk = (float((t.double()[..., :exact.shape[-1]] - exact).norm() / exact.norm()) for t in (chunks, walk))
        print(kind, what, chunks, walk)
        assert chunks <= 1.1 * walk, f"{what}: {chunks:.2e} in chunks, {walk:.2e} token by token"
