"""The chunked kernels of the recurrent mixers (64 rows of a prompt at a time) and those over segments (32 rows at a time, prompts cut
into pieces that run side by side) against the recurrences run row by row in 64 bits, and their error beside that of the row by row
kernels.  Both form products of 32-bit values; the delta rule's walk and all of the segments' on 16-bit matrix instructions, the
operands in three pieces."""
import pytest
import torch
import torch.nn.functional as F

from vllm_distributed_amd.ops import hip

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module", autouse=True)
def _lib():
    hip.load()


def _case(op, heads, groups, dim, vdim, new, lens, dtype, seed, strong=False, pad=0):
    """Packed rows of ``new[i]`` rows per sequence; ``strong``: decays down to 1e-30 beside ones next to 1; ``pad``: columns
    behind the projection (row strides that no vector load divides)."""
    g = torch.Generator(DEV).manual_seed(seed)

    def normal(*shape, std=1.0):
        return torch.randn(*shape, generator=g, device=DEV) * std
    t = sum(new)
    cols = heads * vdim + 2 * groups * dim
    c = {"op": op, "heads": heads, "groups": groups, "dim": dim, "vdim": vdim, "new": new, "lens": lens}
    c["x"] = normal(t, cols + pad).to(dtype)[:, :cols]
    c["state"] = normal(len(new) + 2, heads, dim, vdim, std=0.3)
    c["slots"] = torch.randperm(len(new) + 2, generator=g, device=DEV)[:len(new)].to(torch.int32)
    channels = heads * dim if op == "delta_channel" else heads
    c["beta"] = normal(t, heads + pad).to(dtype)[:, :heads]
    c["dt"] = normal(t, channels + pad, std=4.0 if strong else 0.5).to(dtype)[:, :channels]
    c["dt_bias"] = normal(channels) - (0.0 if strong else 3.0)
    c["a_log"] = normal(heads, std=0.5) + (1.5 if strong else 0.5)
    c["skip"] = normal(heads)
    if op == "linear_channel":
        z = normal(t, heads * dim, std=3.0)
        c["decay"] = torch.sigmoid(z) ** 8 if strong else torch.sigmoid(z + 2.0) ** (1.0 / 16.0)
    else:
        c["decay"] = torch.rand(heads, generator=g, device=DEV) * (0.9 if not strong else 1e-9) + (0.1 if not strong else 0.0)
    return c


def _run(c, chunked):
    state = c["state"].clone()
    qsl = torch.tensor([0] + c["new"]).cumsum(0).to(torch.int32).to(DEV)
    at = (state, c["slots"], qsl, torch.tensor(c["lens"], dtype=torch.int32, device=DEV))
    sizes = (c["heads"], c["groups"], c["dim"], c["vdim"])
    most, op = max(c["new"]), c["op"]
    if op.startswith("delta"):
        out = hip.gated_delta_rule(c["x"], *sizes, c["beta"], c["dt"], c["dt_bias"], c["a_log"], *at, 1e-6, most, 0, chunked)
    elif op == "state_space":
        out = hip.selective_scan(c["x"], c["dt"], c["heads"], c["groups"], c["vdim"], c["dim"], c["a_log"], c["dt_bias"],
                                 c["skip"], *at, most, chunked)
    else:
        out = hip.decay_linear_attention(c["x"], c["heads"], c["dim"], c["vdim"], c["decay"], *at, op == "linear_head", most,
                                         0.25 if op == "linear_channel" else 1.0, chunked)
    return out, state


def _segments(monkeypatch, rows):
    """Calls that choose by size (``chunked`` None) go over segments of ``rows`` rows (0: whole sequences), or fail."""
    def refuse(*args):
        raise AssertionError("the call did not go over segments")
    monkeypatch.setattr(hip, "segment_rows", lambda *sizes: rows)
    monkeypatch.setattr(hip, "_chunked", refuse)
    monkeypatch.setattr(hip, "_chunk_scan", refuse)


def _rows64(c):
    h, gr, d, vd, op = c["heads"], c["groups"], c["dim"], c["vdim"], c["op"]
    xd = c["x"].double()
    t = xd.shape[0]
    if op == "state_space":
        v, k, q = xd.split([h * vd, gr * d, gr * d], -1)
    else:
        q, k, v = xd.split([gr * d, gr * d, h * vd], -1)
    q, k, v = q.reshape(t, gr, d), k.reshape(t, gr, d), v.reshape(t, h, vd)
    if op.startswith("delta"):
        q = q * torch.rsqrt(q.pow(2).sum(-1, keepdim=True) + 1e-6) * d ** -0.5
        k = k * torch.rsqrt(k.pow(2).sum(-1, keepdim=True) + 1e-6)
    if op == "linear_head":
        q, k, v = F.silu(q), F.silu(k), F.silu(v)
    skip = 0.0
    if op.startswith("delta") or op == "state_space":
        step = F.softplus(c["dt"].double() + c["dt_bias"].double(), threshold=60.0).reshape(t, h, -1)
        decay = torch.exp(-torch.exp(c["a_log"].double()).view(1, h, 1) * step)
        if op == "state_space":
            skip, v = c["skip"].double().view(1, h, 1) * v, v * step
    elif op == "linear_channel":
        decay = c["decay"].double().view(t, h, d)
    else:
        decay = c["decay"].double().view(1, h, 1).expand(t, h, 1)
    q, k = q.repeat_interleave(h // gr, 1), k.repeat_interleave(h // gr, 1)
    beta = torch.sigmoid(c["beta"].double())
    out = torch.zeros(t, h, vd, dtype=torch.float64, device=DEV)
    state = c["state"].double()
    at = 0
    for i, (n, ln) in enumerate(zip(c["new"], c["lens"])):
        if n == 0:
            continue
        s = state[c["slots"][i].long()] * (0.0 if ln == n else 1.0)
        for r in range(at, at + n):
            s = s * decay[r].unsqueeze(-1)
            u = v[r].unsqueeze(1)
            if op.startswith("delta"):
                u = beta[r].view(h, 1, 1) * (u - k[r].unsqueeze(1) @ s)
            s = s + k[r].unsqueeze(2) * u
            out[r] = (q[r].unsqueeze(1) @ s).squeeze(1)
        state[c["slots"][i].long()] = s
        at += n
    return (out * (0.25 if op == "linear_channel" else 1.0) + skip).reshape(t, h * vd), state


def _off(a, b):
    return float((a.double() - b).norm() / b.norm())


OPS = ["linear_head", "linear_channel", "state_space", "delta_channel", "delta_head"]


@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("strong", [False, True])
@pytest.mark.parametrize("dim,vdim,new,extra,dtype,pad", [
    (128, 128, [64], [0], torch.bfloat16, 0),                              # one whole chunk
    (128, 128, [200, 1, 63, 0, 65, 17], [0, 9, 70, 3, 0, 1], torch.bfloat16, 8),   # remainders, an empty sequence, states read
    (64, 64, [129, 16], [5, 0], torch.float16, 3),                         # rows no vector load divides
    (96, 80, [70, 33], [0, 12], torch.bfloat16, 4),                        # padded keys
    (20, 24, [67, 40], [2, 0], torch.float32, 0),
    (33, 7, [66], [1], torch.bfloat16, 1)])                                # odd sizes
def test_chunks_match_the_recurrence_in_64_bits(op, strong, dim, vdim, new, extra, dtype, pad):
    """A row's result is a sum over at most a few hundred products of fp32 values, every one formed by at most 64 + 64
    roundings: 3e-6 bounds its relative error in norm (measured: 1e-7 to 4e-7)."""
    groups = 2 if op in ("state_space", "delta_head") else 4
    c = _case(op, 4, groups, dim, vdim, new, [n + e for n, e in zip(new, extra)], dtype, 11, strong, pad)
    want, want_state = _rows64(c)
    out, state = _run(c, True)
    off, off_state = _off(out, want), _off(state, want_state)
    assert off < 3e-6 and off_state < 3e-6, (off, off_state)
    untouched = [i for i in range(c["state"].shape[0]) if i not in c["slots"].tolist()]
    assert torch.equal(state[untouched], c["state"][untouched])
    again, state2 = _run(c, True)
    assert torch.equal(out, again) and torch.equal(state, state2)


def _many(n):
    """Lengths of ``n`` sequences around the chunk's 64 rows, some empty, and rows before them."""
    new = [(0, 1, 17, 64, 65, 5, 0, 33)[i % 8] for i in range(n)]
    return new, [(0, 3, 70)[i % 3] if m else 0 for i, m in enumerate(new)]


@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("heads,dim,vdim,new,extra,dtype,pad", [
    (16, 128, 128, [70, 64, 130, 65], [0, 9, 0, 3], torch.bfloat16, 8),        # 64 pairs and more: tiles of 32 columns
    (16, 128, 112, [33, 200, 1, 64], [0, 2, 5, 0], torch.float16, 0),          # the last tile half empty
    (32, 64, 200, [66, 90], [4, 0], torch.float32, 0),                         # values wider than a pass over them
    (4, 64, 128, [129, 20], [0, 7], torch.bfloat16, 0),
    (4, 64, 128, [80, 65], [1, 0], torch.float32, 3),                          # the same without vector loads
    (2, 128, 256, [65, 100], [0, 6], torch.bfloat16, 1),
    (4, 64, 64, *_many(70), torch.bfloat16, 8),                                # more sequences than a wave has lanes
    (8, 128, 128, *_many(131), torch.bfloat16, 0)])
def test_wide_tiles_wide_values_and_many_sequences(op, heads, dim, vdim, new, extra, dtype, pad):
    """The bound of ``test_chunks_match_the_recurrence_in_64_bits``."""
    groups = heads // 2 if op in ("state_space", "delta_head") else heads
    c = _case(op, heads, groups, dim, vdim, new, [n + e for n, e in zip(new, extra)], dtype, 17, False, pad)
    want, want_state = _rows64(c)
    out, state = _run(c, True)
    assert _off(out, want) < 3e-6 and _off(state, want_state) < 3e-6, (_off(out, want), _off(state, want_state))
    untouched = [i for i in range(c["state"].shape[0]) if i not in [int(x) for x, n in zip(c["slots"], new) if n]]
    assert torch.equal(state[untouched], c["state"][untouched])


@pytest.mark.parametrize("op", OPS)
def test_chunks_are_no_less_exact_than_the_walk(op):
    c = _case(op, 4, 4, 128, 128, [700, 300], [700, 420], torch.bfloat16, 3, False, 0)
    want, want_state = _rows64(c)
    (a, sa), (b, sb) = _run(c, True), _run(c, False)
    assert _off(a, want) <= 1.5 * _off(b, want) + 1e-7 and _off(sa, want_state) <= 1.5 * _off(sb, want_state) + 1e-7


@pytest.mark.parametrize("op", OPS)
def test_short_prompts_lose_no_more_than_row_by_row(op):
    """Root mean squares of the errors over small prompts, where each rounding inside a group of 16 rows shows: 0.94, 0.99, 0.85,
    0.99 and 1.02 times row by row (with a head's decays in the factors and sums in chains of 16: 1.08, 1.07, 0.97, 1.04, 1.10)."""
    sq = [0.0, 0.0]
    for i, (heads, dim, vdim, new) in enumerate([(2, 64, 128, [160]), (4, 64, 64, [88, 54]), (8, 64, 128, [157]),
                                                 (4, 128, 64, [162]), (8, 128, 128, [111, 65]), (4, 64, 128, [309, 134])]):
        c = _case(op, heads, heads, dim, vdim, new, [n + 9 for n in new], torch.bfloat16, 40 + i)
        want, _ = _rows64(c)
        for j in (0, 1):
            sq[j] += _off(_run(c, j == 0)[0], want) ** 2
    assert sq[0] ** 0.5 <= 1.05 * sq[1] ** 0.5


def test_many_heads_are_taken_in_turns(monkeypatch):
    c = _case("delta_channel", 6, 3, 64, 64, [90, 70], [90, 71], torch.bfloat16, 5)
    want = _run(c, True)
    monkeypatch.setattr(hip, "CHUNK_SCRATCH_BYTES", 1)
    got = _run(c, True)
    assert torch.equal(want[0], got[0]) and torch.equal(want[1], got[1])


@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("what,value", [("v", float("nan")), ("v", float("inf")), ("k", float("nan")), ("q", float("nan")),
                                        ("beta", float("nan")), ("dt", float("nan"))])
@pytest.mark.parametrize("heads,dim,vdim", [(4, 128, 128), (64, 64, 64)])      # tiles of 16 and of 32 value columns
def test_what_is_not_finite_stays_in_its_row_and_behind(op, what, value, heads, dim, vdim):
    """A row's NaN or infinity changes nothing in the rows in front of it, nor in other sequences; its own row shows it."""
    if (what == "beta" and not op.startswith("delta")) or (what == "dt" and op.startswith("linear")):
        pytest.skip("the recurrence has no such input")
    new, row, head = [150, 40, 70, 33], 21 + 64, 2                 # the first sequence's second chunk, inside a group of 16
    c = _case(op, heads, heads, dim, vdim, new, [150, 47, 70, 35], torch.float32, 7)
    clean, _ = _run(c, True)
    if what in ("beta", "dt"):
        c[what][row] = value
    else:
        at = {"q": 0, "k": heads * dim, "v": 2 * heads * dim}
        if op == "state_space":
            at = {"v": 0, "k": heads * vdim, "q": heads * vdim + heads * dim}
        c["x"][row, at[what] + head * (vdim if what == "v" else dim) + 5] = value
    got, _ = _run(c, True)
    other = torch.ones(sum(new), dtype=torch.bool, device=DEV)
    other[row:150] = False
    # (a decay that is no number makes its group multiply out the products between two rows: other roundings)
    assert _off(got[other], clean[other].double()) < 3e-6
    assert not torch.isfinite(got[row].view(heads, vdim)[head]).all()


@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("heads,dim,vdim", [(3, 64, 32), (2, 128, 136), (1, 128, 16)])
def test_columns_of_the_walk_are_the_same_numbers_by_16_and_by_32(monkeypatch, op, heads, dim, vdim):
    c = _case(op, heads, 1 if op == "state_space" else heads, dim, vdim, [130, 64, 1, 200], [130, 80, 9, 200], torch.bfloat16, 31)
    got = []
    for columns in (16, 32):
        monkeypatch.setattr(hip, "chunk_columns", lambda *sizes: columns)
        got.append(_run(c, True))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    want, want_state = _rows64(c)
    assert _off(got[1][0], want) < 3e-6 and _off(got[1][1], want_state) < 3e-6


@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("new", [[700, 300, 1, 1], [900] + [1] * 40])
@pytest.mark.parametrize("chunked", [True, None])
def test_the_memory_profile_holds_what_a_step_allocates(monkeypatch, op, new, chunked):
    """``chunk_scan_bytes`` (the runner keeps as much aside) covers the peak of a call, also for a step of fewer rows, and with the
    shortest segments that are made (``chunked`` None)."""
    if chunked is None:
        if op.startswith("delta"):
            pytest.skip("the delta rule has no segments")
        _segments(monkeypatch, 96)
    from vllm_distributed_amd import ops
    heads, groups, dim, vdim = 16, 16, 64, 128
    c = _case(op, heads, groups, dim, vdim, new, new, torch.bfloat16, 9)
    _run(c, chunked)
    state = c["state"].nbytes                                       # (``_run`` works on a copy)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    _run(c, chunked)
    torch.cuda.synchronize()
    used = torch.cuda.max_memory_allocated() - before - state
    bound = ops.recurrence_bytes(2000, len(new), heads, dim, vdim, op.startswith("delta"))
    assert 0 < used <= bound + 65536, (used, bound)                 # (offsets and lengths, rounded up to 512 bytes each)


@pytest.mark.parametrize("op", OPS[:3])
@pytest.mark.parametrize("rows", [0, 32, 96])
@pytest.mark.parametrize("strong", [False, True])
@pytest.mark.parametrize("heads,dim,vdim,new,extra,dtype", [
    (4, 128, 128, [200, 1, 63, 0, 65, 17, 96, 97], [0, 9, 70, 3, 0, 1, 0, 5], torch.bfloat16),     # remainders, states read
    (2, 64, 64, [129, 16, 192], [5, 0, 0], torch.float16),
    (4, 96, 80, [70, 33], [0, 12], torch.bfloat16),                        # keys and columns that end inside a tile
    (2, 24, 40, [67, 40], [2, 0], torch.float32),
    (2, 128, 256, [65, 100], [0, 6], torch.bfloat16),                      # two tiles of columns
    (2, 72, 64, [161], [3], torch.bfloat16),
    (2, 64, 136, [31, 160], [0, 0], torch.float32),
    (3, 64, 64, *_many(70), torch.bfloat16)])                              # more sequences than a wave has lanes
def test_segments_match_the_recurrence_in_64_bits(monkeypatch, op, rows, strong, heads, dim, vdim, new, extra, dtype):
    """The bound of ``test_chunks_match_the_recurrence_in_64_bits``, whatever sequences are cut at (0: nowhere)."""
    _segments(monkeypatch, rows)
    c = _case(op, heads, 1 if op == "state_space" else heads, dim, vdim, new, [n + e for n, e in zip(new, extra)], dtype, 23,
              strong, 8)
    want, want_state = _rows64(c)
    out, state = _run(c, None)
    assert _off(out, want) < 3e-6 and _off(state, want_state) < 3e-6, (_off(out, want), _off(state, want_state))
    untouched = [i for i in range(c["state"].shape[0]) if i not in [int(x) for x, n in zip(c["slots"], new) if n]]
    assert torch.equal(state[untouched], c["state"][untouched])
    again, state2 = _run(c, None)
    assert torch.equal(out, again) and torch.equal(state, state2)


@pytest.mark.parametrize("op", OPS[:3])
@pytest.mark.parametrize("rows", [0, 96])
def test_segments_are_no_less_exact_than_chunks(monkeypatch, op, rows):
    """Products in thirds of 24 digits, whose left-out parts are below 2^-21 of them with either sign."""
    c = _case(op, 4, 4, 128, 128, [700, 300], [700, 420], torch.bfloat16, 3)
    want, want_state = _rows64(c)
    off = []
    for chunked in (True, None):
        if chunked is None:
            _segments(monkeypatch, rows)
        out, state = _run(c, chunked)
        off.insert(0, (_off(out, want), _off(state, want_state)))
    assert off[0][0] <= 1.05 * off[1][0] and off[0][1] <= 1.05 * off[1][1], off


@pytest.mark.parametrize("op", OPS[:3])
@pytest.mark.parametrize("what,value", [("v", float("nan")), ("v", float("inf")), ("k", float("nan")), ("q", float("nan")),
                                        ("dt", float("nan"))])
@pytest.mark.parametrize("rows", [0, 64])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])      # (of 16 bits, operands may be one piece)
def test_what_is_not_finite_stays_in_its_row_and_behind_in_segments(monkeypatch, op, what, value, rows, dtype):
    if what == "dt" and op.startswith("linear"):
        pytest.skip("the recurrence has no such input")
    _segments(monkeypatch, rows)
    heads, dim, vdim, new, row, head = 4, 128, 128, [150, 40, 70, 33], 21 + 64, 2
    c = _case(op, heads, heads, dim, vdim, new, [150, 47, 70, 35], dtype, 7)
    clean, _ = _run(c, None)
    if what == "dt":
        c[what][row] = value
    else:
        at = {"q": 0, "k": heads * dim, "v": 2 * heads * dim}
        if op == "state_space":
            at = {"v": 0, "k": heads * vdim, "q": heads * vdim + heads * dim}
        c["x"][row, at[what] + head * (vdim if what == "v" else dim) + 5] = value
    got, _ = _run(c, None)
    other = torch.ones(sum(new), dtype=torch.bool, device=DEV)
    other[row:150] = False
    assert _off(got[other], clean[other].double()) < 3e-6
    assert not torch.isfinite(got[row].view(heads, vdim)[head]).all()
    if what == "v":                                                 # the columns beside it are as they were
        beside = torch.ones(vdim, dtype=torch.bool, device=DEV)
        beside[5] = False
        there = slice(row, 150)
        assert _off(got[there].view(-1, heads, vdim)[:, :, beside], clean[there].view(-1, heads, vdim)[:, :, beside].double()) < 3e-6


@pytest.mark.parametrize("rows", [-1, 0, 32])                                  # the chunked kernels; segments, whole and cut
def test_activated_inputs_far_below_zero_go_to_zero(monkeypatch, rows):
    """SiLU of what its exponential overflows for.  One row's key and query have one entry, and its value is read out again: a
    product of three activations, each within 2e-7 of 64 bits, and zero (to denormals) where they are."""
    if rows >= 0:
        _segments(monkeypatch, rows)
    heads, dim, new = 1, 64, [48, 48]
    x = torch.zeros(96, 3 * dim, device=DEV)
    entries = torch.tensor([-0.5, -20.0, -80.0, -87.0, -88.0, -90.0, -100.0, -200.0, -1e4, -1e30, -3e38, 3e37], device=DEV)
    x[5, 0], x[5, dim] = 1.5, 2.5
    x[5, 2 * dim:2 * dim + len(entries)] = entries
    c = {"op": "linear_head", "heads": heads, "groups": heads, "dim": dim, "vdim": dim, "new": new, "lens": new, "x": x,
         "state": torch.zeros(2, heads, dim, dim, device=DEV), "slots": torch.tensor([1, 0], dtype=torch.int32, device=DEV),
         "decay": torch.full((heads,), 0.5, device=DEV), "beta": torch.zeros(96, heads, device=DEV)}
    want, want_state = _rows64(c)
    out, state = _run(c, True if rows < 0 else None)
    got, ref = out[5].double(), want[5]
    assert torch.isfinite(out).all() and torch.isfinite(state).all()
    assert ((got - ref).abs() <= 8e-7 * ref.abs() + 1e-36).all(), (got[:len(entries)].tolist(), ref[:len(entries)].tolist())
    assert float((state.double() - want_state).abs().max()) <= 8e-7 * float(want_state.abs().max())


@pytest.mark.parametrize("rate", [0.05, 0.5, 1.0, 4.0, 16.0])
def test_decays_per_channel_are_as_exact_as_row_by_row(rate):
    """Rows that leave the state alone but for its decay, one a sequence: the state is the decays themselves, here and from the library's
    functions in the kernel for decoded rows.  Root mean squares over 2^17 values are known to a part in 500; 1.01 is five of them."""
    heads, dim, rows = 8, 128, 128
    g = torch.Generator(DEV).manual_seed(13)
    for lo, hi in ((-16.0, -6.0), (-6.0, -2.0), (-2.0, 2.0), (2.0, 8.0), (8.0, 30.0)):
        if rate * hi > 80:                                          # (decays beyond 32 bits)
            continue
        x = torch.randn(rows, 3 * heads * dim, generator=g, device=DEV)
        dt = torch.rand(rows, heads * dim, generator=g, device=DEV) * (hi - lo) + lo
        a_log = (rate * torch.exp(torch.rand(heads, generator=g, device=DEV) * 0.2 - 0.1)).log()
        slots = torch.arange(rows, dtype=torch.int32, device=DEV)
        qsl, lens = torch.arange(rows + 1, dtype=torch.int32, device=DEV), torch.full((rows,), 2, dtype=torch.int32, device=DEV)
        arg = dt.double().view(rows, heads, dim)
        want = torch.exp(-a_log.exp().double().view(1, heads, 1) * F.softplus(arg, threshold=60.0))
        off = []
        for chunked in (True, False):
            state = torch.ones(rows, heads, dim, 16, device=DEV)
            hip.gated_delta_rule(torch.cat([x[:, :2 * heads * dim], x[:, :heads * 16]], 1), heads, heads, dim, 16,
                                 torch.full((rows, heads), -1e4, device=DEV), dt, torch.zeros(heads * dim, device=DEV), a_log,
                                 state, slots, qsl, lens, 1e-6, 1, 0, chunked)
            off.append(float(((state.double() - want.unsqueeze(-1)) / want.unsqueeze(-1))[..., 0].pow(2).mean().sqrt()))
        assert 0.0 < off[0] <= 1.01 * off[1], (lo, hi, off)


@pytest.mark.parametrize("rows", [-1, 0])                                      # the chunked kernels, segments
def test_a_key_over_its_decays_is_rounded_once(monkeypatch, rows):
    """Sequences of one group of 16 rows, whose first brings a key and whose queries read it again: the decays behind it, divided by and
    multiplied with, leave the key.  Rounded to nearest, a number is off by 2.5e-8 (root mean square): the quotient, the product,
    and with operands in thirds the 1.9e-8 of what is left out."""
    if rows >= 0:
        _segments(monkeypatch, rows)
    heads, dim, seqs, at = 16, 64, 512, 37
    g = torch.Generator(DEV).manual_seed(29)
    key = torch.randn(seqs, heads, generator=g, device=DEV)
    x = torch.zeros(seqs, 16, 3, heads, dim, device=DEV)
    x[:, :, 0, :, at] = 1.0
    x[:, 0, 1, :, at] = key
    x[:, 0, 2, :, 5] = 1.0
    decay = torch.ones(seqs, 16, heads, dim, device=DEV)
    decay[:, 0, :, at] = torch.rand(seqs, heads, generator=g, device=DEV) * 0.9 + 0.1
    qsl = torch.arange(seqs + 1, dtype=torch.int32, device=DEV) * 16
    lens = torch.full((seqs,), 16, dtype=torch.int32, device=DEV)
    out = hip.decay_linear_attention(x.view(seqs * 16, -1), heads, dim, dim, decay.view(seqs * 16, -1),
                                     torch.zeros(seqs, heads, dim, dim, device=DEV), torch.arange(seqs, dtype=torch.int32, device=DEV),
                                     qsl, lens, False, 0, 1.0, True if rows < 0 else None).view(seqs, 16, heads, dim)
    off = float(((out[:, 15, :, 5].double() - key.double()) / key.double()).pow(2).mean().sqrt())
    parts = [2.53e-8, 2.53e-8] + ([1.9e-8] if rows == 0 else [])
    assert 0.0 < off <= 1.06 * sum(p * p for p in parts) ** 0.5, off
