"""GPU parity of the fused decode-step operations (whisperdrz_amd.decode_ops) against the
reference's own torch ops on the same GPU tensors.

* add_layernorm_: the new residual x + delta bit-identical to torch's add; the LayerNorm within
  one unit in the last place of the 16-bit result of torch's LayerNorm (both compute in fp32;
  the reduction order differs), with at least 99% of the elements bit-identical.
* add_layernorm_partials_: the delta given as fp32 split-K partials of a Linear plus its bias; the
  reference is torch's sequential fp32 sum of the partials plus the bias, rounded to the 16-bit
  type (the Linear's output), then the same add and LayerNorm: the residual bit-identical, the
  LayerNorm to the bar above.
* masked_argmax: token ids identical to the reference's sequence (zero, masked_fill -65504, add,
  repetition-penalty where, argmax; decoding.py:1729-1761, 854-855), ties and NaN logits included
  (a NaN is the maximum, as in torch.argmax).
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _ulp16(t: torch.Tensor) -> torch.Tensor:
    bits = 7 if t.dtype == torch.bfloat16 else 10
    a = t.float().abs().clamp_min(2.0 ** -14)
    return torch.exp2(torch.floor(torch.log2(a)) - bits)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,n", [(64, 1280), (3, 256), (130, 4096), (1, 8)])
def test_add_layernorm(cuda, dtype, rows, n):
    from whisperdrz_amd import add_layernorm_, layer_norm

    g = torch.Generator(device=cuda).manual_seed(rows + n)
    x = (3.0 * torch.randn(rows, n, generator=g, device=cuda) + 0.5).to(dtype)
    delta = torch.randn(rows, n, generator=g, device=cuda).to(dtype)
    ln = torch.nn.LayerNorm(n).to(cuda, dtype)
    with torch.no_grad():
        ln.weight.copy_(1.0 + 0.1 * torch.randn(n, generator=g, device=cuda))
        ln.bias.copy_(0.1 * torch.randn(n, generator=g, device=cuda))
    print(f"add_layernorm {dtype} rows={rows} n={n}", flush=True)
    x_ref = x + delta
    y_ref = ln(x_ref)
    x_in = x.clone()
    y = add_layernorm_(x_in, delta, ln)
    torch.cuda.synchronize()
    assert torch.equal(x_in, x_ref)  # the new residual, in place
    diff = (y.float() - y_ref.float()).abs()
    assert torch.all(diff <= _ulp16(y_ref) * 1.001), float(diff.max())
    assert (diff == 0).float().mean().item() >= 0.99
    # plain LayerNorm leaves x untouched
    x_keep = x.clone()
    y2 = layer_norm(x_keep, ln)
    assert torch.equal(x_keep, x)
    assert torch.all((y2.float() - ln(x).float()).abs() <= _ulp16(ln(x)) * 1.001)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,n,n_split", [(64, 1280, 4), (3, 256, 2), (130, 1536, 4), (1, 8, 4), (5, 1032, 2)])
def test_add_layernorm_partials(cuda, dtype, rows, n, n_split):
    from whisperdrz_amd import add_layernorm_partials_

    g = torch.Generator(device=cuda).manual_seed(rows * 5 + n + n_split)
    x = (3.0 * torch.randn(rows, n, generator=g, device=cuda) + 0.5).to(dtype)
    partials = torch.randn(n_split, rows, n, generator=g, device=cuda)
    fc = torch.nn.Linear(8, n).to(cuda, dtype)  # only its bias is used
    ln = torch.nn.LayerNorm(n).to(cuda, dtype)
    with torch.no_grad():
        fc.bias.copy_(0.5 * torch.randn(n, generator=g, device=cuda))
        ln.weight.copy_(1.0 + 0.1 * torch.randn(n, generator=g, device=cuda))
        ln.bias.copy_(0.1 * torch.randn(n, generator=g, device=cuda))
    print(f"add_layernorm_partials {dtype} rows={rows} n={n} n_split={n_split}", flush=True)
    acc = partials[0].clone()
    for z in range(1, n_split):
        acc = acc + partials[z]
    delta_ref = (acc + fc.bias.float()).to(dtype)
    x_ref = x + delta_ref
    y_ref = ln(x_ref)
    x_in = x.clone()
    y = add_layernorm_partials_(x_in, partials, fc, ln)
    torch.cuda.synchronize()
    assert torch.equal(x_in, x_ref)
    diff = (y.float() - y_ref.float()).abs()
    assert torch.all(diff <= _ulp16(y_ref) * 1.001), float(diff.max())
    assert (diff == 0).float().mean().item() >= 0.99


def test_add_layernorm_partials_errors(cuda):
    from whisperdrz_amd import add_layernorm_partials_

    x = torch.randn(4, 2048, device=cuda).to(torch.bfloat16)
    fc = torch.nn.Linear(8, 2048).to(cuda, torch.bfloat16)
    ln = torch.nn.LayerNorm(2048).to(cuda, torch.bfloat16)
    with pytest.raises(NotImplementedError, match="1536"):
        add_layernorm_partials_(x, torch.zeros(4, 4, 2048, device=cuda), fc, ln)
    with pytest.raises(ValueError):
        add_layernorm_partials_(x, torch.zeros(4, 3, 2048, device=cuda), fc, ln)


def _reference_sampling(logits, blocked, penalty):
    additive = torch.zeros_like(logits)
    if blocked is not None:
        additive.masked_fill_(blocked, -65504)
    masked = logits + additive
    if penalty is not None:
        penalized = torch.where(masked > 0, masked / 1.2, masked * 1.2)
        masked = torch.where(penalty, penalized, masked)
    return masked.argmax(dim=-1)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_masked_argmax(cuda, dtype):
    from whisperdrz_amd import masked_argmax

    rows, V = 64, 51866
    g = torch.Generator(device=cuda).manual_seed(3)
    logits = (4.0 * torch.randn(rows, V, generator=g, device=cuda)).to(dtype)
    logits[5] = torch.round(logits[5].float()).to(dtype)  # many ties: lowest index wins
    blocked = torch.rand(rows, V, generator=g, device=cuda) < 0.3
    blocked[7] = True  # every token blocked
    penalty = torch.rand(rows, V, generator=g, device=cuda) < 0.01
    # the argmax of some rows is a penalised token (positive and negative maxima)
    top = logits.float().argmax(dim=-1)
    penalty[torch.arange(0, rows, 3, device=cuda), top[0::3]] = True
    logits[9] = -logits[9].abs()
    # NaN logits: torch.argmax takes a NaN as the maximum, so does the kernel
    logits[11, 1234] = float("nan")
    logits[12, 60] = float("nan")
    logits[12, 50] = float("nan")
    logits[13] = float("nan")
    print(f"masked_argmax {dtype}", flush=True)
    for b, p in [(blocked, penalty), (blocked, None), (None, penalty), (None, None)]:
        got = masked_argmax(logits, b, p)
        want = _reference_sampling(logits, b, p)
        torch.cuda.synchronize()
        assert torch.equal(got, want), (got != want).nonzero()[:5].tolist()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,V", [(5, V) for V in (1, 7, 8, 9, 2047, 2049, 4096, 4097, 8191, 8193, 57344, 57353)]
                         + [(513, V) for V in (4, 14336, 14337)])
def test_masked_argmax_vector_edges(cuda, dtype, rows, V):
    """Row lengths around the 8-token loads, one round of them (14336 from 256 threads, 57344 from
    1024) and the lines between the two forms, rows and mask rows at odd offsets (unaligned loads), the
    maximum at the first, last and last vectorised token; whole numbers compared exactly."""
    from whisperdrz_amd import masked_argmax

    g = torch.Generator(device=cuda).manual_seed(V)
    logits = torch.randn(rows, V + 3, generator=g, device=cuda).to(dtype)[:, 1 : V + 1]
    blocked = (torch.rand(rows, V + 5, generator=g, device=cuda) < 0.2)[:, 3:]
    penalty = (torch.rand(rows, V + 2, generator=g, device=cuda) < 0.2)[:, 1:]
    for row, i in ((0, 0), (1, V - 1), (2, V // 8 * 8 - 1), (3, V // 2)):
        logits[row, max(i, 0)] = 9.0
    logits[4] = float("-inf")
    for b, p in [(blocked, penalty), (None, None)]:
        got = masked_argmax(logits, b, p)
        want = _reference_sampling(logits, b[:, :V] if b is not None else None, p[:, :V] if p is not None else None)
        assert torch.equal(got, want), (V, got.tolist(), want.tolist())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,sq,n,with_slots", [(1, 1, 1280, True), (5, 1, 8, True), (3, 7, 520, False), (70, 2, 2048, True)])
def test_step_begin_end(cuda, dtype, B, sq, n, with_slots):
    """The prologue against torch's indexing, add and this library's LayerNorm (same bits), and the
    epilogue's bump: repeated and negative slots, strided indices, ids out of range."""
    from whisperdrz_amd import layer_norm
    from whisperdrz_amd.decode_ops import step_begin, step_end_

    g = torch.Generator(device=cuda).manual_seed(B * n + sq)
    V, ctx, layers, n_slots = 50, 20, 3, B + 4
    emb, pos = (torch.randn(r, n, generator=g, device=cuda).to(dtype) for r in (V, ctx))
    ln = torch.nn.LayerNorm(n).to(cuda, dtype)
    with torch.no_grad():
        ln.weight.copy_(1 + 0.1 * torch.randn(n, generator=g, device=cuda))
    tokens = torch.randint(0, V, (B, 2 * sq), generator=g, device=cuda)[:, ::2]
    positions = torch.randint(-ctx, ctx, (B,), generator=g, device=cuda).unsqueeze(1).expand(B, sq)
    lens = torch.randint(0, 9, (layers, n_slots), generator=g, device=cuda, dtype=torch.int32)
    slots = torch.randint(-n_slots, n_slots, (B,), generator=g, device=cuda) if with_slots else None
    x, h, slots32, seqlens = step_begin(tokens, positions, emb, pos, ln, slots, lens)
    want = emb[tokens] + pos[positions]
    assert torch.equal(x, want) and torch.equal(h, layer_norm(want, ln))
    want_lens = lens.clone()
    if with_slots:
        assert torch.equal(slots32, slots.int()) and torch.equal(seqlens, lens[:, slots])
        want_lens[:, slots] += sq
    else:
        assert slots32 is None and torch.equal(seqlens, lens[:, :B])
        want_lens[:, :B] += sq
    step_end_(lens, seqlens, slots, sq)
    assert torch.equal(lens, want_lens)
    # out of range: NaN rows, length -1, nothing bumped; the other rows as before
    tokens = tokens.clone()
    tokens[0, 0] = V
    if with_slots:
        slots[0] = n_slots
    x2, h2, _, seqlens2 = step_begin(tokens, positions, emb, pos, ln, slots, lens)
    assert x2[0, 0].isnan().all() and h2[0, 0].isnan().all()
    assert torch.equal(x2.view(B * sq, n)[1:], x.view(B * sq, n)[1:])
    if with_slots:
        assert (seqlens2[:, 0] == -1).all()


def test_step_ends_operands(cuda):
    """Operands elsewhere, of other types or of sizes that do not fit are refused on the host."""
    from whisperdrz_amd.decode_ops import step_begin, step_end_

    i32, i64, dt = torch.int32, torch.int64, torch.bfloat16
    lens, seqlens = torch.zeros(2, 4, dtype=i32, device=cuda), torch.zeros(2, 3, dtype=i32, device=cuda)
    slots = torch.zeros(3, dtype=i64, device=cuda)
    for bad in ((lens, seqlens.cpu(), slots), (lens, seqlens, slots.cpu()), (lens.cpu(), seqlens, slots)):
        with pytest.raises(RuntimeError, match="is on"):
            step_end_(*bad, 1)
    with pytest.raises(TypeError):
        step_end_(lens.long(), seqlens, slots, 1)
    for bad in ((lens[:1], seqlens, slots), (lens, seqlens[:, ::2], None), (lens, seqlens, slots[:2]),
                (lens, seqlens, slots.int()), (lens[:, :2].contiguous(), seqlens, None)):
        with pytest.raises(ValueError):
            step_end_(*bad, 1)
    tok = torch.zeros(3, 1, dtype=i64, device=cuda)
    emb = torch.zeros(5, 16, dtype=dt, device=cuda)
    with pytest.raises(RuntimeError, match="is on cpu"):
        step_begin(tok, tok, emb, emb, torch.nn.LayerNorm(16).to(dt), slots, lens)


@pytest.mark.parametrize("which", ["token", "position", "slot"])
def test_step_begin_debug_mode_refuses_ids(cuda, monkeypatch, which):
    """WDRZ_DEBUG=1: an id out of range is refused on the host instead of giving a NaN row."""
    from whisperdrz_amd import _lib
    from whisperdrz_amd.decode_ops import step_begin

    monkeypatch.setenv("WDRZ_DEBUG", "1")
    assert _lib.debug_mode()
    ids = {"token": [[1], [2]], "position": [[0], [3]], "slot": [0, 1]}
    emb = torch.zeros(5, 16, dtype=torch.bfloat16, device=cuda)
    ln = torch.nn.LayerNorm(16).to(cuda, torch.bfloat16)
    lens = torch.zeros(2, 4, dtype=torch.int32, device=cuda)
    call = lambda i: step_begin(*(torch.tensor(i[k], device=cuda) for k in ("token", "position")), emb, emb, ln,
                                torch.tensor(i["slot"], device=cuda), lens)
    call(ids)
    ids[which][1] = 9 if which == "slot" else [9]
    with pytest.raises(IndexError, match=which):
        call(ids)
