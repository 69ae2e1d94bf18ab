"""The op wrappers' host module on the GPU: what the autograd functions around it still do
(saved-tensor hooks, side streams, refusals) and the optimiser's copies."""
import copy

import pytest
import torch

pytestmark = pytest.mark.gpu


def _block(dev):
    from fxlm.model import Block, GPTConfig
    torch.manual_seed(0)
    return Block(GPTConfig(vocab_size=64, seq_len=64, n_layer=1, n_head=2, d_model=128)).to(dev).bfloat16()


def _grads(block, x, dy):
    out = block(x)
    return [out, *torch.autograd.grad(out, [x, *block.parameters()], dy)]


def test_block_through_saved_tensor_hooks_and_a_side_stream(dev):
    block = _block(dev)
    x = torch.randn(4, 64, 128, device=dev).bfloat16().requires_grad_()
    dy = torch.randn(4, 64, 128, device=dev).bfloat16()
    ref = _grads(block, x, dy)
    with torch.autograd.graph.save_on_cpu():
        assert all(torch.equal(a, b) for a, b in zip(ref, _grads(block, x, dy)))
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        got = _grads(block, x, dy)
    torch.cuda.current_stream().wait_stream(s)
    assert all(torch.equal(a, b) for a, b in zip(ref, got))


def test_misaligned_and_refused_inputs(dev):
    from fxlm.attention import flash_attention
    from fxlm.norm import add_pre_norm, rms_norm
    w = torch.ones(64, device=dev).bfloat16()
    flat = torch.randn(3 + 10 * 64, device=dev).bfloat16()
    x = flat[3:].view(10, 64)                              # contiguous, 6 bytes past an aligned address
    assert torch.equal(rms_norm(x, w), rms_norm(x.clone(), w))
    assert all(torch.equal(a, b) for a, b in zip(add_pre_norm(x, x, w), add_pre_norm(x.clone(), x.clone(), w)))
    with pytest.raises(TypeError, match="must be bfloat16"):
        rms_norm(x.float(), w)
    with pytest.raises(ValueError, match="contiguous"):
        rms_norm(torch.randn(64, 64, device=dev).bfloat16().t(), w)
    q = torch.randn(1, 8, 2, 64, device=dev).bfloat16()
    with pytest.raises(TypeError, match="q must be bfloat16"):
        flash_attention(q.float(), q.float(), q.float())
    with pytest.raises(ValueError, match="share one 4-D shape"):
        flash_attention(q, q[:, :4], q)
    with pytest.raises(ValueError, match="must be positive"):   # the library's own check
        flash_attention(q, q, q, scale=-1.0)


@pytest.mark.parametrize("M", [1, 65, 256, 300])
@pytest.mark.parametrize("layout", ["offset", "expanded", "windows", "wide", "columns"])
def test_linear_of_any_layout(dev, M, layout):
    # what torch.mm takes: contiguous but not 16-byte aligned, one row repeated, overlapping windows, rows of
    # a wider tensor at an odd stride, a transpose; and gradients that arrive as an expanded row
    from fxgpu.fused_linear import linear
    K, N = 64, 192
    g = torch.Generator(device=dev).manual_seed(M)
    flat = torch.randn(3 + M * (K + 3) + 8 * M + K, device=dev, generator=g).bfloat16()
    x = {"offset": flat[3:3 + M * K].view(M, K), "expanded": flat[:K].expand(M, K), "windows": flat[:8 * (M - 1) + K].unfold(0, K, 8),
         "wide": flat[:M * (K + 3)].view(M, K + 3)[:, :K], "columns": flat[:M * K].view(K, M).t()}[layout]
    w = (torch.randn(N, K, device=dev, generator=g) * K ** -0.5).bfloat16()
    ref = x.float() @ w.float().t()
    # one bf16 rounding of the product, at a result's own size and at the largest's for fp32 sums
    bound = 2.0 ** -8 * ref.abs() + 1e-5 * ref.abs().max()
    assert bool(((linear(x, w).float() - ref).abs() <= bound).all())
    xs, ws = x.detach().requires_grad_(), w.clone().requires_grad_()
    for frozen in (True, False):     # dy of a column sum: one row expanded
        y = linear(xs, w if frozen else ws)
        got = torch.autograd.grad(y.sum(0), [xs] if frozen else [xs, ws], torch.ones(N, device=dev).bfloat16())
        want = [w.float().sum(0).expand(M, K), x.float().sum(0).expand(N, K)]
        for a, b in zip(got, want):
            assert a.shape == b.shape
            assert bool(((a.float() - b).abs() <= 2.0 ** -8 * b.abs() + 1e-4 * b.abs().max()).all())


def test_input_grad_of_rows_that_overlap(dev):
    from fxgpu.fused_linear import input_grad, small_dgrad
    w = (torch.randn(64, 72, device=dev) * 0.1).bfloat16()
    for dy in (torch.randn(64, device=dev).bfloat16().expand(100, 64), torch.randn(900, device=dev).bfloat16().unfold(0, 64, 8)[:100],
               torch.randn(6403, device=dev).bfloat16()[3:].view(100, 64), torch.randn(1, 64, device=dev).bfloat16().as_strided((1, 64), (0, 1))):
        assert small_dgrad(len(dy), 72, 64)
        ref = dy.float() @ w.float()
        assert bool(((input_grad(dy, w).float() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-5 * ref.abs().max()).all())


@pytest.mark.parametrize("M", [16, 256, 300])     # few rows, whole tiles, small tiles
def test_a_weight_on_the_host_is_refused(dev, M):
    # as torch.mm refuses it, and before any launch
    from fxgpu.abi import host
    from fxgpu.fused_linear import fused_linear, input_grad, linear, linear_wgrad
    x, w = torch.randn(M, 512, device=dev).bfloat16(), torch.randn(512, 512).bfloat16()
    b = torch.zeros(512).bfloat16()
    for call in (lambda: linear(x, w), lambda: fused_linear(x, w.to(dev), b, None), lambda: input_grad(x, w),
                 lambda: input_grad(x, w.to(dev), x.cpu()), lambda: host.linear_fwd(x, w, None, 0, False),
                 lambda: host.norm_bwd(x, x.cpu(), w[0].to(dev), x[:, 0].float(), None)):
        with pytest.raises(RuntimeError, match="expected all tensors to be on"):
            call()
    with pytest.raises(TypeError, match="cuda tensors"):
        linear_wgrad(x, x.cpu())


def test_optimizer_deepcopy_takes_the_same_step(dev):
    from fxlm.optim import FlatAdamW
    model = torch.nn.Linear(64, 40).to(dev)
    opt = FlatAdamW(model, init_scale=1.0)
    twin_model, twin = copy.deepcopy((model, opt))
    for m, o in ((model, opt), (twin_model, twin)):
        for p in m.parameters():
            p.grad = torch.ones_like(p)
        o.step()
    assert torch.equal(opt.master, twin.master) and float(opt._step_ctr) == 1


def test_optimizer_pickles_hold_tensors_and_numbers_only(dev):
    # whole-object files, those written before the host module among them: its objects are made anew
    import pickle
    from fxlm.optim import FlatAdamW
    model = torch.nn.Linear(64, 40).to(dev)
    opt = FlatAdamW(model, init_scale=1.0)
    assert b"_host" not in pickle.dumps(opt)
    old = FlatAdamW.__new__(FlatAdamW)
    old.__setstate__({k: v for k, v in opt.__dict__.items() if k not in ("_params", "_layout")})
    for p in model.parameters():
        p.grad = torch.ones_like(p)
    old.step()
    assert int(opt._step_ctr) == 1 and old._params[0] is opt._params[0]
    back = pickle.loads(pickle.dumps((model, opt)))[1]
    assert back._params[0] is not opt._params[0] and torch.equal(back.master, opt.master)
    for o in (back, opt):
        for p in o._params:
            p.grad = torch.ones_like(p)
        o.step()
    assert torch.equal(back.master, opt.master) and int(back._step_ctr) == 2


@pytest.mark.parametrize("B,V,D", [(1, 256, 64), (17, 50304, 768), (64, 1003, 1032)])
def test_decode_step_ends_equal_the_torch_operations(dev, B, V, D):
    # bit for bit: the embedding sum, the graph's inputs, and the head's bf16 logits as fp32
    from fxgpu.abi import host
    from fxgpu.fused_linear import linear_ex
    g = torch.Generator(device=dev).manual_seed(B + V)
    E, P = (torch.randn(n, D, device=dev, generator=g).bfloat16() for n in (V, 96))
    tok = torch.randint(0, V, (B,), device=dev, generator=g)
    tok_out, pos, lens = torch.zeros_like(tok), torch.zeros(1, dtype=torch.int64, device=dev), \
        torch.zeros(B, dtype=torch.int32, device=dev)
    assert host.decode_inputs(tok, 41, tok_out, pos, lens)
    assert torch.equal(tok, tok_out) and int(pos) == 41 and bool((lens == 42).all())
    assert not host.decode_inputs(tok.int(), 41, tok_out, pos, lens)
    x = host.decode_embed(tok_out, pos, E, P)
    assert torch.equal(x, torch.nn.functional.embedding(tok, E)[:, None] + P.index_select(0, pos))
    w = torch.ones(D, device=dev).bfloat16()
    assert torch.equal(host.few_rows_logits(x[:, 0], E, w, 1e-6), linear_ex(x[:, 0], E, norm_weight=w, eps=1e-6).float())


def test_decode_graph_takes_positions_of_any_number_type(dev):
    # a position as a float, a numpy integer or a 0-d tensor, as fill_() takes them
    import numpy as np
    from fxlm import GPT, GPTConfig
    torch.manual_seed(3)
    with torch.device(dev):
        model = GPT(GPTConfig(vocab_size=256, seq_len=64, n_layer=1, n_head=2, d_model=128)).bfloat16()
    cache = [tuple(torch.zeros(2, 64, 2, 64, device=dev).bfloat16() for _ in range(2))]
    step, tok = model.decode_graph(cache, 2), torch.tensor([5, 9], device=dev)
    want = step(tok, 7).clone()
    for pos in (7.0, np.int64(7), torch.tensor(7), torch.tensor(7, device=dev)):
        assert torch.equal(step(tok, pos), want), type(pos)


def test_hooks_on_the_embedding_run_in_cached_steps(dev):
    from fxlm import GPT, GPTConfig
    torch.manual_seed(3)
    with torch.device(dev):
        model = GPT(GPTConfig(vocab_size=256, seq_len=64, n_layer=1, n_head=2, d_model=128)).bfloat16()
    cache = [tuple(torch.zeros(2, 64, 2, 64, device=dev).bfloat16() for _ in range(2))]
    tok = torch.tensor([5, 9], device=dev)
    plain, graph = model.decode_step(tok, cache, 7), model.decode_graph(cache, 2)
    assert torch.equal(graph(tok, 7), plain)
    swap = {5: 9, 9: 5}
    handle = model.tok_emb.register_forward_pre_hook(lambda m, a: (torch.tensor([[swap[int(i)]] for i in a[0].flatten()], device=dev),))
    assert torch.equal(model.decode_step(tok, cache, 7), plain.flip(0))
    handle.remove()
    assert torch.equal(model.decode_step(tok, cache, 7), plain)


def test_rows_outside_the_tables(dev):
    # the graph's call refuses a position on the host; an id that no row has gives NaN to its own sequence
    from fxgpu.abi import host
    from fxlm import GPT, GPTConfig
    with torch.device(dev):
        model = GPT(GPTConfig(vocab_size=256, seq_len=16, n_layer=1, n_head=2, d_model=128)).bfloat16()
    step = model.decode_graph([tuple(torch.zeros(2, 32, 2, 64, device=dev).bfloat16() for _ in range(2))], 2)
    tok = torch.tensor([5, 9], device=dev)
    for pos in (-1, 16, 32, -1.0, torch.tensor(16)):
        with pytest.raises(ValueError, match="position"):
            step(tok, pos)
    assert bool(step(tok, 15).isfinite().all())
    E, P = (torch.randn(n, 72, device=dev).bfloat16() for n in (6, 4))
    ids, pos = torch.tensor([0, -1, 5, 6, 2 ** 40], device=dev), torch.tensor([3], device=dev)
    x = host.decode_embed(ids, pos, E, P)[:, 0]
    assert torch.equal(x[[0, 2]], E[[0, 5]] + P[3]) and bool(x[[1, 3, 4]].isnan().all())
    assert bool(host.decode_embed(ids, pos + 1, E, P).isnan().all())
