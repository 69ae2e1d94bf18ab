"""What the host module refuses before it launches anything (CPU)."""
import threading
import time

import pytest
import torch


@pytest.fixture(scope="module")
def host():
    from fxgpu.abi import host as h
    return h


def test_tensors_off_the_gpu_are_refused(host):
    # each function whose kernels would read or write the tensors' memory; nothing is launched
    x, w = torch.zeros(300, 512).bfloat16(), torch.zeros(512, 512).bfloat16()
    f, t = torch.zeros(300), torch.zeros(300, dtype=torch.int64)
    q = torch.zeros(1, 8, 2, 64).bfloat16()
    lse = torch.zeros(1, 2, 8)
    calls = [lambda: host.linear_fwd(x, w, None, 0, False), lambda: host.linear_fwd(x, w, w[0], 1, True),
             lambda: host.norm_bwd(x, x, w[0], f, None), lambda: host.norm_bwd(x, x, w[0], f, x),
             lambda: host.attn_bwd(q, q, q, q, lse, q, True, 0.125),
             lambda: host.attn_bwd_qkv(torch.zeros(1, 8, 3, 2, 64).bfloat16(), q, lse, q, True, 0.125),
             lambda: host.ce_inv_nvalid(t, -100, None, 1.0), lambda: host.ce_rows(x, t, x, f, f[0], -100),
             lambda: host.ce_finalize(f, f[0]), lambda: host.ce_scale_grad(x, f[0], f, -1),
             lambda: host.ce_lin_scale_inplace(w, x, f[0], None, 1.0),
             lambda: host.decode_inputs(t, 3, t.clone(), t[:1], t.int())]
    for i, call in enumerate(calls):
        with pytest.raises(RuntimeError, match="expected all tensors to be on one GPU"):
            call()
            pytest.fail(f"call {i} was not refused")
    with pytest.raises(TypeError, match="cuda tensors"):
        host.wgrad(x, x)
    for none in (host.norm_fwd(x, w[0], 1e-6), host.norm_add_fwd(x, x, w[0], 1e-6), host.attn_fwd(q, q, q, True, 0.125),
                 host.ce_fwd(x, t, -100, True), host.few_rows_logits(x[:4], w, w[0], 1e-6), host.gather_fwd(x, t.int(), w, w[0], True),
                 host.dgrad(x, w, None, False), host.dgrad(x, w, x, True)):
        assert none is None
    from fxgpu.fused_linear import input_grad
    assert torch.equal(input_grad(x + 1, w + 1), torch.mm(x + 1, w + 1))     # on the CPU as before: torch's product


def test_rows(host):
    # aligned rows that do not overlap: a view where t has them, else a copy
    flat = torch.arange(4096).bfloat16()
    base = flat.data_ptr()
    for t in (flat[:640].view(10, 64), flat[:640].view(2, 5, 64), flat.view(-1, 128)[:, 64:], flat[:64].view(1, 64)):
        r = host.rows(t)
        assert r.data_ptr() == t.data_ptr() and torch.equal(r, t.reshape(-1, 64))
    odd = (flat[3:643].view(10, 64), flat[:64].expand(10, 64), flat.unfold(0, 64, 8)[:10], flat[:640].view(64, 10).t(), flat[:690].view(10, 69)[:, :64],
           flat[:64].as_strided((1, 64), (0, 1)), flat[3:67].as_strided((1, 64), (1, 1)))
    for t in odd:
        r = host.rows(t)
        assert torch.equal(r, t) and r.stride() == (64, 1) and r.data_ptr() % 16 == 0
    assert host.rows(odd[-2]).data_ptr() == base       # one row: its stride alone was odd
    assert host.rows(flat[:0].view(0, 64)).shape == (0, 64)


def test_other_python_threads_run_during_a_call(host):
    stamps, stop = [], threading.Event()

    def tick():
        while not stop.is_set():
            stamps.append(time.perf_counter())
            time.sleep(1e-3)
    other = threading.Thread(target=tick)
    t = torch.ones(12000, 16000, dtype=torch.bfloat16).t()     # a copy of some 0.1 s
    other.start()
    t0 = time.perf_counter()
    host.rows(t)
    t1 = time.perf_counter()
    stop.set()
    other.join()
    third = (t1 - t0) / 3     # the call's middle, away from the switches at its ends
    assert any(t0 + third < s < t1 - third for s in stamps), (t1 - t0, len(stamps))


def test_a_hooked_embedding_is_no_table_lookup():
    from torch import nn

    from fxlm.model import _table_lookup

    class Other(nn.Embedding):
        def forward(self, i):
            return 2 * super().forward(i)
    assert _table_lookup(nn.Embedding(8, 8)) and not _table_lookup(Other(8, 8)) and not _table_lookup(nn.Embedding(8, 8, max_norm=1.0))
    for register in ("register_forward_hook", "register_forward_pre_hook", "register_full_backward_hook"):
        m = nn.Embedding(8, 8)
        handle = getattr(m, register)(lambda *a: None)
        assert not _table_lookup(m)
        handle.remove()
        assert _table_lookup(m)
    m.forward = lambda i: i
    assert not _table_lookup(m)
    handle = nn.modules.module.register_module_forward_hook(lambda *a: None)
    try:
        assert not _table_lookup(nn.Embedding(8, 8))
    finally:
        handle.remove()


def test_positions_outside_the_model_are_refused():
    from fxlm import GPT, GPTConfig
    model = GPT(GPTConfig(vocab_size=64, seq_len=16, n_layer=1, n_head=2, d_model=128))
    tok = torch.tensor([1, 2])
    cache = [tuple(torch.zeros(2, 32, 2, 64) for _ in range(2))]     # longer than the position table
    for pos in (-1, 16, 31, 32):
        with pytest.raises(ValueError, match="position"):
            model.decode_step(tok, cache, pos)
