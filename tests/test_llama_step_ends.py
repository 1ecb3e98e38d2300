"""Both ends of a Llama step: the embedding's rows in one launch (csrc/kernels/norm_act.hip) and the norm behind the last layer
inside the native layer stack (csrc/kernels/llama_exec.hip): the bits of torch's lookup and of the separate norm."""
import pytest
import torch

from k8s_llm_rca_amd.ops import norm as N


@pytest.mark.parametrize("dev", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("dt,W", [(torch.bfloat16, 4096), (torch.bfloat16, 8), (torch.float32, 260), (torch.bfloat16, 12)])
@pytest.mark.parametrize("T", [0, 1, 33])
def test_lookup(dev, dt, W, T):
    g = torch.Generator().manual_seed(W + T)
    embed = torch.randn(50, W, generator=g).to(dt).to(dev)
    ids = torch.randint(0, 50, (T,), generator=g, dtype=torch.int32).to(dev)
    out = N.lookup_rows(ids, embed)
    assert out.dtype == dt and torch.equal(out, embed[ids.long()])


@pytest.mark.gpu
def test_ids_outside_the_table():
    embed = torch.ones(5, 4096, dtype=torch.bfloat16, device="cuda")
    out = N.lookup_rows(torch.tensor([4, 5, -1, 0], dtype=torch.int32, device="cuda"), embed)
    assert torch.isnan(out).all(1).tolist() == [False, True, True, False] and bool((out[[0, 3]] == 1).all())


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 2, 5, 16, 40])
@pytest.mark.parametrize("deferred", [True, False])
def test_last_norm(monkeypatch, T, deferred):
    from k8s_llm_rca_amd.models.llama import LlamaModel
    from k8s_llm_rca_amd.models.registry import get_any_config
    from k8s_llm_rca_amd.ops import layer_exec as LX
    from k8s_llm_rca_amd.ops import linear as LIN
    monkeypatch.setattr(LX, "_fuse_splitk", deferred)
    cfg = get_any_config("llama3-8b", n_layers=2, vocab_size=512)
    m = LlamaModel(cfg, "cuda", seed=3)
    ex = LX.LlamaExecutor(m)
    g = torch.Generator().manual_seed(T)
    x = torch.randn(T, cfg.hidden, generator=g).to(torch.bfloat16).cuda()
    kc = torch.zeros(cfg.n_layers, 4, m.nkv, 64, m.D, dtype=torch.bfloat16, device="cuda")
    vc = torch.zeros(cfg.n_layers, 4, m.nkv, m.D, 64, dtype=torch.bfloat16, device="cuda")

    class Inp:
        n_decode, meta_decode, meta_prefill, slots = 0, None, None, None
        positions = torch.arange(T, dtype=torch.int32, device="cuda")
    LIN.reserve_lib_workspace(torch.device("cuda", torch.cuda.current_device()))
    # (no attention in this step: its buffer is what scratch gives, the same for both)
    monkeypatch.setattr(LX, "scratch", lambda shape, dt, dev: torch.zeros(shape, dtype=dt, device=dev))
    prev, res = ex.run(Inp, x.clone(), kc, vc)
    want = torch.empty_like(res)
    N.rmsnorm(prev, m.final_norm, cfg.rms_eps, residual=res, out=want)
    got = ex.run_normed(Inp, x.clone(), kc, vc, m.final_norm)
    assert torch.isfinite(got).all() and torch.equal(got, want)
