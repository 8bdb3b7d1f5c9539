"""Which calls may go to the row kernels on a layer's parameters: everything
that makes calling the module more than its product, or that the kernels
can't read, keeps the call on the module (decided on the host; no GPU)."""
import pytest
import torch
import torch.nn as nn

import coda_gqa_l

D, H, HKV = 128, 4, 2


def _layer(dtype=torch.bfloat16):
    return coda_gqa_l.CoDAGQA(embed_dim=D, num_heads=H, num_kv_heads=HKV).to(dtype).eval()


def _x(B=2, L=1, width=D, dtype=torch.bfloat16):
    return torch.zeros(B, L, width, dtype=dtype)


class Mine(nn.Linear):
    pass


class MyWeight(nn.Parameter):
    pass


def _set(name, fn):
    def change(m):
        lin = getattr(m, name)
        out = fn(lin)
        if isinstance(out, nn.Module):
            setattr(m, name, out)
    return change


def _weight(fn):
    return lambda lin: setattr(lin, "weight", fn(lin.weight.detach()))


CHANGES = {
    "forward hook": _set("q_proj", lambda l: l.register_forward_hook(lambda *a: None) and None),
    "pre-hook": _set("v_proj", lambda l: l.register_forward_pre_hook(lambda *a: None) and None),
    "own forward": _set("k_proj", lambda l: setattr(l, "forward", lambda x: x)),
    "subclass": _set("lambda_proj", lambda l: Mine(l.in_features, l.out_features).bfloat16()),
    "weight class": _set("q_proj", _weight(lambda w: MyWeight(w.clone()))),
    "other dtype": _set("v_proj", lambda l: l.float()),
    "bias dtype": _set("lambda_proj", lambda l: setattr(l, "bias", nn.Parameter(l.bias.detach().float()))),
    "other device": _set("q_proj", lambda l: l.to("meta")),
    "rows": _set("k_proj", _weight(lambda w: nn.Parameter(w[:-1].clone()))),
    "features": _set("k_proj", lambda l: nn.Linear(D, 2 * l.out_features, bias=False).bfloat16()),
    "width": _set("v_proj", lambda l: nn.Linear(2 * D, l.out_features, bias=False).bfloat16()),
    "column stride": _set("q_proj", _weight(lambda w: nn.Parameter(torch.zeros(w.shape[0], 2 * D, dtype=w.dtype)[:, ::2]))),
    "overlapping rows": _set("q_proj", _weight(lambda w: nn.Parameter(w[:1].expand(w.shape)))),
    "pruned": _set("q_proj", lambda l: torch.nn.utils.prune.identity(l, "weight") and None),
    "parametrized": _set("q_proj", lambda l: nn.utils.parametrize.register_parametrization(l, "weight", nn.Identity()) and None),
}


@pytest.mark.parametrize("what", list(CHANGES))
@torch.no_grad()
def test_not_on_the_kernels(what):
    import torch.nn.utils.parametrize  # noqa: F401
    import torch.nn.utils.prune  # noqa: F401
    m = _layer()
    assert m._front_rows(_x()) is not None
    CHANGES[what](m)
    assert m._front_rows(_x()) is None


@torch.no_grad()
def test_inputs():
    m, f = _layer(), _layer(torch.float32)
    assert m._front_rows(_x(128)) is not None and m._front_rows(_x(129)) is None and m._front_rows(_x(0)) is None
    assert f._front_rows(_x(32, dtype=torch.float32)) is not None and f._front_rows(_x(33, dtype=torch.float32)) is None
    assert m._front_rows(_x(width=2 * D)) is None and m._front_rows(_x(width=D // 2)) is None
    assert m._front_rows(_x(dtype=torch.float32)) is None and f._front_rows(_x()) is None
    assert not m._packed_front_ok(_x(width=2 * D)) and not m._packed_front_ok(_x(65)) and m._packed_front_ok(_x(64))
    # the addresses and strides are the parameters' own
    w, lam = m.k_proj.weight, m.lambda_proj
    got = m._front_rows(_x())
    assert got[3:6] == (w.data_ptr(), D, None) and got[9:] == (lam.weight.data_ptr(), D, lam.bias.data_ptr())
    assert m._front_rows(_x().as_subclass(type("T", (torch.Tensor,), {}))) is None
    with pytest.MonkeyPatch.context() as mp:
        mp.setattr(nn.Linear, "forward", lambda self, x: x)
        assert m._front_rows(_x()) is None
    with torch.autocast("cpu", dtype=torch.bfloat16):
        assert m._front_rows(_x()) is None
    with torch.enable_grad():
        assert m._front_rows(_x()) is None
        assert m.requires_grad_(False)._front_rows(_x()) is not None
        assert m._front_rows(_x().requires_grad_()) is None


@torch.no_grad()
def test_packed_weights_are_checked():
    kw = dict(embed_dim=D, num_heads=H, num_kv_heads=HKV, window=16, num_landmarks_exact=8, num_landmarks_summary=8)
    m = coda_gqa_l.CoDAGQALandmarkPerf2(**kw).bfloat16().eval()
    m._packed_weights(_x())
    with pytest.raises(RuntimeError, match="on cpu"):
        m._packed_weights(torch.empty(2, 1, D, dtype=torch.bfloat16, device="meta"))
    m.v_proj = nn.Linear(D, 2 * D, bias=False).bfloat16()
    with pytest.raises(RuntimeError, match="is not"):
        m._packed_weights(_x())


@pytest.mark.parametrize("what", ["class", "hook", "own forward", "length", "type", "far"])
def test_own_rope_module(what):
    m = _layer()
    dev = torch.device("cpu")
    assert m._angles_rows(dev, 5, 3) is not None
    if what == "class":
        m.rope = type("R", (type(m.rope),), {})(m.head_dim)
    elif what == "hook":
        m.rope.register_forward_hook(lambda *a: None)
    elif what == "own forward":
        m.rope.forward = lambda **k: None
    elif what == "length":
        m.rope.inv_freq = m.rope.inv_freq[:-1]
    elif what == "type":
        m.rope.inv_freq = m.rope.inv_freq.double()
    assert m._angles_rows(dev, (1 << 24) - 2 if what == "far" else 5, 3) is None
