"""The device wrappers of hetero/q4.py check every tensor before the library
sees its pointer: the entry points take raw device pointers and sizes, so a
buffer of the wrong type or size would be read or written past its end by a
kernel.  CPU tensors here: each wrong argument raises before any library
call (a CPU tensor of the right type raises for its device)."""
import pytest
import torch

from hetero import q4


def mat(n_out=64, n_in=256, gs=64, wdt=torch.int32, sdt=torch.int16):
    return (torch.zeros((n_out, n_in // 8), dtype=wdt), torch.zeros((n_out, n_in // gs), dtype=sdt),
            torch.zeros((n_out, n_in // gs), dtype=sdt))


def test_wrong_types_and_sizes_raise_before_the_library():
    m = mat()
    x32 = torch.zeros((1, 256))
    with pytest.raises(TypeError):
        q4.gemv_dev(*m, x32.to(torch.bfloat16))                   # fp32 x only
    with pytest.raises(TypeError):
        q4.gemm_bf16_dev(*m, x32.to(torch.bfloat16))              # rounds fp32 x itself
    with pytest.raises(TypeError):
        q4.gemv_dev(*mat(wdt=torch.float32), x32)                 # packed words
    with pytest.raises(TypeError):
        q4.gemv_dev(*mat(sdt=torch.float32), x32)                 # 16-bit scales
    with pytest.raises(ValueError):
        q4.gemv_dev(m[0], m[1][:, :2], m[2], x32)                 # scales of another group size
    with pytest.raises(ValueError):
        q4.gemv_dev(*m, x32, out=torch.zeros((1, 32)))            # output too small
    with pytest.raises(ValueError):
        q4.gemv_multi_dev([m, mat(n_in=512)], x32)                # n_in differs
    with pytest.raises(TypeError):
        q4.gemm_bf16_gate_up_silu_dev(m, m, x32)                  # bf16 x only
    with pytest.raises(ValueError):
        q4.gate_up_silu_dev(m, mat(n_out=32), x32)                # gate and up differ
    with pytest.raises(ValueError):
        q4.mlp_dev(m, m, mat(n_out=128, n_in=64), x32)            # down does not map back
    with pytest.raises(ValueError):
        q4.norm_gemv_multi_dev([m], x32, None, torch.zeros(128), 1e-6)   # norm weights too short
    with pytest.raises(ValueError):
        q4.dequant_dev(*m, out=torch.zeros((64, 128)))            # output too small
    with pytest.raises(TypeError):
        q4.norm_gemv_argmax_dev(m, x32, None, torch.zeros(256), 1e-6, torch.zeros(1, dtype=torch.int32),
                                torch.zeros(1, dtype=torch.int64))
    with pytest.raises(ValueError, match="GPU tensors"):
        q4.gemv_dev(*m, x32)                                      # right types, but on the CPU


class _At:
    """What _gpu reads of a tensor."""

    def __init__(self, index):
        self.is_cuda, self.device = index is not None, "cpu" if index is None else f"cuda:{index}"
        self.get_device = lambda: index


@pytest.mark.parametrize("at,match", [((0, None, 0), "on cpu"), ((0, 1, 0), "more than one"), ((1, 1, 1), None)])
def test_tensors_on_one_gpu(at, match):
    ts = [_At(i) for i in at]
    if match is None:
        return q4._gpu(None, *ts)
    with pytest.raises(ValueError, match=match):
        q4._gpu(*ts, None)


@pytest.mark.parametrize("bad,err,match", [
    ({"w": lambda t: t.to(torch.int64)}, TypeError, "mats.1.: dtype"),
    ({"w": lambda t: t.t().contiguous().t()}, ValueError, "mats.1.: not contiguous"),
    ({"w": lambda t: t[0]}, ValueError, "2-D"),
    ({"w": lambda t: t[:, :7]}, ValueError, "not contiguous"),
    ({"sc": lambda t: t.repeat(1, 2)[:, :3]}, ValueError, "scale groups"),
    ({"sc": lambda t: t[:, :0]}, ValueError, "scale groups"),
    ({"sc": lambda t: t.float()}, TypeError, "mats.1. scales: dtype"),
    ({"sc": lambda t: t[:3]}, ValueError, "mats.1. scales: shape"),
    ({"b": lambda t: t[:, :1]}, ValueError, "mats.1. biases: shape"),
    ({"b": lambda t: t.t().contiguous().t()}, ValueError, "mats.1. biases: not contiguous"),
    ({"b": lambda t: t.flatten()}, ValueError, "mats.1. biases: shape"),
    ({"sc": lambda t: t.repeat(1, 2), "b": lambda t: t.repeat(1, 2)}, ValueError, "differ in n_in or group size")],
    ids=lambda v: str(v) if isinstance(v, str) else None)
def test_every_matrix_of_a_call_is_checked(bad, err, match):
    def mat(change=None):
        t = {"w": torch.zeros(6, 16, dtype=torch.int32), "sc": torch.zeros(6, 2, dtype=torch.float16),
             "b": torch.zeros(6, 2, dtype=torch.int16)}
        for k, f in (change or {}).items():
            t[k] = f(t[k])
        return t["w"], t["sc"], t["b"]
    assert q4._same_in([mat(), mat()]) == [(6, 128, 64)] * 2
    with pytest.raises(err, match=match):
        q4._same_in([mat(), mat(bad)])
