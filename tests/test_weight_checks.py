"""The weight structs' checks on the host: every call checks the tensors it is given, and a wrong one is refused with its
name, whatever was accepted before."""
import dataclasses

import pytest
import torch

import gfr_moe

E, D, N, BITS = 3, 256, 512, 3


class OnGpu(torch.Tensor):
    """A CPU tensor that says it lives on the GPU (the checks look at is_cuda and device only)."""

    @property
    def is_cuda(self):
        return True

    @property
    def device(self):
        return torch.device("cuda")


def gpu(*shape, dtype):
    return torch.zeros(shape, dtype=dtype).as_subclass(OnGpu)


def experts():
    i32, f16 = torch.int32, torch.float16
    return gfr_moe.Exl3Experts(
        gt=gpu(E, D // 16, N // 16, 8 * BITS, dtype=i32), ut=gpu(E, D // 16, N // 16, 8 * BITS, dtype=i32),
        dt=gpu(E, N // 16, D // 16, 8 * BITS, dtype=i32), suh_g=gpu(E, D, dtype=f16), suh_u=gpu(E, D, dtype=f16),
        suh_d=gpu(E, N, dtype=f16), svh_g=gpu(E, N, dtype=f16), svh_u=gpu(E, N, dtype=f16), svh_d=gpu(E, D, dtype=f16),
        bits=BITS)


def fp8(copies):
    bf, u8 = torch.bfloat16, torch.uint8
    return gfr_moe.Fp8SharedWeights(
        gu=gpu(2 * N, D, dtype=u8), gu_scale=gpu(2 * N, dtype=bf), down=gpu(D, N, dtype=u8), down_scale=gpu(D, dtype=bf),
        gu_bf16=gpu(2 * N, D, dtype=bf) if copies else None, down_bf16=gpu(D, N, dtype=bf) if copies else None)


def test_good_weights_give_their_pointers():
    w = experts()
    st = w.struct()
    assert (st.experts, st.hidden, st.inter, st.bits) == (E, D, N, BITS)
    for name in ("gt", "ut", "dt", "suh_g", "suh_u", "suh_d", "svh_g", "svh_u", "svh_d"):
        assert getattr(st, name) == getattr(w, name).data_ptr(), name
    for copies in (False, True):
        f = fp8(copies)
        st = f.struct()
        assert (st.hidden, st.inter, st.gu, st.down_scale) == (D, N, f.gu.data_ptr(), f.down_scale.data_ptr())
        assert (st.gu_bf16 or 0) == (f.gu_bf16.data_ptr() if copies else 0)


@pytest.mark.parametrize("name", ["gt", "ut", "dt", "suh_g", "suh_u", "suh_d", "svh_g", "svh_u", "svh_d"])
@pytest.mark.parametrize("fault", ["dtype", "shape", "stride", "cpu"])
def test_each_expert_tensor_is_checked(name, fault):
    w = experts()
    w.struct()
    _spoil_and_refuse(w, name, fault)


@pytest.mark.parametrize("name", ["gu", "gu_scale", "down", "down_scale", "gu_bf16", "down_bf16"])
@pytest.mark.parametrize("fault", ["dtype", "shape", "stride", "cpu"])
def test_each_fp8_tensor_is_checked(name, fault):
    w = fp8(True)
    w.struct()
    _spoil_and_refuse(w, name, fault)


@pytest.mark.parametrize("name", ["gu_bf16", "down_bf16"])
def test_one_bf16_copy_alone_is_refused(name):
    _spoil_and_refuse(fp8(True), name, "missing")


def _spoil_and_refuse(w, name, fault):
    t = getattr(w, name)
    if fault == "missing":
        bad = None
    elif fault == "dtype":
        bad = gpu(*t.shape, dtype=torch.float32)
    elif fault == "shape":
        bad = gpu(*t.shape[:-1], t.shape[-1] + 2, dtype=t.dtype)
    elif fault == "stride":
        bad = gpu(*t.shape[:-1], 2 * t.shape[-1], dtype=t.dtype)[..., ::2]
    else:
        bad = torch.zeros(t.shape, dtype=t.dtype)
    setattr(w, name, bad)
    with pytest.raises(ValueError):
        w.struct()
    with pytest.raises(ValueError):
        dataclasses.replace(w).check()
