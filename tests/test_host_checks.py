"""Host-side argument checks of the tensor-level calls (CPU only): the
one-expression checks refuse what the single ones refuse, with the same errors."""

import pytest
import torch

from mla_kv_quant_amd import kernels, writer


@pytest.mark.parametrize("bad,error,text", [
    (None, TypeError, "must be a tensor"),
    ([1, 2], TypeError, "must be a tensor"),
    (torch.zeros(4, dtype=torch.int32), TypeError, "must be torch.int64"),
    (torch.zeros(4, dtype=torch.int64, device="meta"), ValueError, "must be on cpu"),
    (torch.zeros(2, 2, dtype=torch.int64), ValueError, "must have 1 dims"),
    (torch.zeros(8, dtype=torch.int64)[::2], ValueError, "must be contiguous"),
])
def test_need_all_refuses_with_the_single_checks_errors(bad, error, text):
    good = torch.zeros(4, dtype=torch.int64)
    dev = torch.device("cpu")
    kernels._need_all(dev, ((good, "a", torch.int64, 1), (good.view(2, 2), "b", torch.int64, 2)))
    with pytest.raises(error, match=text):
        kernels._need_all(dev, ((good, "a", torch.int64, 1), (bad, "b", torch.int64, 1)))


def test_rows_and_indices_take_every_shape_that_flattens():
    x = torch.arange(24.).view(3, 1, 8)
    assert torch.equal(writer._rows(x, 8), x.reshape(3, 8))
    assert torch.equal(writer._rows(x.view(3, 8), 4), x.reshape(6, 4))
    y = torch.arange(48.).view(3, 16)[:, :8]
    assert writer._rows(y, 8) is y  # strided rows stay views
    i = torch.arange(6, dtype=torch.int32).view(2, 3)
    assert torch.equal(writer._as_int64(i), torch.arange(6))
    assert torch.equal(writer._as_int64(torch.arange(8)[::2]), torch.tensor([0, 2, 4, 6]))
    assert writer._as_int64(torch.arange(8)[::2]).is_contiguous()


def _assemble_args():
    D, R = 512, 64
    return {"slots": torch.ones(3, dtype=torch.int64), "codes": torch.zeros(8, D // 4, dtype=torch.uint8),
            "params": torch.zeros(8, D // 128, 2), "rope_buf": torch.zeros(8, R, dtype=torch.bfloat16),
            "hp_c": torch.zeros(21, D, dtype=torch.bfloat16), "row_of_slot": torch.zeros(8, dtype=torch.int32),
            "owner_of_row": torch.zeros(21, dtype=torch.int32), "rotation": None,
            "out": torch.zeros(3, D + R, dtype=torch.bfloat16)}


@pytest.mark.parametrize("name", ["params", "hp_c", "row_of_slot", "owner_of_row"])
@pytest.mark.parametrize("bad", [None, [1, 2]])
def test_assemble_rows_names_an_argument_that_is_no_tensor(name, bad):
    with pytest.raises(TypeError, match=f"{name} must be a tensor"):
        kernels.assemble_rows(**dict(_assemble_args(), **{name: bad}))


@pytest.mark.parametrize("name", ["loc", "seq_lens", "req_idx"])
def test_writer_names_the_index_of_the_wrong_length(name):
    D, R, n = 512, 64, 3
    a = {"latent": torch.zeros(n, D, dtype=torch.bfloat16), "k_pe": torch.zeros(n, R, dtype=torch.bfloat16),
         "rotation_t": None, "positions": None, **{k: torch.ones(n, dtype=torch.int64) for k in ("loc", "seq_lens", "req_idx")},
         **{k: v for k, v in _assemble_args().items() if k not in ("slots", "rotation", "out")},
         "P": 4, "W": 16, "max_reqs": 1, "threshold": 0.98, "gain": 1.16}
    a[name] = a[name][:2]
    with pytest.raises(ValueError, match=f"^{name} must have 3 entries"):
        kernels.write_rows(**a)
