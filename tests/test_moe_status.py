"""What moe_forward does with the statuses of the one-call block, without a GPU: a stand-in for the library
returns them."""
import pytest

torch = pytest.importorskip("torch")

from loken_amd import lib, moe


class Stub:
    def __init__(self, status):
        self.status, self.calls = status, []

    def __getattr__(self, name):
        def call(*args):
            self.calls.append(name)
            return self.status if name == "lk_moe_forward" else 0
        return call


def forward(monkeypatch, status):
    stub = Stub(status)
    monkeypatch.setattr(moe._lib, "load", lambda: stub)
    monkeypatch.setattr(moe, "_stream", lambda: 0)
    block = torch.zeros(16, dtype=torch.uint8)
    x, choices, w = torch.zeros(2, 256), torch.zeros(2, 2, dtype=torch.int32), torch.zeros(2, 2)
    moe.moe_forward(lib.TYPE_Q4_K, lib.TYPE_Q4_K, x, block, block, block, choices, w, 4, 256)
    return stub.calls


@pytest.mark.parametrize("status", [lib.LK_ERR_TYPE, lib.LK_ERR_ARG, lib.LK_ERR_NOMEM])
def test_a_call_the_block_does_not_take_goes_on_launch_by_launch(monkeypatch, status):
    calls = forward(monkeypatch, status)
    assert calls[0] == "lk_moe_forward" and "loken_moe_gemm_gguf_down_reduce" in calls


@pytest.mark.parametrize("status", [lib.LK_ERR_LAUNCH, lib.LK_ERR_SIZE, -99])
def test_a_launch_that_failed_is_reported(monkeypatch, status):
    with pytest.raises(lib.LokenError):
        forward(monkeypatch, status)


def test_the_block_served_in_one_call_is_the_only_call(monkeypatch):
    assert forward(monkeypatch, lib.LK_OK) == ["lk_moe_forward"]
