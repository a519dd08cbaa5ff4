"""CPU checks of the drop-in block's choice of launch (digital_twin_brain_amd/block.py)
on a stand-in for the native block: which calls ask for the persistent launch
(deliver mode 3), what happens when it is refused, and how weight changes and
large blocks put it off."""
import numpy as np
import pytest

from digital_twin_brain_amd import _native as nat
from digital_twin_brain_amd import block as block_class


class FakeNative:
    def __init__(self, n, nnz, refuse=None):
        self.n, self.nnz, self.refuse = n, nnz, refuse
        self.mode, self.asked = 0, []

    def get_launch(self):
        return dict(deliver_mode=self.mode)

    def set_launch(self, deliver_mode):
        self.asked.append(deliver_mode)
        if deliver_mode == 3 and self.refuse is not None:
            raise nat.DTBError(self.refuse, "refused")
        self.mode = deliver_mode

    def set_weights(self, *a):
        pass


def _block(n, per, refuse=None, src=None):
    b = object.__new__(block_class)
    b.N, b.src = n, src
    b._nb = FakeNative(n, n * per, refuse)
    b._choose_launch()
    return b


@pytest.mark.parametrize("n,per,steps,mode", [
    (1999, 20, 20, 0), (2000, 20, 20, 3), (2000, 100, 20, 3), (2000, 101, 20, 0), (2000, 1000, 20, 0),
    (6000, 300, 20, 3), (6000, 400, 20, 0), (9_999, 1000, 20, 0), (10_000, 400, 20, 3),
    (32_768, 100, 20, 3), (32_769, 100, 20, 0),
    # short calls: at the ends of the range the per-step kernels are the faster ones
    (2000, 20, 1, 0), (2000, 20, 7, 0), (2000, 20, 8, 3), (9_999, 400, 1, 0), (10_000, 100, 1, 3), (10_000, 99, 1, 0),
    (16_384, 100, 1, 3), (16_385, 100, 1, 0), (32_768, 122, 1, 0), (16_384, 20, 8, 3), (16_385, 20, 15, 0),
    (16_385, 20, 16, 3),
])
def test_calls_that_take_the_persistent_launch(n, per, steps, mode):
    b = _block(n, per)
    b._set_mode(steps)
    assert b._nb.mode == mode and b._mode == (2 if mode == 3 else 0)


def test_injected_uniforms_and_sources_keep_the_per_step_kernels():
    b = _block(4000, 20)
    b._set_mode(20)
    assert b._nb.mode == 3
    b._set_mode(1, persist=False)
    assert b._nb.mode == 0
    b = _block(4000, 20, src=np.zeros((1, 1)))
    b._set_mode(1000)
    assert b._nb.asked == []


def test_large_blocks_run_some_steps_before_they_pay_for_the_copy():
    """20 steps of a new block of 32,768 x 1,000 synapses are no reason to build the copy."""
    b = _block(32_768, 1000)
    for _ in range(10):
        b._set_mode(20)
        assert b._nb.asked == []
    b._set_mode(20)
    assert b._nb.mode == 3
    b._set_mode(1)
    assert b._nb.mode == 3


def test_a_weight_change_puts_the_launch_off():
    b = _block(4000, 20)
    b._set_mode(20)
    assert b._nb.mode == 3
    b.w_uij = type("W", (), dict(is_sparse=True))()
    b.update_conn_weight(([0], [1], [2]), [0.5])
    assert b._nb.mode == 0
    for steps in (40, 900, 59, 1):
        b._set_mode(steps)
        assert b._nb.mode == 0
    b._set_mode(40)
    assert b._nb.mode == 3


@pytest.mark.parametrize("code", [nat.DTB_INVALID_PARAMETER, nat.DTB_OUT_OF_MEMORY])
def test_a_block_that_does_not_fit_goes_on_with_the_per_step_kernels(code):
    b = _block(10_000, 400, refuse=code)
    for _ in range(3):
        b._set_mode(20)
        assert b._nb.mode == 0 and b._mode == 0
    assert b._nb.asked == [3]  # not tried again


def test_other_errors_are_raised():
    b = _block(10_000, 400, refuse=nat.DTB_RUNTIME_ERROR)
    with pytest.raises(nat.DTBError):
        b._set_mode(20)
