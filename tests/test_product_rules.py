"""Which operands the products of a few rows take to their fused kernels: rules on the host, checked without a GPU."""
import pytest
import torch

from prelude_amd.ops import kernels as K


def tiled(n, k):
    return K.LinearWeight(torch.zeros(n, k, dtype=torch.bfloat16), K.TiledWeight(torch.zeros(1, dtype=torch.bfloat16), n, k))


def view(shape, off, dtype=torch.bfloat16):
    """A contiguous tensor whose first element lies ``off`` elements behind a 16-byte boundary."""
    n = int(torch.Size(shape).numel())
    buf = torch.zeros(n + 16, dtype=dtype)
    skip = (-buf.data_ptr() % 16) // buf.element_size() + off
    return buf[skip: skip + n].view(shape)


@pytest.mark.parametrize("off", [0, 1, 4, 7, 8])
def test_an_activation_rides_in_a_product_of_aligned_rows_alone(off):
    """The kernel reads rows in 16-byte pieces: an aligned tensor is taken (and refused here, for there is no GPU), another
    goes the way of the product and the activation apart."""
    x, w = view((3, 64), off), tiled(32, 64)
    if off % 8 == 0:
        with pytest.raises(K.NativeError):
            K._linear_few_act(x, w, 1)
    else:
        assert K._linear_few_act(x, w, 1) is None


@pytest.mark.parametrize("which", ["rows", "slices", "residual", "gain"])
def test_the_norm_rides_in_a_product_of_aligned_operands_alone(which):
    off = {"rows": 0, "slices": 0, "residual": 0, "gain": 0, which: 1}
    w, gain = tiled(64, 512), view((512,), off["gain"], torch.float32)
    x = K.SliceSums(view((2, 3, 512), off["slices"], torch.float32), torch.bfloat16) if which == "slices" else view((3, 512), off["rows"])
    assert not K.after_norm_few_supported(x, view((3, 512), off["residual"]), w, gain)
    whole = K.SliceSums(view((2, 3, 512), 0, torch.float32), torch.bfloat16) if which == "slices" else view((3, 512), 0)
    assert K.after_norm_few_supported(whole, view((3, 512), 0), w, view((512,), 0, torch.float32))
