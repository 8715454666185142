"""Few images from bytes (csrc/crb_dataprep.hip: a workgroup an image): the bits of the kernel that takes many."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C,H,W", [(3, 32, 32), (1, 28, 28), (1, 64, 64), (4, 32, 32), (2, 2, 2), (3, 6, 10), (4, 30, 34), (3, 1, 4)])
@pytest.mark.parametrize("images", [1, 3, 256])
def test_few_images_as_among_many(dev, images, C, H, W):
    import torch
    from crusaderbackend_amd import capi

    src = torch.randint(0, 256, (300, C, H, W), dtype=torch.uint8, device=dev)
    many, few = torch.empty(300, C, H, W, device=dev), torch.full((images + 1, C, H, W), 7.0, device=dev)
    capi.images_from_bytes(src, many, 300, C, H, W, capi.NORM_DISTRIBUTION, 0.5, 2.0)
    capi.images_from_bytes(src, few, images, C, H, W, capi.NORM_DISTRIBUTION, 0.5, 2.0)
    torch.cuda.synchronize()
    assert torch.equal(few[:images], many[:images]) and bool((few[images] == 7).all())
