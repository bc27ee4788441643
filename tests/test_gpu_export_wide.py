"""Export of many tiles, which takes 512 threads a tile: whole and ragged last tiles in either direction, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("E,I,H", [(52, 512, 1280), (52, 520, 1032), (60, 456, 1288), (1030, 8, 104), (260, 72, 520)])
def test_export_of_many_tiles(gpu_device, dtype, E, I, H):
    from arctictraining_amd import ops

    print("export", dtype, E, I, H, flush=True)
    g = torch.Generator(device=gpu_device).manual_seed(I + H)
    bits = lambda *shape: torch.randint(-32768, 32768, shape, dtype=torch.int16, device=gpu_device, generator=g)
    gate_up = bits(E, H, 2 * I)
    gate, up = ops.remap_unpack(gate_up.view(dtype), two=True)
    assert torch.equal(gate.view(torch.int16), gate_up[:, :, 0::2].transpose(1, 2))
    assert torch.equal(up.view(torch.int16), gate_up[:, :, 1::2].transpose(1, 2))
    down = bits(E, H, I)
    out = ops.remap_unpack(down.view(dtype), two=False)
    assert torch.equal(out.view(torch.int16), down.transpose(1, 2))
