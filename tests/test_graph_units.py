"""Graph(optimize=True) fuses a BN(+Add)+ReLU chain only when the chain's values and the batch
norm's running statistics are private to it (the reference's
tests/test_bn_activation_fusion.py:71-77): a BN output that another node also reads, or running
statistics that a second BN shares, leave the chain unfused. Graph building only: runs on the CPU."""

import torch

import myflows_amd as mf
from myflows_amd import device, fused, native
from myflows_amd.resnet import BatchNorm2d


def test_shared_bn_outputs_and_reused_running_statistics_are_not_fused():
    previous = device.get_device()
    device.set_device("cpu")
    try:
        x = mf.Variable(torch.ones((2, 3, 3, 3)), trainable=True)
        layer = BatchNorm2d(3)
        bn = layer(x)
        assert not mf.Graph(mf.Add(mf.ReLU(bn), bn), optimize=True)._bn_groups
        assert not mf.Graph(mf.Add(mf.ReLU(bn), mf.ReLU(layer(x))), optimize=True)._bn_groups
        # A private chain is fused.
        assert len(mf.Graph(mf.ReLU(BatchNorm2d(3)(x)), optimize=True)._bn_groups) == 1
    finally:
        device.set_device(previous)


def test_materialize_intermediates_drops_the_fused_units_from_the_plan():
    previous = device.get_device()
    device.set_device("cpu")
    try:
        x = mf.Variable(torch.ones((2, 3, 3, 3)), trainable=True)
        relu = mf.ReLU(BatchNorm2d(3)(x))
        graph = mf.Graph(relu, optimize=True)
        assert graph._plan().groups
        graph.materialize_intermediates()
        assert not graph._plan().groups
        graph.materialize_intermediates(False)
        assert graph._plan().groups
    finally:
        device.set_device(previous)


def test_the_split_loss_keeps_its_scratch_as_long_as_the_loss(monkeypatch):
    """The sums of the loss's workgroups must not go back to the allocator while a launch on another
    stream (native.launch_stream) still uses them: they are part of the returned tensor's storage."""
    calls = []
    library = type("Library", (), {"mfh_mse_loss_workspace": staticmethod(lambda count: 32 if count > 32768 else 0)})
    monkeypatch.setattr(fused, "_f32", lambda tensor, name: tensor)
    monkeypatch.setattr(native, "_library", lambda: library)
    monkeypatch.setattr(native, "_stream", lambda: 0)
    monkeypatch.setattr(native, "_call", lambda *args: calls.append(args))
    for count in (32768, 256000):
        pred = torch.zeros(count)
        loss = fused.mse_loss_forward(pred, pred)
        assert loss.shape == () and loss.dtype == torch.float32 and loss.is_contiguous()
        symbol, *args = calls[-1]
        assert args[2] == loss.data_ptr() and args[3] == count
        if count == 32768:
            assert symbol == "mfh_mse_loss"
            continue
        scratch, doubles = args[4], args[5]
        storage = loss.untyped_storage()
        assert symbol == "mfh_mse_loss_split" and doubles == 32 and scratch % 8 == 0
        assert loss.data_ptr() + 4 <= scratch and scratch + 8 * doubles <= storage.data_ptr() + storage.nbytes()
