"""One programmed layer read on several streams and from several threads: every output is that
of reads one after another."""

import copy
import threading

import pytest
import torch
from torch import nn

from memfast_amd import Config, Nonidealities, Simulator, convert_model
from memfast_amd.nn import AnalogLinear

pytestmark = pytest.mark.gpu

WRITE = Nonidealities(write_variation=0.02)
CONFIGS = {
    "default": Config(nonidealities=WRITE),
    "rows128": Config(array_size=(128, 128), adc_bits=8, nonidealities=WRITE),
    "sliced": Config(input_slice=(1, 1, 2, 2, 2), weight_slice=(1, 1, 2, 2, 2),
                     array_size=(128, 128), rows_per_read=32, adc_bits=7, nonidealities=WRITE),
}


def layer_of(name, device, k=4096, o=512):
    torch.manual_seed(3)
    source = nn.Linear(k, o).to(device)
    layer = AnalogLinear(source, Simulator(CONFIGS[name], device=device), name="layer")
    return layer.set_input_scale(0.03)


@pytest.mark.parametrize("name", list(CONFIGS))
def test_reads_on_two_streams_share_the_terms(hip_device, name):
    """A fixed-scale read returns before it has run: the next read, on another stream, uses the
    terms that the first one samples, and neither sees the other's split totals."""
    gen = torch.Generator().manual_seed(4)
    inputs = [torch.randn(64, 4096, generator=gen).to(hip_device) for _ in range(4)]
    serial = layer_of(name, hip_device)
    expected = [serial(x) for x in inputs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(hip_device) for _ in inputs]
    for _ in range(3):
        layer = layer_of(name, hip_device)
        torch.cuda.synchronize()
        outputs = []
        for x, stream in zip(inputs, streams):
            with torch.cuda.stream(stream):
                outputs.append(layer(x))
        torch.cuda.synchronize()
        for got, want in zip(outputs, expected):
            assert torch.equal(got.view(torch.int32), want.view(torch.int32))


def test_reprogramming_between_streams(hip_device):
    """New weights are sampled while another stream still reads the old terms."""
    x = torch.randn(64, 4096, generator=torch.Generator().manual_seed(5)).to(hip_device)
    other = torch.randn(4096, 512, generator=torch.Generator().manual_seed(6)).to(hip_device)
    layer = layer_of("default", hip_device)
    before = layer(x)
    layer.update_weight(other)
    after = layer(x)
    layer = layer_of("default", hip_device)
    torch.cuda.synchronize()
    side = torch.cuda.Stream(hip_device)
    got = [layer(x)]
    with torch.cuda.stream(side):
        got.append(layer(x))
    # Codes and scales are the program's own: its user orders writes to them.
    torch.cuda.current_stream(hip_device).wait_stream(side)
    layer.update_weight(other)
    got.append(layer(x))
    torch.cuda.synchronize()
    for output, want in zip(got, (before, before, after)):
        assert torch.equal(output.view(torch.int32), want.view(torch.int32))


def test_codes_built_on_another_stream(hip_device):
    """A loaded program's kernel copy of the codes is made by its first read."""
    x = torch.randn(33, 4096, generator=torch.Generator().manual_seed(7)).to(hip_device)
    layer = layer_of("default", hip_device)
    expected = layer(x)
    loaded = layer_of("default", hip_device)
    loaded.load_state_dict(layer.state_dict())
    loaded.reset_read()
    torch.cuda.synchronize()
    outputs = []
    for stream in [torch.cuda.Stream(hip_device) for _ in range(2)]:
        with torch.cuda.stream(stream):
            outputs.append(loaded(x))
    torch.cuda.synchronize()
    for got in outputs:
        assert torch.equal(got.view(torch.int32), expected.view(torch.int32))


@pytest.mark.parametrize("own_stream", [False, True])
def test_threads_read_one_layer(hip_device, own_stream):
    gen = torch.Generator().manual_seed(8)
    inputs = [torch.randn(64, 1024, generator=gen).to(hip_device) for _ in range(4)]
    layer = layer_of("default", hip_device, k=1024, o=256).set_input_scale(None)
    expected = [layer(x) for x in inputs]
    layer = layer_of("default", hip_device, k=1024, o=256).set_input_scale(None)
    torch.cuda.synchronize()
    results = {}

    def work(index):
        stream = torch.cuda.Stream(hip_device) if own_stream else torch.cuda.default_stream(hip_device)
        with torch.cuda.stream(stream):
            results[index] = [layer(inputs[index]) for _ in range(8)]
        stream.synchronize()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(inputs))]
    for thread in threads:
        thread.start()
    for thread in threads:
        thread.join()
    for index, want in enumerate(expected):
        assert len(results[index]) == 8
        for got in results[index]:
            assert torch.equal(got.view(torch.int32), want.view(torch.int32))


def test_copies_and_threads_have_their_own_status_words(hip_device):
    """Fixed-scale reads return on a pinned word: a copied model's is its own and pinned, and two
    threads' reads of one simulator do not see each other's bits."""
    layer = layer_of("default", hip_device, k=256, o=64)
    x = torch.randn(40, 256, generator=torch.Generator().manual_seed(9)).to(hip_device)
    expected = layer(x)
    product = layer.simulator.mm(x, x.T.contiguous())
    clone = copy.deepcopy(layer)
    assert torch.equal(clone(x).view(torch.int32), expected.view(torch.int32))
    assert clone.simulator.mm(x, x.T.contiguous()).shape == product.shape
    bad = x.clone()
    bad[39, 255] = float("nan")
    wrong = []

    def work(value, raises):
        torch.cuda.set_device(hip_device)
        for _ in range(200):
            try:
                layer(value)
                raised = False
            except ValueError:
                raised = True
            if raised != raises:
                wrong.append(raises)

    threads = [threading.Thread(target=work, args=args) for args in ((x, False), (bad, True))]
    for thread in threads:
        thread.start()
    for thread in threads:
        thread.join()
    assert not wrong


def test_recurrent_sequences_on_two_streams(hip_device):
    """The native GRU sequence keeps its hidden program's terms as a layer does."""
    torch.manual_seed(9)
    x = torch.randn(6, 4, 40, device=hip_device)
    source = nn.GRU(40, 128).to(hip_device)
    config = CONFIGS["sliced"]
    expected, _ = convert_model(source, Simulator(config, device=hip_device))(x)
    layer = convert_model(source, Simulator(config, device=hip_device))
    torch.cuda.synchronize()
    outputs = []
    for stream in [torch.cuda.Stream(hip_device) for _ in range(2)]:
        with torch.cuda.stream(stream):
            outputs.append(layer(x)[0])
    torch.cuda.synchronize()
    assert layer.cells[0].hidden._terms_source is not None
    for got in outputs:
        assert torch.equal(got.view(torch.int32), expected.view(torch.int32))
