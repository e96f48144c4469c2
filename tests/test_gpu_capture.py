"""Calls recorded into HIP graphs: on a stream that has no scratch memory yet, and replayed after its scratch has grown."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _buffers(*shapes):
    generator = torch.Generator(device="cuda").manual_seed(7)
    return [torch.randn(*shape, generator=generator, device="cuda") for shape in shapes]


def _gemm(hip, m, n, k):
    a, b, c = _buffers((m, k), (k, n), (m, n))
    return a, c, lambda stream: hip.gemm_bias_act_f32_dev(m, n, k, 0, a.data_ptr(), b.data_ptr(), None, None, c.data_ptr(), stream=stream)


def _conv(hip, batch, c_in, side, c_out):
    x, w, y = _buffers((batch, c_in, side, side), (c_out, c_in, 3, 3), (batch, c_out, side, side))
    return x, y, lambda stream: hip.conv2d_bias_act_f32_dev(batch, c_in, side, side, c_out, (3, 3), (1, 1), (1, 1), (1, 1), 0, x.data_ptr(),
                                                            w.data_ptr(), None, y.data_ptr(), stream=stream)


def _attention(hip, contexts, seq, biased):
    q, k, v, out, zb, ab = _buffers(*[(contexts, seq, 64)] * 4, (contexts, seq), (contexts, seq, seq))
    return v, out, lambda stream: hip.attention_f32_dev(contexts, seq, 64, 0.125, False, q.data_ptr(), k.data_ptr(), v.data_ptr(),
                                                        zb.data_ptr() if biased else None, ab.data_ptr() if biased else None,
                                                        out.data_ptr(), stream=stream)


# a product whose k is split over workgroups (both scratch buffers), one that is not, a convolution, attention whose keys
# are split over workgroups, with biases on rows of no multiple of four and without
CALLS = {"gemm_split_k": (_gemm, (300, 700, 2100)), "gemm": (_gemm, (1233, 1000, 700)), "conv": (_conv, (32, 64, 28, 128)),
         "attention_biased": (_attention, (1, 777, True)), "attention": (_attention, (2, 1025, False))}
LARGER = {_gemm: (600, 1400, 4200), _conv: (32, 128, 56, 128), _attention: (1, 1999, True)}


def _capture(call):
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        call(torch.cuda.current_stream().cuda_stream)
    return graph, stream


@pytest.mark.parametrize("name", CALLS)
def test_replays_match_eager_calls(hip, name):
    """Recorded before the stream has any scratch; then a larger call grows it.  Every replay reads the operands anew."""
    make, sizes = CALLS[name]
    operand, out, call = make(hip, *sizes)
    graph, stream = _capture(call)
    _, _, larger = make(hip, *LARGER[make])
    handle = stream.cuda_stream
    try:
        for replay in range(4):
            operand.mul_(-0.5)
            call(None)
            want = out.clone()
            out.fill_(7.5)
            torch.cuda.synchronize()
            with torch.cuda.stream(stream):
                graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want), replay
            larger(handle)  # grows the stream's scratch: the buffers in the graph have to stay
            torch.cuda.synchronize()
    finally:
        del graph
        hip.release_scratch(handle)
        hip.release_scratch(None)
