"""The frequency table that a bf16 module keeps: one per configuration and device, and safe to ask for from several threads.
(No device needed.)"""
import sys

import torch

from nsa_ref.module.rope import RopeConfig, RotaryEmbedding, _inv_freq


def test_table_follows_configuration_and_device():
    rope = RotaryEmbedding(RopeConfig(head_dim=64)).to(torch.bfloat16)
    cpu = torch.device("cpu")
    t = rope.table(cpu)
    assert t.dtype == torch.float32 and torch.equal(t, _inv_freq(rope.config)) and rope.table(cpu) is t
    assert rope.table(torch.device("meta")).device.type == "meta"
    rope.config.rope_theta = 10000
    assert torch.equal(rope.table(cpu), _inv_freq(rope.config))


def test_another_caller_between_any_two_lines():
    """A second caller, with another configuration each time, comes in before every line of the first one's call (a trace
    function stands in for its thread: that is where threads are switched)."""
    rope = RotaryEmbedding(RopeConfig(head_dim=64, rope_theta=10000)).to(torch.bfloat16)
    cpu, want = torch.device("cpu"), _inv_freq(rope.config)
    visits = []

    def tracer(frame, event, arg):
        if frame.f_code is not RotaryEmbedding.table.__code__:
            return None
        if event == "line":
            rope.config.rope_theta = 20000 + len(visits)
            visits.append(torch.equal(rope.table(cpu), _inv_freq(rope.config)))
            rope.config.rope_theta = 10000
        return tracer

    before = sys.gettrace()
    sys.settrace(tracer)
    try:
        got = rope.table(cpu)
    finally:
        sys.settrace(before)
    assert torch.equal(got, want) and len(visits) > 3 and all(visits)
