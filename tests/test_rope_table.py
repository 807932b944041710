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


def test_another_thread_between_any_two_lines():
    """A second caller with another device comes in before every line of the first one's call (a trace function stands in
    for it: that is where a thread can be switched)."""
    cpu, meta = torch.device("cpu"), torch.device("meta")
    for first in (cpu, meta):
        rope = RotaryEmbedding(RopeConfig(head_dim=64)).to(torch.bfloat16)
        if first is meta:
            rope.table(cpu)
        visits = []

        def tracer(frame, event, arg):
            if frame.f_code is not RotaryEmbedding.table.__code__:
                return None
            if event == "line":
                visits.append(rope.table(meta if first is cpu else cpu).device)
            return tracer

        before = sys.gettrace()
        sys.settrace(tracer)
        try:
            got = rope.table(first)
        finally:
            sys.settrace(before)
        assert got.device == first and len(visits) > 3 and first not in visits
