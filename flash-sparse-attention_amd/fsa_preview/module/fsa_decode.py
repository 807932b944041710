"""One decode step of the whole layer under the reference's name (fsa_preview/module/fsa_decode.py:12-199): same
constructor, parameter names (state_dict-compatible with `FlashSparseAttention`) and forward arguments.

x [1, hidden] is the new token of ONE request; k_cache / v_cache hold the un-rotated k / v projections of the L
tokens before it, cmp_k_cache / cmp_v_cache the un-rotated compressed rows.  As in the reference the caches are
rotated inside every call (they are stored un-rotated) and are not modified; with `return_new_rows=True` the rows
to append come back beside the output.

Default semantics: the output equals what `FlashSparseAttention` computes for this token at the end of the same
sequence.  `as_written=True` keeps the reference's literal behaviour where it differs (query rotated for position 0,
:137; compression fed from the compressed cache, :100-121; decode block-score conventions; key-0-only selected
branch).
"""
import torch

from fsa_hip import ops as _ops
from fsa_preview.module.fsa_decode_kernel import decode_step_attention
from nsa_ref.module.rope import RopeConfig, RotaryEmbedding


class FlashSparseAttentionDecode(torch.nn.Module):
    def __init__(
        self,
        hidden_size: int,
        num_q_heads: int,
        num_kv_heads: int,
        head_dim: int,
        kernel_size: int,
        kernel_stride: int,
        block_size: int,
        topk: int,
        init_blocks: int,
        local_blocks: int,
        window_size: int,
        rope_config: RopeConfig,
    ):
        super().__init__()
        self.hidden_size = hidden_size
        self.num_q_heads = num_q_heads
        self.num_kv_heads = num_kv_heads
        self.head_dim = head_dim
        self.kernel_size = kernel_size
        self.kernel_stride = kernel_stride
        self.block_size = block_size
        self.topk = topk
        self.init_blocks = init_blocks
        self.local_blocks = local_blocks
        self.window_size = window_size
        self.rope_config = rope_config

        self.proj_q = torch.nn.Linear(self.hidden_size, self.num_q_heads * self.head_dim, bias=False)
        self.proj_k = torch.nn.Linear(self.hidden_size, self.num_kv_heads * self.head_dim, bias=False)
        self.proj_v = torch.nn.Linear(self.hidden_size, self.num_kv_heads * self.head_dim, bias=False)
        self.proj_o = torch.nn.Linear(self.num_q_heads * self.head_dim, self.hidden_size, bias=False)

        self.compress_key = torch.nn.Parameter(
            torch.zeros(self.num_kv_heads, self.head_dim * self.kernel_size, self.head_dim))
        self.compress_value = torch.nn.Parameter(
            torch.zeros(self.num_kv_heads, self.head_dim * self.kernel_size, self.head_dim))
        self.intra_block_pe = torch.nn.Parameter(torch.zeros(self.num_kv_heads, self.kernel_size, self.head_dim))
        self.gate = torch.nn.Sequential(torch.nn.Linear(self.hidden_size, 3, bias=False), torch.nn.Sigmoid())
        self.rope = RotaryEmbedding(self.rope_config)

    def _fused_step(self, x, *caches):
        """The step as one native call (four launches, caches neither copied nor rotated), or None where it does not
        apply: projections that are more than a plain Linear, tensor subclasses, head dims or layouts without kernels, no
        compressed key."""
        gate = self.gate
        layers = (self.proj_q, self.proj_k, self.proj_v, gate[0], self.proj_o)
        if (any(c is None for c in caches) or torch.is_autocast_enabled() or not all(map(_ops.is_plain_linear, layers))
                or not _ops.is_plain(gate, torch.nn.Sequential) or len(gate) != 2
                or not _ops.is_plain(gate[1], torch.nn.Sigmoid) or not _ops.is_plain(self.rope, RotaryEmbedding)
                or not _ops.are_plain_tensors(x, *caches, self.compress_key, self.compress_value, self.intra_block_pe)):
            return None
        return _ops.decode_layer(x, caches, [m.weight for m in layers], self.compress_key, self.compress_value,
                                 self.intra_block_pe, self.rope.table(x.device), self.rope.attention_scaling,
                                 (self.num_q_heads, self.num_kv_heads, self.head_dim, self.kernel_size,
                                  self.kernel_stride, self.block_size, self.topk, self.init_blocks, self.local_blocks,
                                  self.window_size))

    @torch.no_grad()
    def forward(
        self,
        x: torch.Tensor,  # [1, hidden_size]
        cu_seqlens_q: torch.Tensor,
        cu_seqlens_k: torch.Tensor,  # [2]: the cache with the new token
        k_cache: torch.Tensor = None,
        v_cache: torch.Tensor = None,
        cmp_k_cache: torch.Tensor = None,
        cmp_v_cache: torch.Tensor = None,
        as_written: bool = False,
        return_new_rows: bool = False,
    ):
        assert x.dtype == torch.bfloat16 or x.dtype == torch.float16
        assert x.shape[-1] == self.hidden_size
        assert x.shape[0] == 1, "one request, one new token per call, as in the reference"
        out = None if as_written else self._fused_step(x, k_cache, v_cache, cmp_k_cache, cmp_v_cache)
        if out is not None:
            return (out[0], out[1:]) if return_new_rows else out[0]
        cu_seqlens_q = cu_seqlens_q.to(torch.int32)
        cu_seqlens_k = cu_seqlens_k.to(torch.int32)
        q = self.proj_q(x).view(x.shape[0], self.num_q_heads, self.head_dim)
        k_new = self.proj_k(x).view(x.shape[0], self.num_kv_heads, self.head_dim)
        v_new = self.proj_v(x).view(x.shape[0], self.num_kv_heads, self.head_dim)
        k = torch.cat([k_cache, k_new], dim=0)
        v = torch.cat([v_cache, v_new], dim=0)
        cmp_out, sel_out, win_out, new_c = decode_step_attention(
            self, q, k, v, k_new, v_new, cmp_k_cache, cmp_v_cache, k, cu_seqlens_q, cu_seqlens_k,
            lambda t, cu, start, stride: self.rope(t, cu, start=start, stride=stride), as_written)
        gate = self.gate(x)
        attn_output = _ops.gate_merge_fwd(cmp_out.reshape(1, -1), sel_out.reshape(1, -1), win_out.reshape(1, -1),
                                          gate.contiguous())
        attn_output = self.proj_o(attn_output)
        if return_new_rows:
            return attn_output, (k_new, v_new) + tuple(new_c)
        return attn_output
