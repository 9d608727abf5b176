"""exactinfer_amd — MI355X (gfx950) Qwen3 attention hot path: QK-norm + RoPE, KV append,
split-K decode and fp32-exact causal prefill on bf16 matrix cores behind the C ABI of include/ei_attn.h."""

__version__ = "0.1.0"
