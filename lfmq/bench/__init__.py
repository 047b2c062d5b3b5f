"""Benchmark harnesses: decode tok/s + delta-ppl."""
from .decode import bench_decode, build_quantized_llama
from .ppl import bench_ppl
