"""Shapes of the prefill GEMM tests: the 4B-shaped miniature (8 q heads, 4 kv
heads, head_dim 256) with (hidden, ffn) chosen so that the prefill's choice
of token tile and column splits takes every instance of the GEMM kernels.
tests/test_lifetime.py checks on the CPU which instances they take;
tests/test_gpu_prefill.py runs them."""

# (hidden, ffn): prompt lengths
Q4_0 = {(288, 352): (2, 15, 16, 17, 32, 33, 64, 65, 128, 129, 257),
        (1056, 6944): (17, 65, 129, 257, 385)}
F32 = {(288, 352): (2, 16, 17, 33, 64, 65, 130, 257),
       (544, 3488): (65, 129, 257)}


def cases(shapes):
    return [(h, f, n) for (h, f), ns in shapes.items() for n in ns]
