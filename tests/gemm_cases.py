"""Calls whose GEMMs run the 256-row kernel (csrc/gemm_mfma.hip) in each of its
forms.  test_gemm_plan.py asserts on the CPU that the plan sends them there;
test_gpu_gemm_mfma.py and others run them."""

# (dtype, rows, dim, hidden, gate/up, down) of one expert, top-1: for each GEMM
# the parts its last tiles are split into along K (1: none; padded widths never are).
ONE_EXPERT = [
    ("f32", 8150, 1024, 256, 4, 2),
    ("bf16", 6100, 1280, 512, 2, 2),
    ("f16", 6100, 1280, 512, 2, 2),
    ("f32", 9000, 1024, 512, 1, 1),
    ("bf16", 9000, 1024, 512, 1, 1),
    # neither width is a whole tile
    ("f32", 8111, 1064, 500, 1, 1),
    ("bf16", 8111, 456, 500, 1, 1),
    ("f16", 8111, 456, 500, 1, 1),
]

# (dtype, rows, dim, experts, top_k, hidden): both GEMMs
EXPERTS = [
    ("bf16", 6001, 520, 4, 2, 700),
    ("f32", 6001, 1064, 4, 2, 500),
]

# dense feed-forwards: (dtype, rows, dim, hidden, gate/up, down), as above
DENSE = [
    ("f32", 9000, 1024, 512, 1, 1),
    ("f32", 9000, 1024, 1024, 4, 1),
    ("f32", 24000, 1024, 2048, 1, 2),
    ("f32", 8111, 1064, 500, 1, 1),
    ("f32", 9000, 1000, 2667, 1, 1),
]
