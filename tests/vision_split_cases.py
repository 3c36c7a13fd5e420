"""The split product's tiles as the tower uses them: (kind, tile, rows, columns, parts), kinds f32 (QKV,
fc2, attn_out and ffn_down unsplit), tanh (ffn_up), erf (fc1), part (attn_out and ffn_down with K
split).  test_host_tables.py checks that no call of the tower runs a pair of kind and tile that is
missing here, test_gpu_vision_split.py runs each."""
CASES = [
    ("f32", 0, 2372, 3456, 1), ("f32", 1, 4612, 3456, 1), ("f32", 2, 1156, 3456, 1), ("f32", 3, 580, 3456, 1),
    ("f32", 4, 452, 3456, 1), ("f32", 5, 132, 3456, 1), ("f32", 6, 4, 3456, 1), ("f32", 6, 65, 4096, 1),
    ("tanh", 0, 1924, 4304, 1), ("tanh", 1, 3844, 4304, 1), ("tanh", 2, 964, 4304, 1), ("tanh", 3, 484, 4304, 1),
    ("tanh", 4, 356, 4304, 1), ("tanh", 5, 100, 4304, 1), ("tanh", 6, 4, 4304, 1), ("tanh", 6, 452, 4304, 1),
    ("erf", 0, 1793, 4608, 1), ("erf", 1, 3585, 4608, 1), ("erf", 2, 897, 4608, 1), ("erf", 3, 449, 4608, 1),
    ("erf", 4, 321, 4608, 1), ("erf", 5, 97, 4608, 1), ("erf", 6, 1, 4608, 1),
    ("part", 0, 2308, 1152, 5), ("part", 1, 4356, 1152, 3), ("part", 2, 1796, 1152, 2), ("part", 3, 324, 1152, 8),
    ("part", 4, 228, 1152, 7), ("part", 5, 68, 1152, 7), ("part", 6, 4, 1152, 8), ("part", 6, 260, 1152, 3),
]


def padded(parts):
    """A padded K for PARTS parts whose shares are uneven where there are more than one."""
    return 192 if parts == 1 else 192 * parts + 64
