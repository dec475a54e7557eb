"""What the tests of the small-tile matmul kernel share: its built shapes and operands whose sums are exact in any order."""
import torch

# blocks per CU, 16-token groups, 16-column groups
SHAPES = [411, 312, 321, 422, 222, 323, 123, 324, 124, 231, 132, 133, 234, 134, 141, 142, 143, 244]


def describe_of(shape):
    """how matmul_describe begins to name a tile of this shape, and what it says of its blocks per CU"""
    blocks, mt, nt = shape // 100, shape // 10 % 10, shape % 10
    return f"{16 * mt}x{16 * nt} x", f" {blocks} per CU,"


def exact_operands(M, N, K, seed, device="cpu"):
    """small integers"""
    g = torch.Generator(device=device).manual_seed(seed)
    a = torch.randint(-2, 3, (M, K), generator=g, device=device).float().to(torch.float8_e4m3fn)
    b = torch.randint(-2, 3, (N, K), generator=g, device=device).float().to(torch.float8_e4m3fn)
    return a, b, g


def exact_scales(M, N, K, kind, g, device="cpu"):
    """powers of two"""
    power = lambda *shape: 2.0 ** torch.randint(-1, 2, shape, generator=g, device=device).float()
    if kind == "block":
        return power(-(-K // 128), -(-M // 4) * 4), power(-(-N // 128), -(-K // 128))
    return power(1, M), power(N, 1)


def exact_case(M, N, K, kind, seed):
    """small integers times powers of two: every sum is exact in any order"""
    a, b, g = exact_operands(M, N, K, seed)
    return a, b, *exact_scales(M, N, K, kind, g)
