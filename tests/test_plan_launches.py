"""Where a compiled program's 16-bit products have their K in parts, which takes a launch more: not where that is the eighth launch
of an execution.  Read from the memory plan, in which the parts have a slot; no GPU is needed."""
import pytest

from tests.test_arena_host import plan_of, sess  # noqa: F401


def program(n_ops, K, et="bf16"):
    """n_ops elementwise operations in front of a product [128,K] x [K,768]."""
    x, w, y = f"tensor<128x{K}x{et}>", f"tensor<{K}x768x{et}>", f"tensor<128x768x{et}>"
    lines, prev = [], "%x"
    for i in range(n_ops):
        lines.append(f"    %v{i} = stablehlo.{'tanh' if i % 2 == 0 else 'exponential'} {prev} : {x}")
        prev = f"%v{i}"
    lines.append(f"    %y = stablehlo.dot_general {prev}, %w, contracting_dims = [1] x [0] : ({x}, {w}) -> {y}")
    return f"func.func @main(%x: {x}, %w: {w}) -> {y} {{\n" + "\n".join(lines) + f"\n    return %y : {y}\n}}"


@pytest.mark.parametrize("n_ops,K,parts", [(1, 3072, True), (5, 3072, True),     # seven launches with the parts
                                           (6, 3072, False),                     # eight, seven without
                                           (7, 3072, True),                      # eight already
                                           (6, 8192, True)])                     # what a long K gains is more than the line costs
def test_parts_of_a_16_bit_product(sess, n_ops, K, parts):  # noqa: F811
    for et in ("bf16", "f16"):
        assert plan_of(sess, program(n_ops, K, et))["slots"] == n_ops + 1 + parts


def test_fp32_products_keep_their_parts(sess):  # noqa: F811
    assert plan_of(sess, program(6, 4096, "f32"))["slots"] == 8
