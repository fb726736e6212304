// Block -> item order that keeps neighbouring items in one L2: workgroup b of a
// launch runs on XCD b % 8, and XCD x takes the x-th eighth of the items in order.
// Every XCD gets items whatever their number (the shares differ by one at most).
// Shared by the kernels and by a host-side check.
#pragma once

namespace uocr_hip {

constexpr int kXcds = 8;

// first item of XCD x's share of n items (x == kXcds: n)
__host__ __device__ inline int xcd_first_item(int x, int n) { return (int)((long long)n * x / kXcds); }

}  // namespace uocr_hip
