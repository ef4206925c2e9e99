// The scalar formulas of vbd_scalar.h on the CPU; driven by test_scalar_formulas.py.
#include "../newton_amd/csrc/vbd_scalar.h"

// out[i]: whether the screen clears block i, its determinant and squared norm in single precision in the kernels' order
extern "C" void screen(int n, const float* blocks, int* out) {
    for (int i = 0; i < n; ++i) {
        const float* h = blocks + 9 * i;
        const float cx = h[4] * h[8] - h[5] * h[7], cy = h[5] * h[6] - h[3] * h[8], cz = h[3] * h[7] - h[4] * h[6];
        const float det = h[0] * cx + h[1] * cy + h[2] * cz;
        float n1 = 0.0f;
        for (int k = 0; k < 9; ++k) n1 += h[k] * h[k];
        out[i] = vbd_scalar::certainly_well_conditioned(det, 1.0f / sqrtf(n1)) ? 1 : 0;
    }
}

extern "C" void sigmoid(int n, const float* z, float* out) {
    for (int i = 0; i < n; ++i) out[i] = vbd_scalar::sigmoid_short(z[i]);
}
