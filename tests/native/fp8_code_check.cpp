// Host-only check of the append's fast e4m3 quantiser (fp8_code in append_body.h)
// against fp8_quantize's steps (kernels.metal:564-601) over every finite positive
// half scale and every half value.  Built and run by tests/test_fp8_quantiser.py
// (no kernel launches); argv: first scale, scale step.
#include <cmath>
#include <cstdio>
#include <cstdlib>

#include "../../pagedattentionmetal_amd/csrc/kernels/append_body.h"

using namespace pam;

static float half_of(uint32_t b) { return (float)__builtin_bit_cast(f16, (uint16_t)b); }

// the reference's steps in float, as pam_device.h's fp8_quantize has them
static uint32_t slow(float value, float scale) {
    float v = value / scale;
    v = fminf(fmaxf(v, -448.0f), 448.0f);
    const uint32_t sign = v < 0.0f ? 0x80u : 0u;
    v = fabsf(v);
    if (v == 0.0f) return 0u;
    if (v < 0x1p-6f) {
        int mi = (int)roundf(v * 512.0f);
        return sign | (uint32_t)(mi > 7 ? 7 : mi);
    }
    int ex;
    float mant = frexpf(v, &ex) * 2.0f;
    ex -= 1;
    if (ex > 8) return sign | 0x7Eu;
    int eb = ex + 7, mi = (int)roundf((mant - 1.0f) * 8.0f);
    if (mi > 7) mi = 0, eb++;
    if (eb > 15) return sign | 0x7Eu;
    if (eb == 15 && mi > 6) mi = 6;
    return sign | ((uint32_t)eb << 3) | (uint32_t)mi;
}

int main(int argc, char **argv) {
    const uint32_t s0 = argc > 1 ? atoi(argv[1]) : 1, ds = argc > 2 ? atoi(argv[2]) : 1;
    float value[65536];
    for (uint32_t v = 0; v < 65536; v++) value[v] = half_of(v);
    for (uint32_t sb = s0; sb < 0x7C00u; sb += ds) {
        const float s = half_of(sb), inv = (1.0f / s) * (1.0f + 0x1p-20f);
        for (uint32_t v = 0; v < 65536; v++) {
            const uint32_t a = fp8_code(value[v], inv), b = slow(value[v], s);
            if (a != b) {
                printf("value %04x scale %04x: %02x, not %02x\n", v, sb, a, b);
                return 1;
            }
        }
    }
    printf("ok\n");
    return 0;
}
