// Host check of the Q8_0 GEMM (gemm.hip, launch_q8_gemm) compiled for the CPU (hip/hip_runtime.h,
// emu.h) under AddressSanitizer, every buffer of exactly the size that the callers allocate: rows
// padded to 32 in the Q8_TILED order, not padded in natural order. No access may leave a buffer, the
// outputs are those of a float64 product, and both orders give the same bits. Test infrastructure
// only.
//
//   gemm_check n k m tile_rows
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "common.h"
#include "layer.h"

namespace gsvk {
static std::string g_err;
void set_error(const char * fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_err = buf;
}
const char * get_error() { return g_err.c_str(); }
}  // namespace gsvk

using namespace gsvk;

template <typename T>
static T * buf(size_t n) { return (T *) std::calloc(n, sizeof(T)); }

int main(int argc, char ** argv) {
    if (argc < 5) return 2;
    const int n = std::atoi(argv[1]), k = std::atoi(argv[2]), m = std::atoi(argv[3]), tile_rows = std::atoi(argv[4]);
    const int nb = k / 32, mp = (m + 31) / 32 * 32;
    std::mt19937 rng(n + k + m);
    auto scale = [&] {
        const _Float16 h = (_Float16) (0.01f + (rng() % 1024) / 65536.0f);
        uint16_t u;
        std::memcpy(&u, &h, 2);
        return u;
    };
    int8_t * wq = buf<int8_t>((size_t) n * k), * xq = buf<int8_t>((size_t) m * k);
    uint16_t * wd = buf<uint16_t>((size_t) n * nb);
    float * xd = buf<float>((size_t) m * nb), * bias = buf<float>(n);
    for (size_t i = 0; i < (size_t) n * k; i++) wq[i] = (int8_t) ((int) (rng() % 255) - 127);
    for (size_t i = 0; i < (size_t) m * k; i++) xq[i] = (int8_t) ((int) (rng() % 255) - 127);
    for (size_t i = 0; i < (size_t) n * nb; i++) wd[i] = scale();
    for (size_t i = 0; i < (size_t) m * nb; i++) xd[i] = h2f(scale());
    for (int i = 0; i < n; i++) bias[i] = (rng() % 2001) / 1000.0f - 1.0f;
    // the same in the Q8_TILED order, rows padded to 32
    int8_t * wt = buf<int8_t>((size_t) n * k), * xt = buf<int8_t>((size_t) mp * k);
    uint16_t * wdt = buf<uint16_t>((size_t) n * nb);
    float * xdt = buf<float>((size_t) mp * nb);
    for (int r = 0; r < n; r++)
        for (int b = 0; b < nb; b++) {
            for (int c = 0; c < 32; c++) wt[q8_tiled_offset(r, nb, b, c)] = wq[(size_t) r * k + 32 * b + c];
            wdt[q8_tiled_scale(r, nb, b)] = wd[(size_t) r * nb + b];
        }
    for (int r = 0; r < m; r++)
        for (int b = 0; b < nb; b++) {
            for (int c = 0; c < 32; c++) xt[q8_tiled_offset(r, nb, b, c)] = xq[(size_t) r * k + 32 * b + c];
            xdt[q8_tiled_scale(r, nb, b)] = xd[(size_t) r * nb + b];
        }
    float * y = buf<float>((size_t) m * n), * yt = buf<float>((size_t) m * n);
    LayerOut out{};
    out.y_stride = n;
    out.n_store = n;
    out.bias = bias;
    out.act = 1;
    Q8Weights w{}, tw{};
    w.qn = wq; w.dn = wd;
    tw.qt = wt; tw.dt = wdt;
    out.y = y;
    if (launch_q8_gemm(w, n, k, m, xq, xd, Q8_NATURAL, out, nullptr, m > 256 ? 0 : tile_rows)) {
        std::fprintf(stderr, "%s\n", get_error());
        return 1;
    }
    out.y = yt;
    if (launch_q8_gemm(tw, n, k, m, xt, xdt, Q8_TILED, out, nullptr, tile_rows)) {
        std::fprintf(stderr, "%s\n", get_error());
        return 1;
    }
    double err = 0, top = 0;
    for (int r = 0; r < m; r++)
        for (int c = 0; c < n; c++) {
            double s = bias[c];
            for (int b = 0; b < nb; b++) {
                int i = 0;
                for (int j = 0; j < 32; j++) i += (int) xq[(size_t) r * k + 32 * b + j] * wq[(size_t) c * k + 32 * b + j];
                s += (double) i * xd[(size_t) r * nb + b] * h2f(wd[(size_t) c * nb + b]);
            }
            s = s > 0 ? s : 0;
            err = std::max({err, std::fabs(y[(size_t) r * n + c] - s), std::fabs(yt[(size_t) r * n + c] - s)});
            top = std::max(top, s);
        }
    // (the order of sums is the kernel's: above 256 rows the natural operands take another one)
    const bool same = m > 256 || std::memcmp(y, yt, sizeof(float) * m * n) == 0;
    std::printf("n %d k %d m %d: %.1e of the largest output, %s\n", n, k, m, err / top, same ? "equal to the bit" : "bits differ");
    return err <= 2e-6 * top && same ? 0 : 1;
}
