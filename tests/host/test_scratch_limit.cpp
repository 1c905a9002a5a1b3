// Products on a device that has no memory left for their partial results.  The library's hipMalloc is this program's: it asks
// the runtime for more than any device has wherever a limit set here is exceeded, so that the runtime fails the allocation, and
// remembers that it did, as on a full device.
#include "weed_hip.h"

#include <cstddef>
#include <cstdint>
#include <cstdio>
#include <dlfcn.h>
#include <vector>

namespace {
size_t g_limit = SIZE_MAX;
unsigned g_refused = 0;
int failures = 0;
} // namespace

extern "C" __attribute__((visibility("default"))) int hipMalloc(void **ptr, size_t bytes)
{
    static const auto real = reinterpret_cast<int (*)(void **, size_t)>(dlsym(RTLD_NEXT, "hipMalloc"));
    if (bytes > g_limit) {
        ++g_refused;
        return real(ptr, (size_t)1 << 60);
    }
    return real(ptr, bytes);
}

#define REQUIRE(cond)                                                                                                  \
    do {                                                                                                               \
        if (!(cond)) {                                                                                                 \
            std::printf("    FAILED %s:%d: %s (last error: %s)\n", __FILE__, __LINE__, #cond, weed_hip_last_error());  \
            ++failures;                                                                                                \
        }                                                                                                              \
    } while (0)

namespace {

// Column-major a (row i: r_i u_k) and b (column j: v_k c_j): every sum is r_i c_j (u . v), a whole number below 2^24.
struct Product {
    uint32_t M, N, K;
    void *a = nullptr, *b = nullptr, *out = nullptr;
    std::vector<float> r, c;
    float dot = 0.0f;

    Product(uint32_t m, uint32_t n, uint32_t k) : M(m), N(n), K(k), r(m), c(n)
    {
        std::vector<float> ha((size_t)M * K), hb((size_t)K * N);
        for (uint32_t i = 0; i < M; ++i) {
            r[i] = (float)(1 + i % 7);
        }
        for (uint32_t j = 0; j < N; ++j) {
            c[j] = (float)((int)(j % 5) - 2);
        }
        for (uint32_t x = 0; x < K; ++x) {
            const float u = (float)(1 + x % 3), v = (float)(1 + x % 11);
            dot += u * v;
            for (uint32_t i = 0; i < M; ++i) {
                ha[(size_t)x * M + i] = r[i] * u;
            }
            for (uint32_t j = 0; j < N; ++j) {
                hb[(size_t)j * K + x] = v * c[j];
            }
        }
        REQUIRE(weed_hip_malloc(&a, ha.size() * sizeof(float)) == WEED_HIP_OK);
        REQUIRE(weed_hip_malloc(&b, hb.size() * sizeof(float)) == WEED_HIP_OK);
        REQUIRE(weed_hip_malloc(&out, (size_t)M * N * sizeof(float)) == WEED_HIP_OK);
        REQUIRE(weed_hip_memcpy_h2d(a, ha.data(), ha.size() * sizeof(float)) == WEED_HIP_OK);
        REQUIRE(weed_hip_memcpy_h2d(b, hb.data(), hb.size() * sizeof(float)) == WEED_HIP_OK);
    }
    int run()
    {
        return weed_hip_matmul_f32(M, N, K, static_cast<float *>(a), 0, 1, M, static_cast<float *>(b), 0, 1, K,
                                   static_cast<float *>(out), 0, 1, M);
    }
    bool right()
    {
        std::vector<float> got((size_t)M * N, -1.0f);
        if (weed_hip_memcpy_d2h(got.data(), out, got.size() * sizeof(float)) != WEED_HIP_OK) {
            return false;
        }
        for (uint32_t j = 0; j < N; ++j) {
            for (uint32_t i = 0; i < M; ++i) {
                if (got[(size_t)j * M + i] != r[i] * c[j] * dot) {
                    return false;
                }
            }
        }
        return true;
    }
};

} // namespace

int main()
{
    REQUIRE(weed_hip_init(0) == WEED_HIP_OK);
    if (failures) {
        return 1;
    }
    Product large(512, 512, 4096), larger(1024, 2048, 8192), small(256, 384, 2048), whole(1024, 1024, 128);

    // no scratch at all: large products of few tiles have whole sums, smaller ones say so, and neither is held against the next call
    g_limit = 0;
    REQUIRE(large.run() == WEED_HIP_OK);
    REQUIRE(g_refused == 1); // (it is a product that asks for scratch)
    REQUIRE(large.right());
    REQUIRE(small.run() == WEED_HIP_ENOMEM);
    REQUIRE(g_refused == 2);
    REQUIRE(whole.run() == WEED_HIP_OK);
    REQUIRE(whole.right());

    // scratch for the smaller ones: it is still there after a larger one was refused
    g_limit = SIZE_MAX;
    REQUIRE(small.run() == WEED_HIP_OK);
    REQUIRE(small.right());
    g_limit = (size_t)256 * 384 * 32 * sizeof(float); // (32 ranges of 64 k at most; the larger one takes 4 of 1024 x 2048 at least)
    REQUIRE(larger.run() == WEED_HIP_OK);
    REQUIRE(g_refused == 3);
    REQUIRE(larger.right());
    g_limit = 0;
    REQUIRE(small.run() == WEED_HIP_OK);
    REQUIRE(small.right());
    REQUIRE(g_refused == 3);

    // and with memory again, as ever
    g_limit = SIZE_MAX;
    REQUIRE(larger.run() == WEED_HIP_OK);
    REQUIRE(larger.right());
    REQUIRE(weed_hip_shutdown() == WEED_HIP_OK);
    std::printf("%d failed\n", failures);
    return failures != 0;
}
