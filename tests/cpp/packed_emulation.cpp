// Test infrastructure: the packed walk (cubiquity_amd/csrc/walk_packed.h) compiled for the host and
// checked against the oracle by tests/test_packed_walk.py before any GPU run.
//   plain  rays for which ray_plain() holds take walk_step_packed, the others (and any ray near its
//          iteration cap) walk_step_packed_any, as the kernels do
//   any    every ray takes walk_step_packed_any
// Prints the number of plain rays. Exits with 6 when the store is not eligible.
// Usage: packed_emulation plain|any nodes.bin sub.bin rays.bin out.bin surf max_footprint max_iters
#define __device__
#define __host__
#define __forceinline__ inline
#define __restrict__
#include "walk_packed.h"

#include <cstdio>
#include <cstdlib>
#include <string_view>
#include <vector>

using namespace cqxd;

static std::vector<char> slurp(const char* path)
{
    std::vector<char> v;
    FILE* f = std::fopen(path, "rb");
    if (!f) return v;
    std::fseek(f, 0, SEEK_END);
    v.resize(size_t(std::ftell(f)));
    std::fseek(f, 0, SEEK_SET);
    if (std::fread(v.data(), 1, v.size(), f) != v.size()) v.clear();
    std::fclose(f);
    return v;
}

int main(int argc, char** argv)
{
    if (argc != 9) return 2;
    const bool any = std::string_view(argv[1]) == "any";
    const std::vector<char> nb = slurp(argv[2]), sb = slurp(argv[3]), rb = slurp(argv[4]);
    if (nb.empty() || sb.size() != 8 * sizeof(cqx_subdag)) return 3;
    const uint32_t* nodes = reinterpret_cast<const uint32_t*>(nb.data());
    const uint64_t count = nb.size() / 32;
    const auto word_of = [&](uint32_t c) {
        uint32_t mask = 0;
        for (uint32_t k = 0; k < 8; k++) mask |= (nodes[uint64_t(c) * 8 + k] ? 1u : 0u) << k;
        return packed_word(c, mask);
    };
    std::vector<uint32_t> packed(count * 8);
    for (uint64_t i = 0; i < count * 8; i++) packed[i] = word_of(nodes[i]);
    cqx_subdag sub[8];
    std::memcpy(sub, sb.data(), sizeof(sub));
    if (!packed_eligible(count, sub)) return 6;
    PackedParams P{};
    uint32_t occ = 0;
    for (int c = 0; c < 8; c++) {
        if (!sub[c].node) continue;
        sub[c].pad0 = word_of(sub[c].node);
        occ |= 1u << c;
        P.top = uint32_t(sub[c].height) > P.top ? uint32_t(sub[c].height) : P.top;
    }
    P.packed = packed.data();
    P.sub = sub;
    P.surf = uint32_t(std::atoi(argv[6]));
    P.max_footprint = float(std::atof(argv[7]));
    P.max_iters = uint32_t(std::strtoul(argv[8], nullptr, 10));
    P.fp_disabled = footprint_is_disabled(P.max_footprint) ? 1u : 0u;
    lod_thresholds(P.max_footprint, P.lod_hi, P.lod_lo);
    const bool lod = !(P.lod_hi == INFINITY);
    const float* rays = reinterpret_cast<const float*>(rb.data());
    const uint64_t n = rb.size() / 24;
    std::vector<cqx_hit> out(n);
    std::vector<char> stack(33 * kRowBytes);
    const uint32_t base = stack_base(0u, P.top);
    uint64_t plain = 0;
    for (uint64_t i = 0; i < n; i++) {
        PackedRay S{};
        const float* r = rays + 6 * i;
        ray_setup_packed(S, r[0], r[1], r[2], r[3], r[4], r[5]);
        const bool fast = !any && S.plain;
        plain += fast;
        while (!is_finished(S.phase)) {
            enter_octants_packed(sub, P, S, stack.data(), base, occ);
            while (S.phase == kWalk) {
                if (fast && P.max_iters >= 2 && S.iters <= P.max_iters - 2) {
                    if (lod) walk_step_packed<true>(P, S, stack.data(), base);
                    else walk_step_packed<false>(P, S, stack.data(), base);
                } else {
                    walk_step_packed_any(P, S, stack.data(), base);
                }
            }
        }
        emit_packed(P, S, out[i]);
    }
    std::printf("%llu\n", (unsigned long long)plain);
    FILE* f = std::fopen(argv[5], "wb");
    if (!f) return 4;
    const size_t w = std::fwrite(out.data(), sizeof(cqx_hit), n, f);
    std::fclose(f);
    return w == n ? 0 : 5;
}
