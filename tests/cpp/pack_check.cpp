// Test infrastructure: packs a store's words as the device does (pack_child of walk_packed.h). The store
// fills its allocation, so that with the address sanitizer a read past it ends the program.
// Usage: pack_check nodes.bin out.bin
#define __device__
#define __host__
#define __forceinline__ inline
#define __restrict__
#include "walk_packed.h"

#include <cstdio>
#include <cstdlib>
#include <memory>

int main(int argc, char** argv)
{
    FILE* f = argc == 3 ? std::fopen(argv[1], "rb") : nullptr;
    if (!f) return 2;
    std::fseek(f, 0, SEEK_END);
    const size_t words = size_t(std::ftell(f)) / 4;
    std::fseek(f, 0, SEEK_SET);
    const std::unique_ptr<uint32_t[]> nodes(new uint32_t[words]), packed(new uint32_t[words]);
    const bool read = std::fread(nodes.get(), 4, words, f) == words;
    std::fclose(f);
    if (!read) return 3;
    for (size_t i = 0; i < words; i++) packed[i] = cqxd::pack_child(nodes.get(), words / 8, nodes[i]);
    f = std::fopen(argv[2], "wb");
    if (!f) return 4;
    const bool written = std::fwrite(packed.get(), 4, words, f) == words;
    return std::fclose(f) == 0 && written ? 0 : 5;
}
