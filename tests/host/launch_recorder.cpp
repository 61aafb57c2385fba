// Stands in for the HIP runtime under the library's host code: what a call would launch is recorded, nothing runs.  attn_params.inc holds the
// attention kernels' argument block, taken out of the library's source.
#include <cstdint>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "warp34_kv.h"

#include "attn_params.inc"

namespace {
struct Dim {
    uint32_t x, y, z;
};
struct Launch {
    std::string name;
    Dim grid, block;
    AttnParams params;
    int merge_slots;
};
struct Config {
    Dim grid, block;
    size_t smem;
    void* stream;
};
std::map<const void*, std::string>& names() {
    static std::map<const void*, std::string> m;
    return m;
}
std::vector<Launch> launches;
Config config;
alignas(256) char symbol_memory[256];
}  // namespace

extern "C" {
void** __hipRegisterFatBinary(const void*) {
    static void* handle;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* fn, char*, const char* name, unsigned, void*, void*, void*, void*, int*) { names()[fn] = name; }
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim grid, Dim block, size_t smem, void* stream) {
    config = Config{grid, block, smem, stream};
    return 0;
}
int __hipPopCallConfiguration(Dim* grid, Dim* block, size_t* smem, void** stream) {
    *grid = config.grid, *block = config.block, *smem = config.smem, *stream = config.stream;
    return 0;
}
int hipLaunchKernel(const void* fn, Dim grid, Dim block, void** args, size_t, void*) {
    Launch l{names()[fn], grid, block, {}, 0};
    const auto is = [&](const char* part) { return l.name.find(part) != std::string::npos; };
    if (is("paged_attn_") || is("paged_prefill_")) memcpy(&l.params, args[0], sizeof(AttnParams));
    if (is("split_merge_")) memcpy(&l.merge_slots, args[2], sizeof(int));
    launches.push_back(l);
    return 0;
}
int hipGetLastError() { return 0; }
int hipGetDevice(int* d) {
    *d = 0;
    return 0;
}
int hipFuncSetAttribute(const void*, int, int) { return 0; }
int hipFuncGetAttributes(void* attr, const void*) {
    memset(attr, 0, 56);  // hipFuncAttributes
    return 0;
}
int hipGetSymbolAddress(void** p, const void*) {
    *p = symbol_memory;
    return 0;
}

void rec_clear() { launches.clear(); }
int rec_count() { return (int)launches.size(); }
const char* rec_name(int i) { return launches[i].name.c_str(); }
void rec_shape(int i, uint32_t* out) {
    const Launch& l = launches[i];
    out[0] = l.grid.x, out[1] = l.grid.y, out[2] = l.grid.z, out[3] = l.block.x, out[4] = (uint32_t)l.merge_slots;
}
void rec_choice(int i, int* out) {
    const AttnParams& p = launches[i].params;
    out[0] = p.max_chunks, out[1] = p.grid_chunks, out[2] = p.short_units, out[3] = p.short_tiles, out[4] = p.short_tok_tile, out[5] = p.q_subgroups;
}
}
