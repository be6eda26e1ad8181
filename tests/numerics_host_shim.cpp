// Host build of csrc/numerics.hpp and csrc/launch_rules.hpp for the CPU tests (g++ -ffp-contract=off): the same text that
// the device and the launchers compile.
#include "../ferrite_amd/csrc/launch_rules.hpp"
extern "C" {
float shim_expf(float x) { return fe::fe_expf(x); }
float shim_sigmoid(float x) { return fe::sigmoid_ref(x); }
float shim_swiglu(float g, float u, float l) { return fe::swiglu_ref(g, u, l); }
unsigned shim_e4m3_encode(float x) { return fe::e4m3_encode(x); }
float shim_e4m3_decode(unsigned b) { return fe::e4m3_decode(b); }
float shim_e2m1_decode(unsigned c) { return fe::e2m1_decode(c); }
float shim_ue8m0_decode(unsigned b) { return fe::ue8m0_decode(b); }
unsigned shim_block_scale_e8m0(float amax) { return fe::block_scale_e8m0(amax); }
void shim_expf_many(const float* x, float* y, long n) { for (long i = 0; i < n; ++i) y[i] = fe::fe_expf(x[i]); }
int shim_max_units(int n, int topk, int n_experts, int shared, int unit_rows) {
    return fe::max_units_for(n, topk, n_experts, shared > 0, unit_rows);
}
// the form that a layer's f32 gate/up (down = 0) and down GEMM take
int shim_f32_split(int n, int hidden, int n_experts, int topk, int inter, int shared, int down) {
    const int units = fe::max_units_for(n, topk, n_experts, shared > 0, 16);
    if (down) return fe::f32_split(n, topk, n_experts, units, hidden, shared > 0 ? hidden : 0, inter, true);
    return fe::f32_split(n, topk, n_experts, units, inter, shared, hidden, false);
}
// split: units and item groups as {routed, shared, groups_r, groups_s}
void shim_stream_raise(int* split, int items_r, int items_s) {
    const fe::StreamSplit s = fe::stream_raise(fe::StreamSplit{split[0], split[1], split[2], split[3]}, items_r, items_s);
    split[2] = s.groups_r;
    split[3] = s.groups_s;
}
unsigned shim_stream_blocks(int several, const int* split) {
    return fe::stream_blocks(several != 0, fe::StreamSplit{split[0], split[1], split[2], split[3]});
}
// how often each of the passes 0 .. total - 1 is gone through; returns the largest number of passes of a block, -1 for one out of range
int shim_stream_cover(int total, int blocks, int* times) {
    int most = 0;
    for (int b = 0; b < blocks; ++b) {
        const fe::StreamShare s = fe::stream_share(total, blocks, b);
        const int count = fe::stream_count(s);
        for (int i = 0; i < count; ++i) {
            const int v = s.first + i * s.step;
            if (v < 0 || v >= total) return -1;
            ++times[v];
        }
        if (count > most) most = count;
    }
    return most;
}
}
