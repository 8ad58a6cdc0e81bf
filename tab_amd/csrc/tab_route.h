// Which kernel a convolution from fp32 takes, between the library and its PyTorch front end; host code without HIP.
//
// A call that goes to the kernel with the input patch in LDS needs room for its weights behind the packed activation, which only the
// rule that sends it there can tell.  tab_conv2d_workspace_bytes_full() is a bound for every call of the sizes; the front end asks for
// the plan first and allocates what the call uses.  (With the bound, every KxK call's block was up to 1 MB larger than its packed
// activation and came from another place of the caching allocator; the step of ternary ResNet-18 layers, three sets of inputs in turn,
// mean of twelve placements of its tensors: N=36 100.3 -> 99.9 us, N=32 98.1 -> 97.8.)
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace tab {

// A convolution's plan for that kernel: shape < 0 where another kernel takes it, of which `tiled` is the shape if it has been looked
// up (else -1).
struct PatchPlan {
    int shape, kc, npix, lds_bytes, tiled;
    size_t weight_bytes;
};

}  // namespace tab

extern "C" {

// The plan of a call; returns the bytes it needs behind those of tab_conv2d_workspace_bytes or tab_layer_workspace_bytes.  Sizes that
// the call will refuse have the plan of no kernel and need none.
size_t tab_internal_conv_plan(int type, int padding1, int padding2, int stride1, int stride2, int N, int H, int W, int C, int KN, int KH, int KW,
                              tab::PatchPlan *plan);
// tab_conv2d and tab_layer_conv2d by a plan of the same sizes.
int tab_internal_conv2d(const float *dev_X, const int64_t *dev_QW, const float *dev_ths, const int32_t *dev_btn, int type, int padding1,
                        int padding2, int stride1, int stride2, int N, int H, int W, int C, int KN, int KH, int KW, float *dev_Y,
                        void *workspace, size_t workspace_bytes, const tab::PatchPlan *plan, void *stream);
int tab_internal_layer_conv2d(const float *dev_X, int nchw, float act_scale, const int64_t *dev_QW, const int32_t *dev_btn, int type,
                              int padding1, int padding2, int stride1, int stride2, int N, int H, int W, int C, int KN, int KH, int KW,
                              float *dev_Y, void *workspace, size_t workspace_bytes, const tab::PatchPlan *plan, void *stream);

}  // extern "C"
