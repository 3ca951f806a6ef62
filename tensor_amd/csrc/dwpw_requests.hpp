// What the launch of a depthwise layer and the pointwise layers behind it (conv_dwpw.hip) requests of blobs and weights that may not be
// there: the bytes of their descriptors and the scalar offsets of its accesses. Plain C++, so that the rule can be gone over without a GPU.
#pragma once

#if defined(__HIPCC__)
#define OHIP_DWPW_FN __host__ __device__ __forceinline__
#else
#define OHIP_DWPW_FN inline
#endif

namespace ohip {

// A buffer access is out of range where the lane's offset is not below the descriptor's bytes minus the scalar offset. That difference must
// not wrap: no scalar offset here is beyond the bytes.

// Step `step` of the `steps` reduction steps of row tiles 2 pair, 2 pair + 1 (mt tiles a step, 1024 bytes each). A step that does not exist is
// asked for at the weights' very end, where every lane is out of range.
OHIP_DWPW_FN unsigned dwpw_weights_at(int step, int steps, int mt, int pair) {
    return step < steps ? ((unsigned)step * (unsigned)mt + 2u * (unsigned)pair) * 1024u : (unsigned)steps * (unsigned)mt * 1024u;
}

// An fp32 blob of `bytes` bytes of which a lane reads or writes two elements of four channels for a pair of row tiles, `half` bytes apart, and
// 128 HW bytes further for the next pair. One that is not there has a descriptor of no bytes: what is read of it is zero, what is written dropped.
struct DwPwFloats {
    unsigned bytes, pair, half;
    OHIP_DWPW_FN unsigned at(int pr, int h) const { return (unsigned)pr * pair + (unsigned)h * half; }
};
OHIP_DWPW_FN DwPwFloats dwpw_floats(bool there, unsigned bytes, unsigned HW, unsigned half) {
    return {there ? bytes : 0u, there ? 128u * HW : 0u, there ? half : 0u};
}

}  // namespace ohip
