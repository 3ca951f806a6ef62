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

// The pixels of a channel octet that a tile of consecutive output pixels reads where input and output have the same sides and stride 1: one
// run of the batch's pixels (those of another image in it are outside the windows, as are the neighbouring rows' at either end of a row). They
// are copied in pairs, a pair from one image: where an image has an odd count, a place is left free behind it.
struct DwPwStage {
    unsigned pitch;            // places of 8 bytes of an octet: `slots` pixels and zeros behind them; 0: nothing is staged
    unsigned slots, before;    // the window of a tile's first pixel begins `before` places in front of it; the run begins there, or one earlier
    unsigned image;            // places of an image
    unsigned units, lg_lanes;  // pairs of places of an octet, log2 of the lanes that an octet takes of a copy
    unsigned octets;           // room for them: whole copies
    unsigned image_m, image_s; // (division by image)
};
// where the run of a tile begins, its first pixel the `pixel`-th of the batch, in image `image`; where the window of pixel `pix` of an image begins
OHIP_DWPW_FN int dwpw_run(const DwPwStage& st, unsigned HW, unsigned pixel, unsigned image) { return (int)(pixel + image * (st.image - HW) - st.before) & ~1; }
OHIP_DWPW_FN int dwpw_window(const DwPwStage& st, unsigned image, unsigned pix) { return (int)(image * st.image + pix - st.before); }
// the byte of the blob that the pair at place `at` of an image begins with, octet `oct` of C8 (behind an odd image's last pixel: anything)
OHIP_DWPW_FN unsigned dwpw_copied(const DwPwStage& st, unsigned HW, unsigned C8, unsigned image, unsigned oct, unsigned at) {
    return ((image * C8 + oct) * HW + at - image * st.image) * 8u;
}
inline DwPwStage dwpw_stage(int C, int H, int W, int ks, int ph, int pw, int dh, int dw, int pixels) {
    DwPwStage st{};
    const unsigned HW = (unsigned)(H * W), span = (unsigned)(pixels + (ks - 1) * (dh * W + dw)), C8 = (unsigned)C / 8;
    st.image = HW + HW % 2, st.before = (unsigned)(ph * W + pw);
    const unsigned free_places = HW % 2 ? ((unsigned)pixels + HW - 2) / HW : 0;  // (images that begin in the tile)
    st.slots = (1 + span + free_places + 1) / 2 * 2;
    st.units = st.slots / 2 + 1;
    while (st.lg_lanes < 6 && 1u << st.lg_lanes < st.units) ++st.lg_lanes;
    const unsigned sets = 64u >> st.lg_lanes;
    st.pitch = st.units > 64 ? 2 * st.units : 2u << st.lg_lanes;
    st.octets = ((C8 + 1) / 2 * 2 + sets - 1) / sets * sets;
    return st;
}

}  // namespace ohip
