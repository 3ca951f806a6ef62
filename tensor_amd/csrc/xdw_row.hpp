// What the pointwise + depthwise launch (conv_xdw.hip) requests of an input row: the bytes of its descriptor and the scalar offsets of
// its loads. Plain C++, so that the rule can be gone over without a GPU.
#pragma once

#if defined(__HIPCC__)
#define OHIP_ROW_FN __host__ __device__ __forceinline__
#else
#define OHIP_ROW_FN inline
#endif

namespace ohip {

// from a lane's first input octet to the others of its reduction bytes: + 1, and + 8, + 9 in the second reduction step
struct XdwOctets {
    unsigned o1, o8, o9;
};
// octets: of the input blob; those that it does not have stay at the first one's place (every lane's own offset is beyond the blob there)
OHIP_ROW_FN XdwOctets xdw_octets(unsigned plane_bytes, int octets) {
    return {octets > 1 ? plane_bytes : 0u, octets > 8 ? 8u * plane_bytes : 0u, octets > 9 ? 9u * plane_bytes : 0u};
}

struct XdwRow {
    unsigned bytes, at, at1, at8, at9;
};
// A buffer load is out of range where the lane's offset is not below the descriptor's bytes minus the scalar offset. That difference must
// not wrap: no scalar offset here is beyond the bytes. A row outside the image (`there` is false; `row` may then be any number) has a
// descriptor of no bytes and reads zero at offset 0.
OHIP_ROW_FN XdwRow xdw_row(bool there, unsigned blob_bytes, unsigned row, const XdwOctets& o) {
    return {there ? blob_bytes : 0u, there ? row : 0u, there ? row + o.o1 : 0u, there ? row + o.o8 : 0u, there ? row + o.o9 : 0u};
}

}  // namespace ohip
