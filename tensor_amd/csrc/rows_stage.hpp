// What the launch on staged rows (conv_rows.hip) requests of the input octets of a stage: who asks for which of them, and the scalar
// offsets of its loads. Plain C++, so that the rules can be gone over without a GPU.
#pragma once

#if defined(__HIPCC__)
#define OHIP_ROWS_FN __host__ __device__ __forceinline__
#else
#define OHIP_ROWS_FN inline
#endif

namespace ohip {

// Planes of at most 128 places (pixel pairs) are dealt to a half, a quarter or an eighth of a workgroup's 256 threads each, as many of them
// as hold a plane: 1 << rows_parts_shift parts of the threads take an octet each.
OHIP_ROWS_FN int rows_parts_shift(int places) { return places > 128 ? 0 : places > 64 ? 1 : places > 32 ? 2 : 3; }

// The octets of a stage, `plane` bytes apart, are dealt to `sub` parts of the threads: part p walks p, p + sub, ..., its lanes' own offsets p
// planes ahead. The scalar offsets of part 0 serve all of them. A buffer load is out of range where the lane's offset is not below the
// descriptor's bytes minus the scalar offset, and that difference must not wrap: where the walk asks for octets that the stage does not have
// (beyond the blob in every lane's own offset), the scalar offset stays at the last octet, and may be any number up to there.
struct RowsWalk {
    unsigned at, on, last;
    OHIP_ROWS_FN unsigned next() {
        const unsigned now = at < last ? at : last;
        at += on;  // (wraps where such octets are 4 GB further)
        return now;
    }
};
OHIP_ROWS_FN RowsWalk rows_walk(unsigned plane, int first, int count, int sub) {
    return {(unsigned)first * plane, (unsigned)sub * plane, (unsigned)(first + count - 1) * plane};
}

}  // namespace ohip
