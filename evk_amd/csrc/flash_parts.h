// How the flash backward of head sizes 32, 64 and 128 splits dK/dV: key
// blocks, and row parts of the flattened query rows within one.  Plain C++, so
// that the rules can be checked without a GPU.
#pragma once
#include <cstddef>
#include <cstdint>

#ifdef __HIPCC__
#define EVK_HOST_DEVICE __host__ __device__
#else
#define EVK_HOST_DEVICE
#endif

namespace evkhip {

constexpr int BKB = 128;       // keys per workgroup (4 waves x 32)
constexpr int BRC = 32;        // flattened query rows per chunk

// Chunks of flattened rows that key block kb of a batch interacts with.
EVK_HOST_DEVICE inline int bwd_kv_chunks(int kb, int N, int H, bool causal) {
    const int64_t r_lo = causal ? (int64_t)kb * BKB * H : 0;
    return (int)(((int64_t)N * H - r_lo + BRC - 1) / BRC);
}
EVK_HOST_DEVICE inline int bwd_kv_parts(int kb, int N, int H, bool causal, int part_log2) {
    return (bwd_kv_chunks(kb, N, H, causal) + (1 << part_log2) - 1) >> part_log2;
}

// Chunks per row part, as a power of two: as long as leaves about 128 parts
// (fewer fp32 partials to write and read) and short enough that a small call
// still spreads over the chip.  Head sizes up to 64 stop at 16: two workgroups
// share a CU there, and longer parts lengthen the launch.  Forward and
// backward, us with this rule and with parts of 16 throughout: Dh 128, B=2
// N=2000 H=8 163 and 177, B=16 N=160 H=4 27.5 and 40.1, B=1 N=130 H=2 22.3
// and 26.6; Dh 64, B=1 N=600 H=4 24.5 and 33.7, B=16 N=160 H=4 20.9 and 32.3;
// Dh 32, B=1 N=888 H=1 19.9 and 27.7.
// A part's partials are 1 KB times the head size, and with parts of a fixed
// length their number grows with N^2 H (34 GB at Dh 128, B=1 N=65536 H=16).
// More than a dozen parts for each CU balance nothing, so from BWD_PARTS on
// they get longer instead (2048 to 4095 of them; B=2 N=16384 H=8 causal,
// backward alone, 64 chunks -> 256: 5578 -> 5293 us, Dh 64 16 -> 128: 2889 ->
// 2351).  From BWD_BLOCKS key blocks on (four for each CU) each is one part,
// heavy ones first over all batches (flash_bwd_kvq), and nothing is summed:
// B=64 N=2048 H=8 causal 3434 -> 3194 us, B=32 N=4096 6301 -> 5820.
constexpr int BWD_PARTS = 4096, BWD_BLOCKS = 1024;
inline int bwd_part_log2(int dh, int64_t blocks, int64_t chunks, int64_t longest) {
    const int most = dh <= 64 ? 4 : 6;
    int l = 2;
    while (l < most && (chunks >> (l + 1)) >= 96) ++l;
    while ((blocks >= BWD_BLOCKS || (chunks >> l) >= BWD_PARTS) && ((int64_t)1 << l) < longest) ++l;
    return l;
}

struct BwdKvPlan {
    int part_log2;  // chunks per row part
    int per_batch;  // parts of a batch
    size_t bytes;   // fp32 partials: one slot for every part, none where every key block is one part
};
inline BwdKvPlan bwd_kv_plan(int dh, int B, int N, int H, bool causal) {
    const int nkb = (N + BKB - 1) / BKB;
    int64_t chunks = 0;
    for (int kb = 0; kb < nkb; ++kb) chunks += bwd_kv_chunks(kb, N, H, causal);
    BwdKvPlan p{bwd_part_log2(dh, (int64_t)nkb * B, chunks * B, bwd_kv_chunks(0, N, H, causal)), 0, 0};
    for (int kb = 0; kb < nkb; ++kb) p.per_batch += bwd_kv_parts(kb, N, H, causal, p.part_log2);
    if (p.per_batch > nkb) p.bytes = (size_t)B * p.per_batch * 4 * (2 * 2 * (dh / 16)) * 64 * 16;
    return p;
}

}  // namespace evkhip
