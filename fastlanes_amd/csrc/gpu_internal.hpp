// gpu_internal.hpp -- shared host-side pieces of the HIP layer.
#pragma once
#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "format.hpp"

namespace fls {

int fail(int code, const std::string& msg);
int hip_fail(hipError_t e, const char* what);

// Device-side FSST symbol table (include/fls/cor/prm/fsst/fsst.h:92-98 without the version/terminator fields).
struct FsstTableDev {
    uint64_t symbol[256];
    uint64_t packed[256];  // kind 0 (symbols of at most 3 bytes): symbol, 8 len above bit 32; 1 (at most 7): symbol, len
                           // above bit 56; 2: symbol
    uint8_t  len[256];
    uint32_t kind;
};

struct StringPlan {
    FsstTableDev* d_tables = nullptr;  // one per page entry
    void*         d_segs   = nullptr;  // FsstSeg of every segment (k_fsst.hip)
    uint64_t*     d_vecs   = nullptr;  // every vector's decoded bytes, then the sums before each
    uint32_t*     d_ends   = nullptr;  // every string's end within its segment
    uint16_t*     d_sizes  = nullptr;  // decoded bytes of every 32 compressed bytes (k_fsst.hip)
    uint32_t*     d_err    = nullptr;  // error bits: capacity
    uint64_t      n_vec    = 0;
};

int  strings_prepare(const Column& col, const uint8_t* host, StringPlan& sp);
void strings_release(StringPlan& sp);
int  strings_offsets(const Column& col, StringPlan& sp, const uint8_t* dev_enc, uint64_t* dev_offsets, hipStream_t s);
int  strings_check(StringPlan& sp, hipStream_t s);
int  strings_decode(const Column& col, StringPlan& sp, const uint8_t* dev_enc, const uint64_t* dev_offsets,
                    uint8_t* dev_bytes, uint64_t cap, hipStream_t s);
int  strings_decode_all(const Column& col, StringPlan& sp, const uint8_t* dev_enc, uint64_t* dev_offsets,
                        uint8_t* dev_bytes, uint64_t cap, hipStream_t s);

}  // namespace fls
