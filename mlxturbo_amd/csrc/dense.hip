// Instantiations of the kernels over stream_tile.cuh for one (dtype, bits)
// pair (the wide kernel; 8-bit: the thin grouped kernel), compiled once per
// pair with -DMQ_INST_DT=<0|1> and -DMQ_INST_BITS=<4|8> and with
// -fno-slp-vectorize: the vectorizer joins the blocks' scale arithmetic into
// vectors formed after the last of them, which takes the dequantization out of
// its places between the MFMAs.
#include "dense.cuh"
#include "grouped8.cuh"

#if !defined(MQ_INST_DT) || !defined(MQ_INST_BITS)
#error "compile with -DMQ_INST_DT=<0|1> -DMQ_INST_BITS=<4|8>"
#endif

namespace mq {
#define MQ_INST(GS) template struct WideLaunch<MQ_INST_DT, MQ_INST_BITS, GS>;
MQ_INST(32)
MQ_INST(64)
MQ_INST(128)
#undef MQ_INST
#if MQ_INST_BITS == 8
#define MQ_INST(GS)                               \
  template struct Thin8Launch<MQ_INST_DT, GS, false>; \
  template struct Thin8Launch<MQ_INST_DT, GS, true>;
MQ_INST(32)
MQ_INST(64)
MQ_INST(128)
#undef MQ_INST
#endif
}  // namespace mq
