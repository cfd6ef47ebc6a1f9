// Wide-kernel instantiations of one (dtype, bits) pair, compiled once per pair
// with -DMQ_INST_DT=<0|1> and -DMQ_INST_BITS=<4|8> and with
// -fno-slp-vectorize: the vectorizer joins the blocks' scale arithmetic into
// vectors formed after the last of them, which takes the dequantization out of
// its places between the MFMAs.
#include "dense.cuh"

#if !defined(MQ_INST_DT) || !defined(MQ_INST_BITS)
#error "compile with -DMQ_INST_DT=<0|1> -DMQ_INST_BITS=<4|8>"
#endif

namespace mq {
template struct WideLaunch<MQ_INST_DT, MQ_INST_BITS, 32>;
template struct WideLaunch<MQ_INST_DT, MQ_INST_BITS, 64>;
template struct WideLaunch<MQ_INST_DT, MQ_INST_BITS, 128>;
}  // namespace mq
