// Row blocks that form the next block's keys and values, up to 128 tokens.
#include "row_block.hpp"

namespace tah {

template void launch_row_next<4, 2, 1>(const RowLaunch &);
template void launch_row_next<4, 2, 2>(const RowLaunch &);
template void launch_row_next<4, 1, 3>(const RowLaunch &);
template void launch_row_next<4, 1, 4>(const RowLaunch &);

}  // namespace tah
