// Row blocks that form the next block's keys and values, 129 to 256 tokens.
#include "row_block.hpp"

namespace tah {

template void launch_row_next<8, 1, 5>(const RowLaunch &);
template void launch_row_next<8, 1, 6>(const RowLaunch &);
template void launch_row_next<8, 1, 7>(const RowLaunch &);
template void launch_row_next<8, 1, 8>(const RowLaunch &);

}  // namespace tah
