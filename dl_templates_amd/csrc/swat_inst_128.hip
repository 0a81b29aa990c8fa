#define DLT_D 128
#include "swat_inst.hpp"
