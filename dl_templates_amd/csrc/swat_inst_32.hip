#define DLT_D 32
#include "swat_inst.hpp"
