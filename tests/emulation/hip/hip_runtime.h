// In place of the HIP headers when device code is compiled for the emulation.
#pragma once
#include "../emulation.hpp"
