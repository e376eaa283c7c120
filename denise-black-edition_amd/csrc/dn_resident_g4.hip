// Chip-resident time loop, FDORDER 8, acoustic, VTI, TTI and SH.
#define DN_F 4
#define DN_GROUP 1
#include "dn_resident_inst.inc"
